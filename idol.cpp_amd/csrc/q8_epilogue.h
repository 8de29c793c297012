// Device code shared by the Q8_0 GEMM kernels on GGUF row-major weights (q8_gemm.hip, q8_gemm_exact.hip): codes to
// operands, and the epilogue through LDS.
#pragma once

#include <algorithm>

#include "q8_gemm.h"

namespace idolq {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Eight int8 codes (in a uint2) to eight 16-bit operand values: exact codes, or T(fp32(d) * q). Pairs are rounded
// together (one v_cvt_pk_bf16_f32 for bf16).
template <typename T, int MODE>
__device__ __forceinline__ uint4 codes_to_operand(uint2 raw, float d) {
    typedef typename std::conditional<std::is_same<T, __bf16>::value, bf16x2, f16x2>::type T2;
    uint32_t out[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t word = e < 2 ? raw.x : raw.y;
        const int sh = 16 * (e & 1);
        f32x2 f;
        f.x = (float)(int)(int8_t)(uint8_t)(word >> sh);
        f.y = (float)(int)(int8_t)(uint8_t)(word >> (sh + 8));
        if (MODE == MODE_DEQUANT) f = f * d;
        out[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, T2));
    }
    return make_uint4(out[0], out[1], out[2], out[3]);
}

// A run of 8 consecutive columns of one row (rounded and with its bias): residual, activation and store, as whole
// vectors where y_vec allows and the run is inside n.
__device__ __forceinline__ void store_run(const GemmParams& p, int grow, int gcol, float (&v)[8]) {
    const int cnt = min(8, p.n - gcol);
    if (cnt == 8 && p.y_vec) {
        float r[8];
        if (p.res) {
            const char* rp = static_cast<const char*>(p.res) + ((int64_t)grow * p.ldr + gcol) * (p.res_dt == IDOLQ_F32 ? 4 : 2);
            if (p.res_dt == IDOLQ_F32) {
                const float4 a = reinterpret_cast<const float4*>(rp)[0], b = reinterpret_cast<const float4*>(rp)[1];
                r[0] = a.x, r[1] = a.y, r[2] = a.z, r[3] = a.w, r[4] = b.x, r[5] = b.y, r[6] = b.z, r[7] = b.w;
            } else {
                const uint4 u = *reinterpret_cast<const uint4*>(rp);
                const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint16_t bits = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
                    r[e] = p.res_dt == IDOLQ_BF16 ? bf16_bits_to_float(bits) : half_bits_to_float(bits);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = apply_act(p.act, p.res ? v[e] + r[e] : v[e]);
        char* yp = static_cast<char*>(p.y) + ((int64_t)grow * p.ldy + gcol) * (p.y_dt == IDOLQ_F32 ? 4 : 2);
        if (p.y_dt == IDOLQ_F32) {
            reinterpret_cast<float4*>(yp)[0] = make_float4(v[0], v[1], v[2], v[3]);
            reinterpret_cast<float4*>(yp)[1] = make_float4(v[4], v[5], v[6], v[7]);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint16_t a = p.y_dt == IDOLQ_BF16 ? float_to_bf16_bits(v[2 * e]) : float_to_half_bits(v[2 * e]);
                const uint16_t b = p.y_dt == IDOLQ_BF16 ? float_to_bf16_bits(v[2 * e + 1]) : float_to_half_bits(v[2 * e + 1]);
                w[e] = (uint32_t)a | ((uint32_t)b << 16);
            }
            *reinterpret_cast<uint4*>(yp) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    } else {
        for (int e = 0; e < cnt; ++e) {
            float x = v[e];
            if (p.res) x += load_as_float(p.res, p.res_dt, (int64_t)grow * p.ldr + gcol + e);
            store_from_float(p.y, p.y_dt, (int64_t)grow * p.ldy + gcol + e, apply_act(p.act, x));
        }
    }
}

// Epilogue through LDS: the accumulator tile is written to LDS as fp32 ([BM][BN + 4]), then each thread takes runs of
// 8 consecutive columns of one row and applies the epilogue with vector loads of bias and residual and one 16-byte
// (32-byte for fp32) store per run, so each wave writes whole row segments instead of 2-byte scattered stores.
// KS == 2: the workgroup's waves form two depth groups and only the first group's accumulators (which already hold
// the second group's sums) are written.
template <int BM, int BN, int TM, int TN, int WM, int WN, int THREADS, int KS = 1>
__device__ __forceinline__ void write_tile_staged(const GemmParams& p, const f32x16 (&acc)[TM][TN], int m0, int n0,
                                                  float* stage) {
    constexpr int kPitch = BN + 4;
    constexpr int kRuns = BN / 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wq = wave % (THREADS / 64 / KS);
    const int wm = wq >> 1, wn = wq & 1;
    const bool round_first = (p.flags & IDOLQ_FLAG_ROUND_BEFORE_BIAS) != 0;
    __syncthreads();
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
        if (KS == 2 && wave >= THREADS / 128) break;
        const int col = wn * WN + tn * 32 + (lane & 31);
        const float bias = p.bias && n0 + col < p.n ? load_as_float(p.bias, p.bias_dt, n0 + col) : 0.0f;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = wm * WM + tm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float v = acc[tm][tn][r];
                if (round_first) v = round_through(p.y_dt, v);
                stage[row * kPitch + col] = v + bias;
            }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < BM * kRuns; c += THREADS) {
        const int row = c / kRuns, col = (c % kRuns) * 8;
        const int grow = m0 + row, gcol = n0 + col;
        if (grow >= p.m || gcol >= p.n) continue;
        float v[8];
        const float4 lo = *reinterpret_cast<const float4*>(stage + row * kPitch + col);
        const float4 hi = *reinterpret_cast<const float4*>(stage + row * kPitch + col + 4);
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
        store_run(p, grow, gcol, v);
    }
}

// The second depth group's sums (waves 4 .. 7 of 8, odd blocks) through LDS into the first's: a fixed order.
template <int BN, int TM, int TN, int WM, int WN>
__device__ __forceinline__ void add_depth_groups(f32x16 (&acc)[TM][TN], float* red) {
    constexpr int kPitch = BN + 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    __syncthreads();
    if (kg == 1)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[(wm * WM + tm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kPitch + wn * WN + tn * 32 +
                        (lane & 31)] = acc[tm][tn][r];
    __syncthreads();
    if (kg == 0)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[tm][tn][r] += red[(wm * WM + tm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kPitch +
                                          wn * WN + tn * 32 + (lane & 31)];
}

}  // namespace

// Tile choice: one workgroup per CU fits in LDS, so a launch runs in ceil(tiles / 256) rounds on the 256 CUs; pick
// the tile with the smallest rounds * tile area / efficiency (the per-CU critical path). `eff` is the tile's measured
// throughput relative to the 256 x 128 eight-wave tile on a large GEMM (4096 x 6144 x 1536).
struct TileChoice {
    int bm, bn;
    float eff;
};

inline TileChoice choose_tile(int m, int n, const TileChoice* cands, int count) {
    constexpr long kCUs = 256;
    TileChoice best = cands[0];
    float best_cost = -1.0f;
    for (int i = 0; i < count; ++i) {
        const long tiles = (long)((m + cands[i].bm - 1) / cands[i].bm) * ((n + cands[i].bn - 1) / cands[i].bn);
        const float cost = (float)((tiles + kCUs - 1) / kCUs * cands[i].bm * cands[i].bn) / cands[i].eff;
        if (best_cost < 0.0f || cost < best_cost) {
            best = cands[i];
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace idolq
