// The INT8 mode on GGUF row-major weights: int8 activations (quantize_act_launch) times the blocks' codes with
// v_mfma_i32_16x16x32_i8, each block's exact sum folded as acc = fma(dot, s_a d, acc) in block order, so every tile
// shape gives the same bits (and those of the tiled weights' whole tiles).
//
// Bound by the fold, three vector instructions per result and block (a result lane and block: 12 cycles against the
// MFMA's 1), and, where few tiles leave one workgroup on a CU, by the latency of a stage. So the tiles are small (64 x 64
// fills 256 CUs at 1024 x 1024), eight waves share one, two to a SIMD, and a stage holds four blocks (128 of k): its
// loads are issued two stages ahead into registers, the weight bytes go to LDS unchanged and the operands are taken out
// of them with alignbyte (the 34-byte blocks put every other block's codes two bytes past a dword).
// With quantization, against 128 x 128 tiles of four waves with two blocks a stage, which this replaced (us): 1000 x
// 1024 x 4096 209 -> 42, 4096 x 4096 x 4096 566 -> 348, 256 x 1024 x 1024 64 -> 15, 1 x 1024 x 4096 183 -> 19.
#include "q8_gemm.h"

namespace idolq {
namespace {

constexpr int kBlocks = 4;                   // Q8_0 blocks per stage
constexpr int kStageK = kBlocks * kQ8Block;  // 128
constexpr int kAPitch = kStageK + 16;        // bytes per activation row in LDS (conflict-free 8-byte reads)
constexpr int kWPitch = 36;                  // dwords per weight row in LDS (34 used)

// BM x BN tile, WAVES waves in a WR x (WAVES / WR) grid, each TM x TN tiles of 16 x 16. W4: weight rows are 4-byte
// aligned (else 2). DOTS stores the int32 block sums instead (the bit-exact test entry point).
template <int BM, int BN, int WAVES, int WR, bool W4, bool DOTS>
__global__ __launch_bounds__(64 * WAVES, WAVES == 8 ? 2 : 1) void q8_gemm_i8_kernel(GemmParams p) {
    constexpr int THREADS = 64 * WAVES, WC = WAVES / WR, TM = BM / (16 * WR), TN = BN / (16 * WC);
    constexpr int kAPer = BM * (kStageK / 16) / THREADS;
    constexpr int kUnitsPerRow = W4 ? 34 : 68, kUnits = BN * kUnitsPerRow;
    constexpr int kWPer = (kUnits + THREADS - 1) / THREADS;
    constexpr int kWRows = (kWPer * THREADS + kUnitsPerRow - 1) / kUnitsPerRow;  // rows past BN take the unused units
    constexpr int kSPer = (BM * kBlocks + THREADS - 1) / THREADS, kSPitch = kSPer * THREADS / kBlocks;
    static_assert(BM * (kStageK / 16) % THREADS == 0 && TM * WR * 16 == BM && TN * WC * 16 == BN, "tile size");
    __shared__ __attribute__((aligned(16))) uint8_t a_lds[2][BM * kAPitch];
    __shared__ __attribute__((aligned(16))) uint32_t w_lds[2][kWRows * kWPitch];
    __shared__ __attribute__((aligned(16))) float s_lds[2][kBlocks * kSPitch];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WC, wn = wave % WC, lr = lane & 15, lg = lane >> 4;
    int tile_m, tile_n;
    tile_coords(p.tiles_m, p.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int nblocks = p.k / kQ8Block, nfull = nblocks / kBlocks;

    // The places of this thread's units, which no stage changes: byte offsets into x's codes, the weight window and the
    // scales, to which a stage adds a scalar offset (a full stage's loads and stores are then free of vector
    // arithmetic), and offsets into LDS. Rows outside x or the window, whose results are not written, read row 0. The
    // GEMM's entry point keeps codes and window below 2^32 bytes; the block sums' does not, and DOTS reads by pointer.
    typedef typename std::conditional<DOTS, int64_t, uint32_t>::type Offset;
    Offset a_off[kAPer], w_off[kWPer];
    uint32_t s_off[kSPer];
    int a_at[kAPer], w_at[kWPer], s_at[kSPer];
#pragma unroll
    for (int i = 0; i < kAPer; ++i) {
        const int u = tid + i * THREADS, row = u / (kStageK / 16), cu = u % (kStageK / 16);
        a_off[i] = (m0 + row < p.m ? (Offset)(m0 + row) * p.k : 0) + cu * 16;
        a_at[i] = row * kAPitch + cu * 16;
    }
#pragma unroll
    for (int i = 0; i < kWPer; ++i) {
        const int u = tid + i * THREADS, row = u / kUnitsPerRow, part = u % kUnitsPerRow;
        w_off[i] = (row < BN && n0 + row < p.n ? (Offset)((int64_t)(n0 + row) * p.row_bytes) : 0) + part * (W4 ? 4 : 2);
        w_at[i] = row * kWPitch * (W4 ? 1 : 2) + part;
    }
#pragma unroll
    for (int i = 0; i < kSPer; ++i) {
        const int u = tid + i * THREADS, row = u / kBlocks, b = u % kBlocks;
        s_off[i] = ((row < BM && m0 + row < p.m ? (uint32_t)(m0 + row) * (uint32_t)nblocks : 0) + b) * 4;
        s_at[i] = b * kSPitch + row;
    }
    auto rsrc = [](const void* base) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xffffffff, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ra = rsrc(p.qa), rw = rsrc(p.w), rs = rsrc(p.sa);

    struct Regs {
        uint4 a[kAPer];
        uint32_t w[kWPer];
        float s[kSPer];
    };
    // TAIL: the last stage of fewer blocks, whose units past the row's end become 0 and read the buffer's start
    auto load = [&](Regs& r, int st, auto tail) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail)::value;
        const int blk0 = st * kBlocks;
        auto in = [&](int block) __attribute__((always_inline)) { return !TAIL || blk0 + block < nblocks; };
#pragma unroll
        for (int i = 0; i < kAPer; ++i) {
            const bool ok = in((tid + i * THREADS) % (kStageK / 16) / 2);
            if constexpr (DOTS)
                r.a[i] = *reinterpret_cast<const uint4*>(p.qa + (ok ? a_off[i] + blk0 * kQ8Block : 0));
            else
                r.a[i] = __builtin_bit_cast(
                    uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, ok ? a_off[i] : 0, ok ? blk0 * kQ8Block : 0, 0));
            if (TAIL && !ok) r.a[i] = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < kWPer; ++i) {
            // (a dword straddles the first two or the last two blocks of a stage; W4 rows hold an even number)
            const bool ok = in((tid + i * THREADS) % kUnitsPerRow * (W4 ? 4 : 2) / kQ8Bytes);
            const int at = ok ? (int)w_off[i] : 0, st_off = ok ? blk0 * kQ8Bytes : 0;
            if constexpr (DOTS) {
                const uint8_t* src = p.w + (ok ? w_off[i] + st_off : 0);
                r.w[i] = W4 ? *reinterpret_cast<const uint32_t*>(src) : *reinterpret_cast<const uint16_t*>(src);
            } else {
                r.w[i] = W4 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, at, st_off, 0)
                            : (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw, at, st_off, 0);
            }
            if (TAIL && !ok) r.w[i] = 0;
        }
        if (!DOTS)
#pragma unroll
            for (int i = 0; i < kSPer; ++i) {
                const bool ok = in((tid + i * THREADS) % kBlocks);
                r.s[i] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rs, ok ? (int)s_off[i] : 0, ok ? blk0 * 4 : 0, 0));
                if (TAIL && !ok) r.s[i] = 0.0f;
            }
    };
    auto store = [&](const Regs& r, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kAPer; ++i) *reinterpret_cast<uint4*>(a_lds[buf] + a_at[i]) = r.a[i];
#pragma unroll
        for (int i = 0; i < kWPer; ++i) {
            if (W4)
                w_lds[buf][w_at[i]] = r.w[i];
            else
                reinterpret_cast<uint16_t*>(w_lds[buf])[w_at[i]] = (uint16_t)r.w[i];
        }
        if (!DOTS)
#pragma unroll
            for (int i = 0; i < kSPer; ++i) s_lds[buf][s_at[i]] = r.s[i];
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto multiply = [&](int st, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            // the last stage's blocks past the end hold zeros: their sums fold as +0 (DOTS skips them)
            if (DOTS && st * kBlocks + b >= nblocks) break;
            long af[TM], bf[TN];
            f32x4 sa[TM];
            float dw[TN];
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const int row = (wm * TM + t) * 16;
                af[t] = *reinterpret_cast<const long*>(a_lds[buf] + (row + lr) * kAPitch + b * kQ8Block + 8 * lg);
                if (!DOTS)
                    sa[t] = *reinterpret_cast<const f32x4*>(&s_lds[buf][b * kSPitch + row + 4 * lg]);
            }
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const uint32_t* w = w_lds[buf] + ((wn * TN + t) * 16 + lr) * kWPitch;
                // block b starts at byte 34 b: its scale, then its codes, for odd b on a dword
                uint32_t lo, hi;
                if (b & 1) {
                    const int at = (kQ8Bytes * b + 2) / 4 + 2 * lg;
                    lo = w[at], hi = w[at + 1];
                    dw[t] = half_bits_to_float((uint16_t)(w[kQ8Bytes * b / 4] >> 16));
                } else {
                    const int at = kQ8Bytes * b / 4 + 2 * lg;
                    const uint32_t x0 = w[at], x1 = w[at + 1], x2 = w[at + 2];
                    lo = __builtin_amdgcn_alignbyte(x1, x0, 2), hi = __builtin_amdgcn_alignbyte(x2, x1, 2);
                    dw[t] = half_bits_to_float((uint16_t)(w[kQ8Bytes * b / 4] & 0xffffu));
                }
                bf[t] = (long)((uint64_t)lo | ((uint64_t)hi << 32));
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const i32x4 dots = __builtin_amdgcn_mfma_i32_16x16x32_i8(af[i], bf[j], i32x4{0, 0, 0, 0}, 0, 0, 0);
                    if (DOTS) {
                        const int col = n0 + (wn * TN + j) * 16 + lr;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int row = m0 + (wm * TM + i) * 16 + 4 * lg + r;
                            if (row < p.m && col < p.n)
                                p.dots[((int64_t)row * p.n + col) * nblocks + st * kBlocks + b] = dots[r];
                        }
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[i][j][r] = fmaf((float)dots[r], sa[i][r] * dw[j], acc[i][j][r]);
                    }
                }
        }
    };

    // Two register sets and two LDS buffers, one barrier per stage: in stage st the registers of stage st + 1 go to the
    // other buffer (last read in stage st - 1) and are loaded again for stage st + 3. Past the last full stage the
    // loads are clamped and what they store is not read, so the loop has no branch for the compiler's waits to merge
    // over; a last stage of fewer blocks follows by itself.
    const std::false_type full;
    Regs r0, r1;
    if (nfull > 0) {
        load(r0, 0, full);
        load(r1, min(1, nfull - 1), full);
        store(r0, 0);
        load(r0, min(2, nfull - 1), full);
        __syncthreads();
        for (int st = 0; st < nfull; st += 2) {
            store(r1, 1);
            load(r1, min(st + 3, nfull - 1), full);
            multiply(st, 0);
            __syncthreads();
            if (st + 1 >= nfull) break;
            store(r0, 0);
            load(r0, min(st + 4, nfull - 1), full);
            multiply(st + 1, 1);
            __syncthreads();
        }
    }
    if (nfull * kBlocks < nblocks) {
        load(r0, nfull, std::true_type{});
        store(r0, 0);
        __syncthreads();
        multiply(nfull, 0);
    }
    if (DOTS) return;
    const bool round_first = (p.flags & IDOLQ_FLAG_ROUND_BEFORE_BIAS) != 0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = n0 + (wn * TN + j) * 16 + lr;
        if (col >= p.n) continue;
        const float bias = p.bias ? load_as_float(p.bias, p.bias_dt, col) : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + (wm * TM + i) * 16 + 4 * lg + r;
                if (row >= p.m) continue;
                float v = acc[i][j][r];
                if (round_first) v = round_through(p.y_dt, v);
                v += bias;
                if (p.res) v += load_as_float(p.res, p.res_dt, (int64_t)row * p.ldr + col);
                store_from_float(p.y, p.y_dt, (int64_t)row * p.ldy + col, apply_act(p.act, v));
            }
    }
}

template <int BM, int BN, int WAVES, int WR>
int launch_tile(GemmParams p, bool w4, hipStream_t stream) {
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    const dim3 grid((unsigned)p.tiles_m * (unsigned)p.tiles_n), block(64 * WAVES);
    if (p.dots)
        hipLaunchKernelGGL(w4 ? (q8_gemm_i8_kernel<BM, BN, WAVES, WR, true, true>)
                              : (q8_gemm_i8_kernel<BM, BN, WAVES, WR, false, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL(w4 ? (q8_gemm_i8_kernel<BM, BN, WAVES, WR, true, false>)
                              : (q8_gemm_i8_kernel<BM, BN, WAVES, WR, false, false>), grid, block, 0, stream, p);
    return check_launch("q8_gemm_i8_kernel");
}

}  // namespace

int launch_i8_rows(const GemmParams& p, bool w4, hipStream_t stream) {
    // Up to 16 rows: the weights are what is read, in 32-row tiles for more of them in flight. From 256 tiles of 128 x
    // 128 on (a round of the CUs) those, but for shallow depths, where their epilogue and the few stages of the one
    // workgroup a CU holds leave it waiting: k of 64, 1300 x 5586 32.1 us against 26.0 with 64 x 64; 1024, 4096^2 123
    // against 119; 1536, 160 against 162; 2048^3 59 against 63, 4096^3 347 against 389. Below 256 tiles 64 x 64: 2000 x
    // 1024 x 1024 (128 tiles) 23.3 against 34.5.
    if (p.m <= 16) return launch_tile<16, 32, 2, 1>(p, w4, stream);
    const int64_t large = (int64_t)((p.m + 127) / 128) * ((p.n + 127) / 128);
    if (large >= 256 && p.k > 1024) return launch_tile<128, 128, 8, 4>(p, w4, stream);
    return launch_tile<64, 64, 8, 4>(p, w4, stream);
}

}  // namespace idolq
