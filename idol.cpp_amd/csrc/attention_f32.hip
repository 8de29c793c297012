// fp32 attention on the bf16 matrix cores: every fp32 operand as the sum of three bf16 values.
//
// The fp32 matrix instructions (v_mfma_f32_32x32x2_f32) take 64 cycles for the products the bf16 ones do in 4, so an
// fp32 product made of six bf16 products has 2.7 times the rate. h = bf16(x), m = bf16(x - h) and l = bf16(x - h - m)
// hold all 24 bits of x at its own exponent: no operand has a scale, and none loses bits to a larger one beside it (a
// key may carry 1e12 in one channel, V 1e20 at a key of no weight, a query's weights may fall to 1e-30). Of the nine
// products hh, hm, mh, mm, hl and lh are kept; lm, ml and ll are at most 2^-25 of one. Everything is accumulated in
// fp32, hh of the product with V in an accumulator of its own: it rounds once per 16 keys where the fp32 instruction
// rounds after 2, so the result's 2-norm error is no larger than that kernel's (below). Q is scaled (log2(e) /
// sqrt(head_dim), one rounding, where that kernel rounds the scaled scores) before it is split: the maximum is then one
// of the scores and not another rounding of it, which at scores beyond 2^31 would differ by more than an exponent holds.
//
// attn_f32_split<HD, NW>: a workgroup of NW waves owns 32 NW queries of one (batch, head) and a range of 32-key tiles.
// The tile's K and V are split once per workgroup on their way into LDS (K planes [key][d], V planes transposed
// [d][key], the keys of a 16-chunk in the order in which a lane of the score accumulator holds them), two tile buffers,
// one barrier per tile. Scores are computed transposed, S^T = K Q^T, so a lane holds 16 scores of one query and its
// probabilities, split in registers, are the B operand of O^T = V^T P^T.
//
// Q and K of 2^60 and more, V of 2^70 and more and infinities are not split: a workgroup that meets one starts its part
// again with the fp32 matrix instructions on the same tiles in fp32, so that overflow and infinities go through the
// arithmetic of the plain fp32 product. A NaN splits into NaNs and needs no path of its own.
//
// 1000 queries x 8192 keys x 16 heads of 64, N(0, 1), against attn_f32_mfma on the same card: 185 us (181 TFLOP/s), 415;
// 2-norm error against fp64 3.3e-7, 8.8e-7. Where one channel decides the scores 4.0e-7 against 5.9e-7, with Q five
// times as large 5.0e-7 against 1.3e-6. With an infinite V, parts that start again: 333 us against 392. Q and K as fp16
// pairs under powers of two, 22 bits in half the products, took 160 us, but 7.2e-7 with one channel: not kept. Counters
// of that call: MFMA busy 197 k and vector instructions 151 k of 320 k cycles a SIMD, waves waiting 27% of their time:
// little of the one runs under the other (the barrier of every tile holds the two waves of a SIMD in the same phase).
//
// The key range is cut into parts (attn_f32_plan) where the query tiles alone leave CUs idle: each part writes its
// maxima, sums and unnormalized output, and attn_f32_combine merges them.
#include "attention.h"

#include "q8_dma.h"

namespace idolq {
namespace {

constexpr int kTile = 32;       // keys per tile
constexpr int kVP = kTile + 8;  // elements per d row of a V plane (80 bytes: conflict-free 16-byte reads)

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Q and K of 2^60 and more are not split: below, no product leaves fp32's range, and what bf16 has no bits for under
// 2^-126 is below 2^-60 in a score.
constexpr float kSplitLimit = 1152921504606846976.0f;
// The products kept besides hh: hl, lh, mm, hm, mh (lm, ml and ll are at most 2^-25 of a product).
constexpr int kSmall[5][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}};
// A lane's 16 probabilities 2^(score - maximum) of a tile sum to less than 2^kSumBits (to at most 16 where the maximum
// is the largest).
constexpr int kSumBits = 5;
// V is held times 2^24, so the lowest part of every normal value is one too; from 2^70 on it is not split (o stays
// below 2^94 times the number of keys and 2^kSumBits).
constexpr float kVScale = 16777216.0f, kVUnit = 1.0f / kVScale, kVLimit = 1180591620717411303424.0f;

// Two values as bf16 triples h, m, l: 8 bits each, all 24 bits of an fp32 value between them (down to 2^-109).
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    auto pack = [](float x, float y) __attribute__((always_inline)) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), bf16x2));
    };
    auto low = [](uint32_t w) __attribute__((always_inline)) { return __builtin_bit_cast(float, w << 16); };
    auto high = [](uint32_t w) __attribute__((always_inline)) { return __builtin_bit_cast(float, w & 0xffff0000u); };
    h = pack(a, b);
    const float ra = a - low(h), rb = b - high(h);
    m = pack(ra, rb);
    l = pack(ra - low(m), rb - high(m));
}

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// part_o [parts][batch][heads][lq][HD] unnormalized outputs, part_ml [...][lq][2] their maxima (base-2 domain) and sums
template <int HD, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attn_f32_split(AttnParams p, int qblocks, int parts, int per,
                                                             float* __restrict__ part_o,
                                                             float* __restrict__ part_ml) {
    constexpr int kBQ = 32 * NW;  // queries per workgroup
    constexpr int HH = HD / 2;    // depth per lane half of the fp32 instruction
    constexpr int DC = HD / 16;   // 16-deep chunks of the scores
    constexpr int DB = HD / 32;   // 32-wide d blocks of the output
    constexpr int EV = kTile * HD / (64 * NW);  // staged values per thread of K and of V
    constexpr int KP = HD + 8;    // elements per key row of a K plane (conflict-free 16-byte reads)
    __shared__ __attribute__((aligned(16))) uint16_t k_lds[2][3][kTile * KP];
    __shared__ __attribute__((aligned(16))) uint16_t v_lds[2][3][HD * kVP];
    __shared__ uint32_t beyond[2];  // the tile has values that are not split (never taken back)

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    // Workgroups go to the 8 XCDs in turn; the query blocks of one (batch, head, part) read the same keys, so where
    // the number of those groups allows it they are dealt to one XCD, whose L2 then serves the repeats.
    const int64_t groups = p.batch * p.heads * parts;
    int64_t g, qb;
    if (groups % 8 == 0) {
        const int64_t j = blockIdx.x >> 3;
        qb = j % qblocks;
        g = j / qblocks * 8 + (blockIdx.x & 7);
    } else {
        qb = blockIdx.x % qblocks;
        g = blockIdx.x / qblocks;
    }
    const int64_t part = g % parts, bh = g / parts, h = bh % p.heads, b = bh / p.heads;
    const int64_t lq = p.lq, lk = p.lk, ldkv = p.ldkv;
    const int64_t q0 = qb * kBQ + wave * 32, qi = q0 + col;
    const bool active = q0 < lq;  // wave-uniform: the others only stage
    const float* qbase = static_cast<const float*>(p.q) + b * p.q_bs + h * HD;
    const float* kbase = static_cast<const float*>(p.k) + b * p.kv_bs + h * HD;
    const float* vbase = static_cast<const float*>(p.v) + b * p.kv_bs + h * HD;

    // the lane's half of its query: x[8 c + e] is d = 16 c + 8 half + e
    float x[HH];
    auto load_query = [&]() __attribute__((always_inline)) {
        const float* qrow = qbase + (qi < lq ? qi : lq - 1) * p.ldq;
#pragma unroll
        for (int i = 0; i < HH; i += 4) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(qrow + 16 * (i >> 3) + 8 * half + (i & 4));
            x[i] = a[0], x[i + 1] = a[1], x[i + 2] = a[2], x[i + 3] = a[3];
        }
    };
    load_query();

    const int64_t tiles = (lk + kTile - 1) / kTile;
    const int64_t t0 = part * per, t1 = t0 + per < tiles ? t0 + per : tiles;
    float mc = -INFINITY, l_part = 0.0f;  // the running maximum (base-2 domain) and this lane's half of the sum
    f32x16 o[DB], small[DB];  // the sums of the products hh, and of the others
#pragma unroll
    for (int t = 0; t < DB; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f, small[t][r] = 0.0f;

    // Staging. K: thread t takes EV values of a key, a row to HD / EV consecutive threads. V: thread t takes d row
    // t % HD and EV keys whose places in that row of the plane are contiguous: place 16 kc + 8 half + e holds key
    // 16 kc + 8 (e / 4) + 4 half + e % 4.
    const int skey = tid / (HD / EV), sd = EV * (tid % (HD / EV));
    const int vd = tid % HD, vplace = tid / HD * EV;
    const int vkey = (vplace >> 4) * 16 + ((vplace >> 2) & 1) * 8 + ((vplace >> 3) & 1) * 4 + (vplace & 3);
    // a full tile's loads: per-thread byte offsets that no tile changes from a base that only the tile moves (both the
    // base and a V key's row offset are scalar); the host keeps 32 rows below 2^31 bytes
    const int koff = (int)(skey * ldkv + sd) * 4, voff = (int)(vkey * ldkv + vd) * 4;
    float kr[EV], vr[EV];
    auto load_tile = [&](int64_t t) __attribute__((always_inline)) {
        const int64_t k0 = t * kTile;
        if (k0 + kTile <= lk) {
            const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(kbase + k0 * ldkv), 0, 0x7fffffff, 0x00020000);
            const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(vbase + k0 * ldkv), 0, 0x7fffffff, 0x00020000);
            if constexpr (EV == 2) {
                const uint64_t v = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(rk, koff, 0, 0));
                kr[0] = __builtin_bit_cast(float, (uint32_t)v), kr[1] = __builtin_bit_cast(float, (uint32_t)(v >> 32));
            } else {
#pragma unroll
                for (int i = 0; i < EV; i += 4) {
                    const f32x4 v =
                        __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, koff + 4 * i, 0, 0));
                    kr[i] = v[0], kr[i + 1] = v[1], kr[i + 2] = v[2], kr[i + 3] = v[3];
                }
            }
            const int row = (int)ldkv * 4;
#pragma unroll
            for (int i = 0; i < EV; ++i)
                vr[i] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rv, voff, ((i >> 2) * 8 + (i & 3)) * row, 0));
        } else {  // the last tile: keys past lk are 0 (their scores are masked)
            const int64_t kk = k0 + skey;
#pragma unroll
            for (int i = 0; i < EV; ++i) kr[i] = kk < lk ? kbase[kk * ldkv + sd + i] : 0.0f;
#pragma unroll
            for (int i = 0; i < EV; ++i) {
                const int64_t vk = k0 + vkey + (i >> 2) * 8 + (i & 3);
                vr[i] = vk < lk ? vbase[vk * ldkv + vd] : 0.0f;
            }
        }
    };
    if (t0 < t1) load_tile(t0);

    bf16x8 qf[3][DC];  // Q^T operand planes, times the scale: scores come in the base-2 domain
    float qmax = 0.0f;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
        uint32_t w[3][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = x[8 * c + 2 * e], b = x[8 * c + 2 * e + 1];
            split3(a * p.scale_log2, b * p.scale_log2, w[0][e], w[1][e], w[2][e]);
            qmax = fmaxf(qmax, fmaxf(fabsf(a), fabsf(b)));
        }
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
            qf[pl][c] = __builtin_bit_cast(bf16x8, make_uint4(w[pl][0], w[pl][1], w[pl][2], w[pl][3]));
    }
    if (tid < 2) beyond[tid] = 0;
    __syncthreads();
    if (!(qmax < kSplitLimit)) beyond[0] = 1;

    auto stage_tile = [&](int buf) __attribute__((always_inline)) {
        float kmax = 0.0f, vmax = 0.0f;
        uint32_t w[3][EV / 2];
        auto store = [&](uint16_t* dst, int pl) __attribute__((always_inline)) {
            if constexpr (EV == 8)
                *reinterpret_cast<uint4*>(dst) = make_uint4(w[pl][0], w[pl][1], w[pl][2], w[pl][3]);
            else if constexpr (EV == 4)
                *reinterpret_cast<uint2*>(dst) = make_uint2(w[pl][0], w[pl][1]);
            else
                *reinterpret_cast<uint32_t*>(dst) = w[pl][0];
        };
#pragma unroll
        for (int e = 0; e < EV / 2; ++e) {
            split3(kr[2 * e], kr[2 * e + 1], w[0][e], w[1][e], w[2][e]);
            kmax = fmaxf(kmax, fmaxf(fabsf(kr[2 * e]), fabsf(kr[2 * e + 1])));
        }
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) store(&k_lds[buf][pl][skey * KP + sd], pl);
#pragma unroll
        for (int e = 0; e < EV / 2; ++e) {
            split3(vr[2 * e] * kVScale, vr[2 * e + 1] * kVScale, w[0][e], w[1][e], w[2][e]);
            vmax = fmaxf(vmax, fmaxf(fabsf(vr[2 * e]), fabsf(vr[2 * e + 1])));
        }
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) store(&v_lds[buf][pl][vd * kVP + vplace], pl);
        if (!(kmax < kSplitLimit && vmax < kVLimit)) beyond[buf] = 1;
    };

    // MASK: the last tile, with fewer than 32 keys; FIRST: the part's first tile, whose largest score sets the maximum
    auto compute = [&](int buf, int64_t k0, auto mask_tag, auto first_tag) __attribute__((always_inline)) {
        constexpr bool MASK = decltype(mask_tag)::value, FIRST = decltype(first_tag)::value;
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
        bf16x8 kf[3][DC];
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
#pragma unroll
            for (int c = 0; c < DC; ++c)
                kf[pl][c] = *reinterpret_cast<const bf16x8*>(&k_lds[buf][pl][col * KP + 16 * c + 8 * half]);
#pragma unroll
        for (int i = 0; i < 5; ++i)
#pragma unroll
            for (int c = 0; c < DC; ++c) s = mfma(kf[kSmall[i][0]][c], qf[kSmall[i][1]][c], s);
#pragma unroll
        for (int c = 0; c < DC; ++c) s = mfma(kf[0][c], qf[0][c], s);
        if (MASK) {
            const int valid = (int)(lk - k0);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (8 * (r >> 2) + 4 * half + (r & 3) >= valid) s[r] = -INFINITY;
        }
        // The maximum mc is the first tile's, raised only where a lane's probabilities of a tile sum to 2^kSumBits or
        // more, infinity and NaN included: no maximum is taken of the other tiles, the sum is needed anyway (a
        // wave-uniform branch). It is one of the scores as they are, so that the largest difference is 0 however large
        // they are. While every score was -inf, mc is -inf and 0 is subtracted: no weight.
        auto largest = [&]() __attribute__((always_inline)) {
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
            return fmaxf(mx, __shfl_xor(mx, 32));
        };
        if (FIRST) mc = largest();
        f32x16 pr;
        float lt;
        auto probabilities = [&]() __attribute__((always_inline)) {
            const float sub = mc == -INFINITY ? 0.0f : mc;
            float l2[2] = {0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                pr[r] = __builtin_amdgcn_exp2f(s[r] - sub);
                l2[r & 1] += pr[r];
            }
            lt = l2[0] + l2[1];
        };
        probabilities();
        if (!FIRST && __builtin_amdgcn_ballot_w64(!(lt < (float)(1 << kSumBits)) || mc == -INFINITY) != 0) {
            const float raised = fmaxf(mc, largest());
            const float alpha = mc < raised ? __builtin_amdgcn_exp2f(mc - raised) : 1.0f;
            mc = raised;
            l_part *= alpha;
#pragma unroll
            for (int t = 0; t < DB; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[t][r] *= alpha, small[t][r] *= alpha;
            probabilities();
        }
        l_part += lt;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            uint32_t w[3][4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                split3(pr[8 * kc + 2 * e], pr[8 * kc + 2 * e + 1], w[0][e], w[1][e], w[2][e]);
            bf16x8 pf[3], vf[DB][3];
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                pf[pl] = __builtin_bit_cast(bf16x8, make_uint4(w[pl][0], w[pl][1], w[pl][2], w[pl][3]));
#pragma unroll
            for (int t = 0; t < DB; ++t)
#pragma unroll
                for (int pl = 0; pl < 3; ++pl)
                    vf[t][pl] = *reinterpret_cast<const bf16x8*>(
                        &v_lds[buf][pl][(t * 32 + col) * kVP + 16 * kc + 8 * half]);
#pragma unroll
            for (int i = 0; i < 5; ++i)
#pragma unroll
                for (int t = 0; t < DB; ++t) small[t] = mfma(vf[t][kSmall[i][0]], pf[kSmall[i][1]], small[t]);
#pragma unroll
            for (int t = 0; t < DB; ++t) o[t] = mfma(vf[t][0], pf[0], o[t]);
        }
    };

    // tile t (in buffer buf): the next tile's loads, the product, the next tile's staging and the barrier that
    // publishes it; false where the tile has values that are not split
    int buf = 0;
    bool plain = false;  // uniform over the workgroup
    auto step = [&](int64_t t, auto mask_tag, auto first_tag) __attribute__((always_inline)) {
        const uint32_t out = beyond[buf];  // written before the last barrier, and next after this step's
        if (t + 1 < t1) load_tile(t + 1);
        if (active) compute(buf, t * kTile, mask_tag, first_tag);
        if (t + 1 < t1) stage_tile(buf ^ 1);
        __syncthreads();
        buf ^= 1;
        return __builtin_amdgcn_readfirstlane(out) == 0;
    };
    const int64_t full = t1 * kTile <= lk ? t1 : t1 - 1;  // the last tile of all may hold fewer keys
    if (t0 < t1) {
        stage_tile(0);
        __syncthreads();
        if (full > t0)
            plain = !step(t0, std::false_type{}, std::true_type{});
        else
            plain = !step(t0, std::true_type{}, std::true_type{});
        for (int64_t t = t0 + 1; t < full && !plain; ++t) plain = !step(t, std::false_type{}, std::false_type{});
        if (full < t1 && full > t0 && !plain) plain = !step(full, std::true_type{}, std::false_type{});
    }

    // The part with fp32 matrix instructions on the values themselves: tiles of fp32 in the same buffers, K [key][d], V
    // transposed as above. A lane half's 8 values of d or of keys are an instruction's two depths with the other's.
    constexpr int KF = HD + 4, VF = kTile + 4;  // floats per row (conflict-free 16-byte reads)
    static_assert(kTile * KF * 4 <= sizeof(k_lds[0]) && HD * VF * 4 <= sizeof(v_lds[0]), "the tiles fit");
    auto k_f32 = [&](int b) __attribute__((always_inline)) { return reinterpret_cast<float*>(k_lds[b][0]); };
    auto v_f32 = [&](int b) __attribute__((always_inline)) { return reinterpret_cast<float*>(v_lds[b][0]); };
    auto stage_plain = [&](int b) __attribute__((always_inline)) {
        auto store = [&](float* dst, const float (&v)[EV]) __attribute__((always_inline)) {
            if constexpr (EV == 2)
                *reinterpret_cast<f32x2*>(dst) = f32x2{v[0], v[1]};
            else
#pragma unroll
                for (int i = 0; i < EV; i += 4)
                    *reinterpret_cast<f32x4*>(dst + i) = f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
        };
        store(k_f32(b) + skey * KF + sd, kr);
        store(v_f32(b) + vd * VF + vplace, vr);
    };
    auto compute_plain = [&](int b, int64_t k0) __attribute__((always_inline)) {
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < HH; i += 4) {
            const f32x4 k4 = *reinterpret_cast<const f32x4*>(k_f32(b) + col * KF + 16 * (i >> 3) + 8 * half + (i & 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[e], x[i + e], s, 0, 0, 0);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = k0 + 8 * (r >> 2) + 4 * half + (r & 3) < lk ? s[r] * p.scale_log2 : -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        const float m_new = fmaxf(mc, fmaxf(mx, __shfl_xor(mx, 32)));
        const float sub = m_new == -INFINITY ? 0.0f : m_new;  // every score so far -inf: no weight
        const float alpha = __builtin_amdgcn_exp2f(mc - sub);
        mc = m_new;
        l_part *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = __builtin_amdgcn_exp2f(s[r] - sub);
            l_part += s[r];
        }
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; r += 4)
#pragma unroll
            for (int d = 0; d < DB; ++d) {
                const f32x4 v4 = *reinterpret_cast<const f32x4*>(v_f32(b) + (d * 32 + col) * VF + 16 * (r >> 3) +
                                                                 8 * half + (r & 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v4[e], s[r + e], o[d], 0, 0, 0);
            }
    };
#pragma unroll
    for (int t = 0; t < DB; ++t) o[t] += small[t];
    if (plain) {  // (after a barrier: no wave reads the buffers any more)
        mc = -INFINITY, l_part = 0.0f;
#pragma unroll
        for (int t = 0; t < DB; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
        load_query();
        if (t0 < t1) {
            load_tile(t0);
            stage_plain(0);
        }
        __syncthreads();
        buf = 0;
#pragma unroll 1
        for (int64_t t = t0; t < t1; ++t) {
            if (t + 1 < t1) load_tile(t + 1);
            if (active) compute_plain(buf, t * kTile);
            if (t + 1 < t1) stage_plain(buf ^ 1);
            __syncthreads();
            buf ^= 1;
        }
    }
    const float unit = plain ? 1.0f : kVUnit;  // of o

    const float l = l_part + __shfl_xor(l_part, 32);
    if (qi >= lq) return;
    if (parts > 1) {
        const int64_t row = ((part * p.batch + b) * p.heads + h) * lq + qi;
#pragma unroll
        for (int t = 0; t < DB; ++t)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const int d = t * 32 + 2 * r + 4 * half;
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = o[t][r + e] * unit;
                *reinterpret_cast<f32x4*>(part_o + row * HD + d) = v;
            }
        if (half == 0) *reinterpret_cast<f32x2*>(part_ml + 2 * row) = f32x2{mc, l};
        return;
    }
    const float inv = 1.0f / l;
    const int64_t obase = b * p.o_bs + qi * p.ldo + h * HD;
#pragma unroll
    for (int t = 0; t < DB; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const int d = t * 32 + 2 * r + 4 * half;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = o[t][r + e] * inv * unit;
            if (p.out_vec) {
                *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + obase + d) = f32x4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) store_from_float(p.out, p.out_dt, obase + d + e, v[e]);
            }
        }
}

// out = sum_s O_s 2^(m_s - m*) / sum_s l_s 2^(m_s - m*) over the parts; a wave per (batch, head, query) row: HD / 4
// lanes of 4 columns each, the parts dealt to the 64 / (HD / 4) groups of lanes, whose sums meet through shuffles (a
// fixed order). Reads every partial once; with the parts in groups their loads are in flight together.
template <int HD>
__global__ __launch_bounds__(256) void attn_f32_combine(AttnParams p, int parts, const float* __restrict__ part_o,
                                                        const float* __restrict__ part_ml) {
    constexpr int TPR = HD / 4, G = 64 / TPR;
    const int64_t rows = p.batch * p.heads * p.lq;
    const int64_t row = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63, group = lane / TPR, d = 4 * (lane % TPR);
    float mstar = -INFINITY, lsum = 0.0f;
    for (int s = lane; s < parts; s += 64) mstar = fmaxf(mstar, part_ml[2 * (s * rows + row)]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mstar = fmaxf(mstar, __shfl_xor(mstar, off));
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int s = group; s < parts; s += G) {
        const f32x2 ml = *reinterpret_cast<const f32x2*>(part_ml + 2 * (s * rows + row));
        const f32x4 v = *reinterpret_cast<const f32x4*>(part_o + (s * rows + row) * HD + d);
        // a part whose scores are all -inf has no weight (its sums are 0 unless NaN, which is kept)
        const float wgt = ml.x == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(ml.x - mstar);
        lsum = fmaf(ml.y, wgt, lsum);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(v[e], wgt, acc[e]);
    }
#pragma unroll
    for (int off = TPR; off < 64; off <<= 1) {
        lsum += __shfl_xor(lsum, off);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off);
    }
    if (group != 0) return;
    const float inv = 1.0f / lsum;
    const int64_t q = row % p.lq, bh = row / p.lq;
    const int64_t at = bh / p.heads * p.o_bs + q * p.ldo + bh % p.heads * HD + d;
    if (p.out_vec) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + at) = acc * inv;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) store_from_float(p.out, p.out_dt, at + e, acc[e] * inv);
    }
}

}  // namespace

// The cheapest of the kernel's forms (waves per workgroup), numbers of parts and, with waves 0, attn_f32_mfma, from
// measured times in microseconds: a tile step of the 4-wave form alone on its CU and of two there, of the 8-wave form
// with one wave of a SIMD at work (up to 128 queries) and with both; the steps' worth of a workgroup's start and end,
// and the merge (a launch and the partials written and read back). attn_f32_mfma steps 32 keys in each of its 4 waves,
// and each round of its workgroups starts anew. At heads of 64, the form taken against the next: 12 heads, 100 queries
// x 64 keys attn_f32_mfma 6.5 us, 4 waves 7.9; 16 heads, 1000 x 128 4 waves 12.2, attn_f32_mfma 14.5; 736 x 181 4 waves
// 16.3, parts of two 18.8, attn_f32_mfma 20.2; 128 x 700 8 waves in 11 parts 15.2, 4 waves in 22 18.2, attn_f32_mfma
// 22.3; 1000 x 8192 8 waves in 4 parts 176, 4 waves 195; 4096 x 421 8 waves 44.3, 4 waves 48.4.
AttnF32Plan attn_f32_plan(int64_t batch, int64_t lq, int64_t lk, int64_t heads, int64_t head_dim) {
    struct Steps {
        double mfma, mfma_start, mfma_first, alone, two, half, both;  // mfma_first: less for the first round's start
    };
    constexpr Steps kSteps64{2.85, 2.9, 1.8, 1.7, 2.75, 1.45, 2.45}, kSteps32{1.65, 0.7, 0.0, 1.08, 1.56, 1.0, 1.5};
    const Steps& c = head_dim == 64 ? kSteps64 : kSteps32;
    const int64_t cus = cu_count(), tiles = (lk + kTile - 1) / kTile;
    AttnF32Plan best{0, 1};
    double best_cost =
        (((lq + 31) / 32 * heads * batch + cus - 1) / cus) * ((tiles + 3) / 4 * c.mfma + c.mfma_start) - c.mfma_first;
    for (int nw = 4; nw <= 8; nw += 4) {
        const int64_t base = (lq + 32 * nw - 1) / (32 * nw) * heads * batch, slots = nw == 4 ? 2 * cus : cus;
        for (int s = 1; s <= 64 && s <= tiles && (s == 1 || s * base <= slots); ++s) {
            const int64_t per = (tiles + s - 1) / s, wgs = s * base;
            if (s > 1 && (tiles + per - 1) / per != s) continue;  // every part has tiles
            const double step = nw == 8 ? (lq <= 128 ? c.half : c.both) : wgs <= cus ? c.alone : c.two;
            const double merge = s == 1 ? 0.0 : 4.0 + 2.5e-6 * head_dim * (s * batch * heads * lq);
            const double cost = (per + (nw == 8 ? 1.9 : 1.5)) * step * ((wgs + slots - 1) / slots) + merge;
            if (cost < best_cost) best = {nw, s}, best_cost = cost;
        }
    }
    return best;
}

size_t attn_f32_workspace_bytes(int64_t batch, int64_t lq, int64_t heads, int64_t head_dim, int parts) {
    return parts <= 1 ? 0 : (size_t)parts * batch * heads * lq * (head_dim + 2) * sizeof(float);
}

int launch_attn_f32_split(const AttnParams& p, AttnF32Plan plan, float* workspace, hipStream_t s) {
    const int64_t bq = 32 * plan.waves, qblocks = (p.lq + bq - 1) / bq, rows = p.batch * p.heads * p.lq;
    const int64_t tiles = (p.lk + kTile - 1) / kTile, grid = qblocks * p.batch * p.heads * plan.parts;
    const int64_t per = (tiles + plan.parts - 1) / plan.parts;
    if (grid > 0x7fffffff || per > 0x7fffffff) return fail(IDOLQ_EINVAL, "grid too large");
    float* part_ml = plan.parts > 1 ? workspace + (size_t)plan.parts * rows * p.head_dim : nullptr;
    const dim3 g((unsigned)grid), block((unsigned)(64 * plan.waves));
    const auto kernel = p.head_dim == 64 ? (plan.waves == 8 ? attn_f32_split<64, 8> : attn_f32_split<64, 4>)
                                         : (plan.waves == 8 ? attn_f32_split<32, 8> : attn_f32_split<32, 4>);
    hipLaunchKernelGGL(kernel, g, block, 0, s, p, (int)qblocks, plan.parts, (int)per, workspace, part_ml);
    const int rc = check_launch("attn_f32_split");
    if (rc || plan.parts <= 1) return rc;
    const dim3 cgrid((unsigned)((rows + 3) / 4));
    hipLaunchKernelGGL(p.head_dim == 64 ? attn_f32_combine<64> : attn_f32_combine<32>, cgrid, dim3(256), 0, s, p,
                       plan.parts, workspace, part_ml);
    return check_launch("attn_f32_combine");
}

}  // namespace idolq
