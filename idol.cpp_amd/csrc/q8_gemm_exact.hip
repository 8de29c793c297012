// The EXACT mode with fp32 activations on GGUF row-major weights: x split into bf16 high and low parts, the codes exact
// in bf16, each block's fp32 sum of four v_mfma_f32_32x32x16_bf16 (high, then low) folded as acc = fma(sum, d, acc).
//
// Eight waves share a BM x BN tile: a 2 x 2 grid of wave tiles in two depth groups, the even and the odd blocks, whose
// sums meet at the end (a fixed order). x is split once per workgroup on its way into LDS; the weight bytes go to LDS
// unchanged, and each wave takes its operands out of them in registers (alignbyte for the blocks that start two bytes
// past a dword, a byte conversion and half a pack per code), so nothing waits for a second trip through LDS. Loads are
// issued two stages ahead into registers; a full stage's carry no masks. At 1024 rows a CU has one workgroup, and what
// bounds it is the chain of a stage (LDS round trip, conversion, MFMAs, fold): two blocks a stage, or four for 64 x 64
// tiles of deep products (launch_exact_rows); the larger tiles' LDS holds no more than two. Against the kernel this
// replaced, which converted the weights to bf16 in LDS: 1024 x 4096 x 1024 40 -> 36 us, 8192 x 2048 x 1024 157 -> 134,
// 310 x 5572 x 512 18.1 -> 14.6.
#include "q8_dma.h"
#include "q8_epilogue.h"

namespace idolq {
namespace {

// XA: x rows are 16-byte aligned (else 4). W4: weight rows are 4-byte aligned (else 2).
template <int BM, int BN, int NB, bool XA, bool W4>
__global__ __launch_bounds__(512, 2) void q8_gemm_exact_kernel(GemmParams p) {
    constexpr int THREADS = 512, WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int kStageK = NB * kQ8Block;
    constexpr int kXPitch = kStageK + 8;  // elements per row of an x plane (conflict-free 16-byte reads)
    constexpr int kXUnits = kStageK / 4;  // 4-value units per row
    constexpr int kXPer = BM * kXUnits / THREADS;
    constexpr int kUnitsPerRow = NB * (W4 ? 17 : 34) / 2, kUnits = BN * kUnitsPerRow;
    constexpr int kWPitch = (NB * 17 / 2) | 1;  // dwords per weight row (odd: conflict-free)
    constexpr int kWPer = (kUnits + THREADS - 1) / THREADS;
    constexpr int kWRows = (kWPer * THREADS + kUnitsPerRow - 1) / kUnitsPerRow;  // rows past BN take the unused units
    constexpr int kXBytes = BM * kXPitch * 2, kWBytes = (kWRows * kWPitch * 4 + 15) / 16 * 16;
    constexpr int kLoopBytes = 2 * (2 * kXBytes + kWBytes), kStageBytes = BM * (BN + 4) * 4;
    static_assert(NB % 2 == 0 && BM * kXUnits % THREADS == 0, "tile size");
    __shared__ __attribute__((aligned(16))) char smem[kLoopBytes > kStageBytes ? kLoopBytes : kStageBytes];
    auto x_lds = [&](int buf, int part) __attribute__((always_inline)) {
        return reinterpret_cast<uint16_t*>(smem + (2 * buf + part) * kXBytes);
    };
    auto w_lds = [&](int buf) __attribute__((always_inline)) {
        return reinterpret_cast<uint32_t*>(smem + 4 * kXBytes + buf * kWBytes);
    };

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1, lr = lane & 31, lg = lane >> 5;
    int tile_m, tile_n;
    tile_coords(p.tiles_m, p.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int nblocks = p.k / kQ8Block, nfull = nblocks / NB;

    // The places of this thread's units, which no stage changes. Rows outside x or the weight window, whose results
    // are not written, read row 0.
    const float* x_at[kXPer];
    int x_to[kXPer];
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
        const int u = tid + i * THREADS, row = u / kXUnits, c = u % kXUnits * 4;
        x_at[i] = static_cast<const float*>(p.x) + (m0 + row < p.m ? (int64_t)(m0 + row) * p.ldx : 0) + c;
        x_to[i] = row * kXPitch + c;
    }
    uint32_t w_off[kWPer];
    int w_to[kWPer];
#pragma unroll
    for (int i = 0; i < kWPer; ++i) {
        const int u = tid + i * THREADS, row = u / kUnitsPerRow, part = u % kUnitsPerRow;
        w_off[i] = (row < BN && n0 + row < p.n ? (uint32_t)((int64_t)(n0 + row) * p.row_bytes) : 0) + part * (W4 ? 4 : 2);
        w_to[i] = row * kWPitch * (W4 ? 1 : 2) + part;
    }
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), 0, 0xffffffff, 0x00020000);

    struct Regs {
        f32x4 x[kXPer];
        uint32_t w[kWPer];
    };
    // TAIL: the last stage of fewer blocks, whose units past the row's end become 0 and read the buffers' start
    auto load = [&](Regs& r, int st, auto tail) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail)::value;
        const int blk0 = st * NB;
        auto in = [&](int block) __attribute__((always_inline)) { return !TAIL || blk0 + block < nblocks; };
#pragma unroll
        for (int i = 0; i < kXPer; ++i) {
            const bool ok = in((tid + i * THREADS) % kXUnits * 4 / kQ8Block);
            const float* src = ok ? x_at[i] + blk0 * kQ8Block : static_cast<const float*>(p.x);
            if (XA)
                r.x[i] = *reinterpret_cast<const f32x4*>(src);
            else
                r.x[i] = f32x4{src[0], src[1], src[2], src[3]};
            if (TAIL && !ok) r.x[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int i = 0; i < kWPer; ++i) {
            // (a dword straddles a stage's even block and the odd one after it; W4 rows hold an even number)
            const bool ok = in((tid + i * THREADS) % kUnitsPerRow * (W4 ? 4 : 2) / kQ8Bytes);
            const int at = ok ? (int)w_off[i] : 0, st_off = ok ? blk0 * kQ8Bytes : 0;
            r.w[i] = W4 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, at, st_off, 0)
                        : (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw, at, st_off, 0);
            if (TAIL && !ok) r.w[i] = 0;
        }
    };
    auto store = [&](const Regs& r, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kXPer; ++i) {
            uint32_t h[2], l[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float a = r.x[i][2 * e], b = r.x[i][2 * e + 1];
                h[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
                const f32x2 rest = {a - __builtin_bit_cast(float, h[e] << 16),
                                    b - __builtin_bit_cast(float, h[e] & 0xffff0000u)};
                l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
            }
            *reinterpret_cast<uint2*>(x_lds(buf, 0) + x_to[i]) = make_uint2(h[0], h[1]);
            *reinterpret_cast<uint2*>(x_lds(buf, 1) + x_to[i]) = make_uint2(l[0], l[1]);
        }
#pragma unroll
        for (int i = 0; i < kWPer; ++i) {
            if (W4)
                w_lds(buf)[w_to[i]] = r.w[i];
            else
                reinterpret_cast<uint16_t*>(w_lds(buf))[w_to[i]] = (uint16_t)r.w[i];
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // the group's blocks of a stage: 2 b + kg
    auto multiply = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB / 2; ++b) {
            const int k0 = (2 * b + kg) * kQ8Block;
            bf16x8 xf[TM][2][2], wf[TN][2];
            float d[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        xf[i][part][h] = *reinterpret_cast<const bf16x8*>(
                            x_lds(buf, part) + (wm * WM + i * 32 + lr) * kXPitch + k0 + 16 * h + 8 * lg);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                // a pair of blocks is 17 dwords: the even one's scale starts it and its codes lie two bytes past a dword,
                // the odd one's the other way round (alignbyte by 0 takes the first dword)
                const uint32_t* w = w_lds(buf) + (wn * WN + j * 32 + lr) * kWPitch + 17 * b + 9 * kg;
                d[j] = half_bits_to_float((uint16_t)(w[-kg] >> (16 * kg)));
                uint2 c[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t* q = w + 4 * h + 2 * lg;
                    c[h] = make_uint2(__builtin_amdgcn_alignbyte(q[1], q[0], 2 - 2 * kg),
                                      __builtin_amdgcn_alignbyte(q[2], q[1], 2 - 2 * kg));
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    wf[j][h] = __builtin_bit_cast(bf16x8, codes_to_operand<__bf16, MODE_EXACT>(c[h], 0.0f));
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    f32x16 sum;
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[r] = 0.0f;
#pragma unroll
                    for (int part = 0; part < 2; ++part)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[i][part][h], wf[j][h], sum, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(sum[r], d[j], acc[i][j][r]);
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
        // (pinned in this order: were stage 1's loads moved past stage 2's, the loop's waits for the one would cover
        // the other in every stage)
        load(r0, 0, full);
        load(r1, min(1, nfull - 1), full);
        __builtin_amdgcn_sched_barrier(0);
        store(r0, 0);
        load(r0, min(2, nfull - 1), full);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        int st = 0;
        for (; st + 1 < nfull; st += 2) {
            store(r1, 1);
            load(r1, min(st + 3, nfull - 1), full);
            __builtin_amdgcn_sched_barrier(0);  // issued before the stage's work, not sunk to its end
            multiply(0);
            __syncthreads();
            store(r0, 0);
            load(r0, min(st + 4, nfull - 1), full);
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
            __syncthreads();
        }
        if (st < nfull) {
            multiply(0);
            __syncthreads();
        }
    }
    if (nfull * NB < nblocks) {
        load(r0, nfull, std::true_type{});
        store(r0, 0);
        __syncthreads();
        multiply(0);
        __syncthreads();
    }
    add_depth_groups<BN, TM, TN, WM, WN>(acc, reinterpret_cast<float*>(smem));
    write_tile_staged<BM, BN, TM, TN, WM, WN, THREADS, 2>(p, acc, m0, n0, reinterpret_cast<float*>(smem));
}

// A 64 x 64 tile whose eight waves each take every eighth pair of blocks for the whole tile: each converted code and
// each x operand feeds twice the products of a 32 x 32 wave tile, and a wave stages its pair in LDS of its own, so the
// loop has no barrier; the waves' sums meet in LDS at the end, in wave order. 1024 x 1024 x 4096 37 us against 43 with the
// kernel above, 1024 x 1024 x 1024 14.2 against 15.5; 1024 x 4096 x 1024, four rounds of such tiles, 52 against 36 with
// 128 x 128. Vector work (conversion, split, fold: about 430 instructions per pair and
// wave) and the MFMAs bound it, little of the one under the other.
__global__ __launch_bounds__(512, 2) void q8_gemm_exact_split_kernel(GemmParams p) {
    constexpr int kTileMN = 64, kWaves = 8;
    constexpr int kXPitch = kQ8Block + 8;           // elements per row of an x plane of one block (conflict-free reads)
    constexpr int kXLoads = kTileMN * kQ8Block / 4 / 64;  // 16-byte loads per lane of a block of x
    constexpr int kWUnits = 17;                     // dwords per row of a pair of weight blocks
    constexpr int kXBytes = kTileMN * kXPitch * 2, kWBytes = kTileMN * 17 * 4;
    constexpr int kWaveBytes = 2 * kXBytes + kWBytes;
    constexpr int kPitch = kTileMN + 4, kSumBytes = kTileMN * kPitch * 4;
    constexpr int kBytes = kWaves * (kWaveBytes > kSumBytes ? kWaveBytes : kSumBytes);
    __shared__ __attribute__((aligned(16))) char smem[kBytes];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, lg = lane >> 5;
    uint16_t* x_lds = reinterpret_cast<uint16_t*>(smem + wave * kWaveBytes);
    uint32_t* w_lds = reinterpret_cast<uint32_t*>(smem + wave * kWaveBytes + 2 * kXBytes);
    int tile_m, tile_n;
    tile_coords(p.tiles_m, p.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * kTileMN, n0 = tile_n * kTileMN;
    const int npairs = p.k / (2 * kQ8Block);

    // Load i of x: row 8 i + lane / 8, values 4 (lane % 8) .. of a block. Unit lane + 64 i of the weights' flat run of 64
    // rows. Rows outside x or the window lie past their buffer's end and read 0.
    const int xrow = lane >> 3, xc = 4 * (lane & 7), ldx4 = (int)p.ldx * 4;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(static_cast<const float*>(p.x) + (int64_t)m0 * p.ldx), 0,
        (uint32_t)min(p.m - m0, kTileMN) * (uint32_t)ldx4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.w), 0, (uint32_t)((int64_t)p.n * p.row_bytes), 0x00020000);
    const int x_off = xrow * ldx4 + xc * 4;
    f32x4 xr[2][kXLoads];
    uint32_t wr[kWUnits];
    auto load_x = [&](int b, int pair) __attribute__((always_inline)) {
        const int at = (2 * pair + b) * kQ8Block * 4;
#pragma unroll
        for (int i = 0; i < kXLoads; ++i)
            xr[b][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, x_off + 8 * i * ldx4, at, 0));
    };
    auto load_w = [&](int pair) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kWUnits; ++i) {
            const int u = lane + 64 * i;
            const uint32_t at = (uint32_t)(n0 + u / kWUnits) * (uint32_t)p.row_bytes + 4 * (u % kWUnits);
            wr[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rw, (int)at, pair * 2 * kQ8Bytes, 0);
        }
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    if (wave < npairs) {
        load_x(0, wave);
        load_w(wave);
        load_x(1, wave);
    }
    // the wave's LDS operations run in order; the fences keep the compiler from moving reads above writes or the
    // other way round
    auto in_order = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (int pair = wave; pair < npairs; pair += kWaves) {
        const int next = min(pair + kWaves, npairs - 1);  // past the last pair: loaded, not read
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
            for (int i = 0; i < kXLoads; ++i) {
                uint32_t h[2], l[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float a = xr[blk][i][2 * e], b = xr[blk][i][2 * e + 1];
                    h[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
                    const f32x2 rest = {a - __builtin_bit_cast(float, h[e] << 16),
                                        b - __builtin_bit_cast(float, h[e] & 0xffff0000u)};
                    l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
                }
                uint16_t* to = x_lds + (8 * i + xrow) * kXPitch + xc;
                *reinterpret_cast<uint2*>(to) = make_uint2(h[0], h[1]);
                *reinterpret_cast<uint2*>(to + kXBytes / 2) = make_uint2(l[0], l[1]);
            }
            if (blk == 0) {
#pragma unroll
                for (int i = 0; i < kWUnits; ++i) w_lds[lane + 64 * i] = wr[i];
            }
            load_x(blk, next);
            if (blk == 0) load_w(next);
            in_order();
            bf16x8 xf[2][2][2], wf[2][2];
            float d[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        xf[i][part][h] = *reinterpret_cast<const bf16x8*>(x_lds + part * (kXBytes / 2) +
                                                                          (i * 32 + lr) * kXPitch + 16 * h + 8 * lg);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t* w = w_lds + (j * 32 + lr) * 17;
                d[j] = half_bits_to_float((uint16_t)(blk ? w[8] >> 16 : w[0] & 0xffffu));
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t* q = w + (blk ? 9 : 0) + 4 * h + 2 * lg;
                    const uint2 c = blk ? make_uint2(q[0], q[1])
                                        : make_uint2(__builtin_amdgcn_alignbyte(q[1], q[0], 2),
                                                     __builtin_amdgcn_alignbyte(q[2], q[1], 2));
                    wf[j][h] = __builtin_bit_cast(bf16x8, codes_to_operand<__bf16, MODE_EXACT>(c, 0.0f));
                }
            }
            in_order();
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    f32x16 sum;
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[r] = 0.0f;
#pragma unroll
                    for (int part = 0; part < 2; ++part)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[i][part][h], wf[j][h], sum, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(sum[r], d[j], acc[i][j][r]);
                }
        }
    }

    __syncthreads();
    float* sums = reinterpret_cast<float*>(smem) + wave * (kTileMN * kPitch);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                sums[(i * 32 + 8 * (r >> 2) + 4 * lg + (r & 3)) * kPitch + j * 32 + lr] = acc[i][j][r];
    __syncthreads();
    const int row = tid >> 3, col = 8 * (tid & 7);
    if (m0 + row >= p.m || n0 + col >= p.n) return;
    float v[8];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const float* from = reinterpret_cast<const float*>(smem) + w * (kTileMN * kPitch) + row * kPitch + col;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(from), hi = *reinterpret_cast<const f32x4*>(from + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (w ? v[e] : 0.0f) + (e < 4 ? lo[e & 3] : hi[e & 3]);
    }
    const bool round_first = (p.flags & IDOLQ_FLAG_ROUND_BEFORE_BIAS) != 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if (round_first) v[e] = round_through(p.y_dt, v[e]);
        v[e] += p.bias && n0 + col + e < p.n ? load_as_float(p.bias, p.bias_dt, n0 + col + e) : 0.0f;
    }
    store_run(p, m0 + row, n0 + col, v);
}

template <int BM, int BN, int NB>
int launch_tile(GemmParams p, bool w4, hipStream_t stream) {
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    const dim3 grid((unsigned)p.tiles_m * (unsigned)p.tiles_n), block(512);
    if (w4 && p.x_aligned)
        hipLaunchKernelGGL((q8_gemm_exact_kernel<BM, BN, NB, true, true>), grid, block, 0, stream, p);
    else if (w4)
        hipLaunchKernelGGL((q8_gemm_exact_kernel<BM, BN, NB, false, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((q8_gemm_exact_kernel<BM, BN, NB, false, false>), grid, block, 0, stream, p);
    return check_launch("q8_gemm_exact_kernel");
}

int launch_split(GemmParams p, hipStream_t stream) {
    p.tiles_m = (p.m + 63) / 64;
    p.tiles_n = (p.n + 63) / 64;
    const dim3 grid((unsigned)p.tiles_m * (unsigned)p.tiles_n);
    hipLaunchKernelGGL(q8_gemm_exact_split_kernel, grid, dim3(512), 0, stream, p);
    return check_launch("q8_gemm_exact_split_kernel");
}

}  // namespace

int launch_exact_rows(const GemmParams& p, bool w4, hipStream_t stream) {
    // Measured with each tile over 23 shapes at depths of 256, 1024 and 4096, the choice is within 2% of the best. At
    // 1024 x 1024 x 1024 the split kernel takes 14.2 us, 128 x 64 21.5; at 1024 x 1280 x 1024, past one round of 64 x 64
    // tiles, 24.3 against 21.7; at 1024 x 3072 x 1024 128 x 64 takes 39.8, 128 x 128 32.8.
    static const TileChoice cands[] = {{128, 128, 1.0f}, {128, 64, 1.0f}, {64, 64, 0.75f}};
    const TileChoice t = choose_tile(p.m, p.n, cands, 3);
    if (t.bn == 128) return launch_tile<128, 128, 2>(p, w4, stream);
    if (t.bm == 128) return launch_tile<128, 64, 2>(p, w4, stream);
    // 64 x 64, measured in us as split kernel / four blocks a stage / two. Two leave room for two workgroups a CU and take
    // the fewest bytes of a short row: best up to a depth of 512 in one round of the CUs (1000 x 1024 x 64 8.1 / 7.0 / 6.3,
    // x 512 10.8 / 10.6 / 10.8, x 1024 13.7 / 14.7 / 15.4), up to 2048 in more (310 x 5572 x 64 13.9 / 11.8 / 7.4, x 1024
    // 24.4 / 26.6 / 21.7, x 2048 37.6 / 43.5 / 37.5, x 4096 62.8 / 76.7 / 66.5). Beyond, the split kernel for aligned rows
    // of whole pairs of blocks, 64 rows of x below 2^31 bytes.
    const bool one_round = (int64_t)((p.m + 63) / 64) * ((p.n + 63) / 64) <= cu_count();
    const bool shallow = p.k <= (one_round ? 512 : 2048);
    if (!shallow && w4 && p.x_aligned && p.ldx < 1 << 23) return launch_split(p, stream);
    if (!shallow && one_round) return launch_tile<64, 64, 4>(p, w4, stream);
    return launch_tile<64, 64, 2>(p, w4, stream);
}

}  // namespace idolq
