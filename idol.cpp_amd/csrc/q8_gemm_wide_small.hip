// Small tiles of the grouped-layout GEMM (q8_wide.h): 32 or 64 rows of x by 128 weight rows, for calls whose larger
// tiles would leave most CUs idle (and the Q4_K GEMM's few-row calls, which have no other kernel). Whole tiles, k in
// order: the same bits as the larger tiles. Bound, alone on a CU, by the chain of a stage: barrier, LDS round trip and
// the conversion of 32 codes a lane (about 780 cycles, of which the MFMAs take 140 or 270). Several workgroups share a
// CU (kWideSlots), so one's chain passes under another's. 128 x 128 tiles measured slower than one or the other
// everywhere (1000 x 1536 x 1536 17 us against 14.6).
#include "q8_wide.h"

namespace idolq {
namespace {

template <typename T, bool Q4K>
int launch_small(const GemmParams& p, int rt, hipStream_t stream) {
    const long tiles = (long)((p.m + 32 * rt - 1) / (32 * rt)) * ((p.n + 127) / 128);
    WideSplit sp{0, 0, 0, 0, nullptr, nullptr};
    sp.G = (int)std::min(tiles, (long)wide_small_slots(rt) * cu_count());
    if (rt == 1) return launch_wide_s<T, 1, 1, false, Q4K>(p, sp, stream);
    return launch_wide_s<T, 2, 1, false, Q4K>(p, sp, stream);
}

}  // namespace

int wide_small_slots(int rt) { return rt == 1 ? kWideSlots<1, 1, 0> : kWideSlots<2, 1, 0>; }

int launch_wide_small(const GemmParams& p, int xt, bool q4k, int rt, hipStream_t stream) {
    if (q4k) return xt == XT_BF16 ? launch_small<__bf16, true>(p, rt, stream) : launch_small<_Float16, true>(p, rt, stream);
    return xt == XT_BF16 ? launch_small<__bf16, false>(p, rt, stream) : launch_small<_Float16, false>(p, rt, stream);
}

}  // namespace idolq
