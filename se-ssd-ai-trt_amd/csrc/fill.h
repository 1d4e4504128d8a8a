// fill.h -- the fill pass: as a launch of its own (fill.hip) and beside the blocks of other passes (coord.hip).
#pragma once

#include "common.h"

namespace sessd {

// One launch clears up to N regions.  The blocks are flat: region i owns the blocks [first_block[i],
// first_block[i+1]), as many as its size asks for (a small region gets one block, not the grid of the largest one), and
// its blocks stride over it with 16-byte stores (pure write stream, HBM-bound).
// N = regions the kernel's argument has room for.  The host copies the whole argument on every launch: with all 48 it
// is 1.4 KB and a launch takes the host 4.2 us, with the few that one plugin clears 2.8.
template <int N>
struct FillPlan {
    FillRegion r[N];
    uint32_t first_block[N + 1];
    int32_t n;
};
constexpr int kFewRegions = 8;

// -> blocks of the plan, or 0 for none; -1 when a region is not 16-byte aligned
template <int N>
inline int make_fill_plan(const FillArgs& a, FillPlan<N>& p) {
    p.n = a.n;
    uint32_t total = 0;
    for (int i = 0; i < a.n; ++i) {
        if (reinterpret_cast<uintptr_t>(a.r[i].ptr) & 15) return -1;
        // 4 stores of 16 B per thread is enough to saturate HBM; at most 8 blocks per CU for one region
        uint64_t blocks = (a.r[i].words / 4 + 256 * 4 - 1) / (256 * 4);
        if (blocks > 2048) blocks = 2048;
        if (blocks < 1) blocks = 1;
        p.r[i] = a.r[i];
        p.first_block[i] = total;
        total += (uint32_t)blocks;
    }
    for (int i = a.n; i <= N; ++i) p.first_block[i] = total;
    return (int)total;
}

#ifdef __HIPCC__
template <int N>
__device__ __forceinline__ void fill_pass(const FillPlan<N>& p, uint32_t block) {
    int i = 0;
    while (i + 1 < p.n && block >= p.first_block[i + 1]) ++i;  // (uniform: scalar loads of the arguments)
    const FillRegion r = p.r[i];
    const uint32_t blocks = p.first_block[i + 1] - p.first_block[i];
    const uint32_t local = block - p.first_block[i];
    const uint64_t vec = r.words / 4;
    uint4* p4 = reinterpret_cast<uint4*>(r.ptr);
    const uint4 v4 = make_uint4(r.value, r.value, r.value, r.value);
    const uint64_t stride = (uint64_t)blocks * blockDim.x;
    for (uint64_t j = (uint64_t)local * blockDim.x + threadIdx.x; j < vec; j += stride) p4[j] = v4;
    if (local == 0 && threadIdx.x < (r.words & 3)) r.ptr[vec * 4 + threadIdx.x] = r.value;
}
#endif

}  // namespace sessd
