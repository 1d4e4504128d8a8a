// pad_rows.h -- the rows of an output tensor beyond the active ones, for the gather-GEMM kernels on the matrix cores.
#pragma once

#include "kernels.h"

namespace sessd {

#ifdef __HIPCC__
// Rows n .. max_voxels - 1 <- epilogue(0), as the reference's zero fill followed by BN + ReLU.  `epi` holds the layer's
// scale and shift in LDS.
//
// Called behind a workgroup's last tile: loads and stores of a wave are counted together and in order, so that with these
// stores in front of the tile every first load of it waited for memory to take them (43 000 rows of 64 FP32 channels made
// a 29 us launch one of 39; the stores alone are 11 MB).  A lane writes 16 bytes of one column group, the same ones for
// all its rows.
template <typename T, int COUT, int THREADS>
__device__ __forceinline__ void write_pad_rows(T* __restrict__ out, int n, int max_voxels, const float* epi, bool has_scale,
                                               bool has_shift, int relu) {
    constexpr int kPer = 16 / (int)sizeof(T), kVecPerRow = COUT / kPer;
    static_assert(COUT % kPer == 0 && THREADS % kVecPerRow == 0, "a lane keeps its columns from row to row");
    const int c0 = ((int)threadIdx.x % kVecPerRow) * kPer;
    union {
        T t[kPer];
        uint4 v;
    } pad;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        float s = 0.f;
        if (has_scale) s = s * epi[c0 + e];
        if (has_shift) s = s + epi[COUT + c0 + e];
        if (relu) s = s > 0.f ? s : 0.f;
        if constexpr (sizeof(T) == 2) pad.t[e] = __float2half_rn(s);
        else pad.t[e] = s;
    }
    uint4* dst = reinterpret_cast<uint4*>(out + (size_t)n * COUT);
    const size_t total = (size_t)(max_voxels - n) * kVecPerRow;
    for (size_t i = (size_t)blockIdx.x * THREADS + threadIdx.x; i < total; i += (size_t)gridDim.x * THREADS) dst[i] = pad.v;
}
#endif

}  // namespace sessd
