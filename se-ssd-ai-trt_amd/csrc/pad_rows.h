// pad_rows.h -- the rows of an output tensor beyond the active ones, for the gather-GEMM kernels on the matrix cores.
#pragma once

#include "kernels.h"

namespace sessd {

#ifdef __HIPCC__
// Rows n .. max_voxels - 1 <- epilogue(0), as the reference's zero fill followed by BN + ReLU.
//
// Loads and stores of a wave are counted together and in order, so that with these stores in front of a workgroup's tile every first
// load of it waited for memory to take them (43 000 rows of 64 FP32 channels, 11 MB, made a 29 us launch one of 39).  They are written
// behind the workgroup's last tile (write_pad_rows()), when nothing else is left to do, or, a KB at a time, by the waves that multiply
// (PadRows).  Which of them is for the kernels to choose (conv_wide.hip, conv_tile.hip): a launch without rows to write, or with few, must
// not pay for the steps.

// What a lane writes: 16 bytes of one column group, the same ones for all its rows.
template <typename T, int COUT>
struct PadRow {
    typedef unsigned int Words __attribute__((__vector_size__(16)));
    static constexpr int kPer = 16 / (int)sizeof(T), kBytes = COUT * (int)sizeof(T);  // elements of a lane, bytes of a row
    // `epi`: the layer's scale and shift in LDS
    static __device__ __forceinline__ Words vector(const float* epi, bool has_scale, bool has_shift, int relu) {
        const int c0 = (int)(threadIdx.x & (kBytes / 16 - 1)) * kPer;
        union {
            T t[kPer];
            Words v;
        } pad;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const float scale = epi[c0 + e], shift = epi[COUT + c0 + e];  // (read without branches: behind each was a trip to LDS of its own)
            float s = has_scale ? 0.f * scale : 0.f;
            s = has_shift ? s + shift : s;
            s = !relu || s > 0.f ? s : 0.f;
            if constexpr (sizeof(T) == 2) pad.t[e] = __float2half_rn(s);
            else pad.t[e] = s;
        }
        return pad.v;
    }
};

// Thread `thread` of `threads`.  (A wave beyond the end does nothing at all: 4 -> 16 at 50 000 rows, 2 000 to write, 9.8 -> 9.6 us)
template <typename T, int COUT>
__device__ __forceinline__ void write_pad_rows(T* __restrict__ out, int n, int max_voxels, unsigned thread, unsigned threads, const float* epi,
                                               bool has_scale, bool has_shift, int relu) {
    using Row = PadRow<T, COUT>;
    const size_t total = (size_t)(max_voxels - n) * (Row::kBytes / 16);
    if (thread >= total) return;
    const typename Row::Words v = Row::vector(epi, has_scale, has_shift, relu);
    typename Row::Words* dst = reinterpret_cast<typename Row::Words*>(out + (size_t)n * COUT);
    for (size_t i = thread; i < total; i += threads) dst[i] = v;
}

// A wave asks for a KB where it multiplies (step()), and memory has taken it by the time that the loads behind it are waited for.  What
// is left when its products are done follows then (rest()).  The addresses are the wave's own: the KBs first, first + waves, ...
template <typename T, int COUT>
class PadRows {
    using Row = PadRow<T, COUT>;
    static_assert(Row::kBytes <= 1024 && 1024 % Row::kBytes == 0, "a lane keeps its columns from KB to KB");
    __amdgpu_buffer_rsrc_t rows_;
    unsigned bytes_ = 0, at_ = 0, stride_, lane16_;  // (nothing is left before begin())
    typename Row::Words value_;

public:
    // whether a buffer descriptor and a 32-bit offset reach them
    static __device__ __forceinline__ bool reach(int n, int max_voxels) { return (size_t)(max_voxels - n) * Row::kBytes < 0x7ffffc00u; }
    // wave: of all `waves` that write (uniform)
    __device__ __forceinline__ void begin(T* out, int n, int max_voxels, unsigned wave, unsigned waves) {
        bytes_ = (unsigned)(max_voxels - n) * Row::kBytes;
        rows_ = __builtin_amdgcn_make_buffer_rsrc(out + (size_t)n * COUT, 0, (int)bytes_, 0x00020000);
        at_ = wave * 1024u;
        stride_ = waves * 1024u;
        lane16_ = (threadIdx.x & 63) * 16u;
    }
    __device__ __forceinline__ void layer(const float* epi, bool has_scale, bool has_shift, int relu) { value_ = Row::vector(epi, has_scale, has_shift, relu); }
    // (no branch: beyond the end the request points out of range and is dropped)
    __device__ __forceinline__ void step() {
        __builtin_amdgcn_raw_buffer_store_b128(value_, rows_, at_ + lane16_, 0, 0);
        at_ += at_ < bytes_ ? stride_ : 0u;
    }
    __device__ __forceinline__ bool left() const { return at_ < bytes_; }
    __device__ __forceinline__ void rest() {
        while (left()) step();
    }
};

// ... by nobody, or not here
struct NoPadRows {
    template <typename T>
    __device__ __forceinline__ void begin(T*, int, int, unsigned, unsigned) {}
    __device__ __forceinline__ void layer(const float*, bool, bool, int) {}
    __device__ __forceinline__ void step() {}
    __device__ __forceinline__ bool left() const { return false; }
    __device__ __forceinline__ void rest() {}
};
#endif

}  // namespace sessd
