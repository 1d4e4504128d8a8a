// pad_rows.h -- the rows of an output tensor beyond the active ones, for the gather-GEMM kernels on the matrix cores.
#pragma once

#include "kernels.h"

namespace sessd {

#ifdef __HIPCC__
// Rows n .. max_voxels - 1 <- epilogue(0), as the reference's zero fill followed by BN + ReLU.
//
// Loads and stores of a wave are counted together and in order, so that with these stores in front of a workgroup's tile every first
// load of it waited for memory to take them (43 000 rows of 64 FP32 channels, 11 MB, made a 29 us launch one of 39), and behind its last
// one nothing else was left to do meanwhile.  A wave writes 1 KB at a time instead, and asks for that where it multiplies (step()): memory
// has taken it by the time that the loads behind it are waited for.  What is left when its products are done follows then (rest()).
// The addresses are the wave's own: the KBs first, first + waves, ...
// (Calls that write 60 000 - 160 000 rows: SubM 64 -> 64 FP32 with its rulebook 34.99 -> 34.31 us, 128 -> 128 FP16 29.84 -> 29.18, strided 32 -> 64
// FP16 35.45 -> 34.53, a frame of 20 000 points 314.5 -> 309.7.)
template <typename T, int COUT>
class PadRows {
    typedef unsigned int Words __attribute__((__vector_size__(16)));
    static constexpr int kPer = 16 / (int)sizeof(T), kRow = COUT * (int)sizeof(T);
    static constexpr unsigned kMost = 0x7ffffc00u;  // bytes that a buffer descriptor and a 32-bit offset reach; rest() writes more
    static_assert(kRow <= 1024 && 1024 % kRow == 0, "a lane keeps its columns from KB to KB");
    __amdgpu_buffer_rsrc_t rows_;
    T* begin_;
    size_t total_;
    unsigned bytes_, first_, at_, stride_, lane16_;
    Words value_;

public:
    // wave: of all `waves` that write (uniform)
    __device__ __forceinline__ PadRows(T* out, int n, int max_voxels, unsigned wave, unsigned waves) {
        begin_ = out + (size_t)n * COUT;
        total_ = (size_t)(max_voxels - n) * kRow;
        bytes_ = total_ < kMost ? (unsigned)total_ : kMost;
        rows_ = __builtin_amdgcn_make_buffer_rsrc(begin_, 0, (int)bytes_, 0x00020000);
        first_ = at_ = wave * 1024u;
        stride_ = waves * 1024u;
        lane16_ = (threadIdx.x & 63) * 16u;
    }
    // `epi`: the layer's scale and shift in LDS
    __device__ __forceinline__ void layer(const float* epi, bool has_scale, bool has_shift, int relu) {
        const int c0 = (int)(threadIdx.x & (kRow / 16 - 1)) * kPer;
        union {
            T t[kPer];
            Words v;
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
        value_ = pad.v;
    }
    // (no branch: beyond the end the request points out of range and is dropped)
    __device__ __forceinline__ void step() {
        __builtin_amdgcn_raw_buffer_store_b128(value_, rows_, at_ + lane16_, 0, 0);
        at_ += at_ < bytes_ ? stride_ : 0u;
    }
    __device__ __forceinline__ bool left() const { return at_ < bytes_; }
    __device__ __forceinline__ void rest() {
        while (left()) step();
        // (bytes that step() does not reach)
        for (size_t at = (size_t)kMost + first_ + lane16_; at < total_; at += stride_) *reinterpret_cast<Words*>(begin_ + at / sizeof(T)) = value_;
    }
};

// ... in a launch that leaves those rows alone
struct NoPadRows {
    __device__ __forceinline__ void layer(const float*, bool, bool, int) {}
    __device__ __forceinline__ void step() {}
    __device__ __forceinline__ bool left() const { return false; }
    __device__ __forceinline__ void rest() {}
};
#endif

}  // namespace sessd
