// conv_tall.h -- the device side of conv_tall.hip, whose head says how it works and why: a workgroup's rows times all of W in LDS.  Its kernels
// have the launch to themselves (conv_tall.hip) or share it with a pass over coordinates (coord.hip).
#pragma once

#include <type_traits>

#include "pad_rows.h"

namespace sessd {

struct TallArgs {
    const int32_t* num_out = nullptr;
    const int32_t* nbr = nullptr;
    const void* in = nullptr;
    const void* w = nullptr;  // operand order (pack_weights())
    void* out = nullptr;
    const float* scale = nullptr;
    const float* shift = nullptr;
    int max_voxels = 0, relu = 0;
};
// Whether a layer's products can be made this way, and the arguments
bool tall_takes(const GemmArgs& a);
TallArgs tall_args(const GemmArgs& a);

#ifdef __HIPCC__
namespace tall {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned int v4u32 __attribute__((__vector_size__(16)));

constexpr int KC = 27;                  // kernel offsets: the 3x3x3 layers
constexpr int kSteps = (KC + 3) / 4;    // of four offsets
constexpr unsigned kOutOfRange = 0x80000000u;
constexpr int kRawBuffer = 0x00020000;
// steps whose rows are on their way (with 32 FP16 channels 3: the same times, 16 registers more)
constexpr int depth(int row_bytes) { return row_bytes == 64 ? 2 : 3; }

__device__ __forceinline__ void store4h(__half* dst, const float (&o)[4]) {
    union {
        __half2 h[2];
        uint2 u;
    } p;
    p.h[0] = __floats2half2_rn(o[0], o[1]);
    p.h[1] = __floats2half2_rn(o[2], o[3]);
    *reinterpret_cast<uint2*>(dst) = p.u;
}

// This wave's LDS accesses are done, and everybody else's.  (__syncthreads() would wait for the rows on their way as well.)
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): vmcnt and expcnt fields at their maximum = no wait
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ void store4(__half* dst, const float (&o)[4]) { store4h(dst, o); }
__device__ __forceinline__ void store4(float* dst, const float (&o)[4]) { *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]); }

// (COUT: columns of a workgroup, COLS: of the layer)
template <int CIN, int COUT, typename T, int WAVES, int COLS = COUT>
struct Lds {
    static constexpr int kOffsetBytes = CIN * COUT * (int)sizeof(T);
    static constexpr int kSums = WAVES * (COUT / 16) * 1024;  // of waves that share a block
    static constexpr int kWeights = kSteps * 4 * kOffsetBytes;  // (one offset more than there are, of zeros)
    static_assert(kSteps * 4 == KC + 1, "steps");
    alignas(16) unsigned char w[kWeights > kSums ? kWeights : kSums];
    float epi[2 * COLS];  // (scale and shift of all columns)
};

template <typename TO>
struct Tensors {
    __amdgpu_buffer_rsrc_t in, nbr;
    TO* out;
    unsigned stride4;  // bytes from offset to offset of the rulebook
    int n, relu;
    bool has_scale, has_shift;
};

// Where the neighbours of the lane's row are, at the lane's offset of steps first, first + BY, ... (-1: none)
template <int BY, typename TO>
__device__ __forceinline__ void ask_lists(const Tensors<TO>& t, int lane, int row0, int first, int (&idx)[kSteps]) {
    const int row = row0 + (lane & 15), q = lane >> 4;
#pragma unroll
    for (int m = 0; m < (kSteps + BY - 1) / BY; ++m) {
        const int k = 4 * (first + m * BY) + q;
        const bool some = k < KC && row < t.n;
        idx[m] = (int)__builtin_amdgcn_raw_buffer_load_b32(t.nbr, some ? (unsigned)k * t.stride4 + (unsigned)row * 4u : kOutOfRange, 0, 0);
        idx[m] = some ? idx[m] : -1;
    }
}

// Steps first, first + BY, ... of the block.  FP16: eight channels of four offsets an MFMA, one sum over all steps.  FP32: one channel of four
// offsets; a step is summed by itself, the channels of a piece apart, and the steps' sums two by two (in one chain over all steps 16 -> 16
// is 1.03e-7 from 64-bit sums at 41 489 rows, so 0.75e-7, on the pair lists of conv_wide.hip 0.80e-7).
template <int CIN, int COUT, typename T, int BY, typename TO>
__device__ __forceinline__ void multiply(const Tensors<TO>& t, int lane, const int (&idx)[kSteps], int first, const unsigned char* s_w, bool wait_for_w,
                                         v4f (&acc)[COUT / 16]) {
    constexpr bool kHalf = sizeof(T) == 2;
    constexpr int NB = COUT / 16, N = (kSteps + BY - 1) / BY, kPieces = CIN * (int)sizeof(T) / 16;  // (16 bytes of a row each)
    constexpr int kRowBytes = CIN * (int)sizeof(T);
    constexpr int kDepth = depth(kRowBytes) < N ? depth(kRowBytes) : N;
    constexpr int kSums = kHalf ? 1 : 4, kTotals = kHalf ? 1 : (CIN == 4 && COUT == 16 ? 4 : 2);
    const int i = lane & 15, q = lane >> 4;
    v4u32 x[kDepth][kPieces];
    auto request = [&](int m) {  // (m < N)
        const unsigned at = idx[m] >= 0 ? (unsigned)idx[m] * (unsigned)kRowBytes : kOutOfRange;
#pragma unroll
        for (int p = 0; p < kPieces; ++p) x[m % kDepth][p] = __builtin_amdgcn_raw_buffer_load_b128(t.in, at + p * 16u, 0, 0);
    };
#pragma unroll
    for (int m = 0; m < kDepth; ++m) request(m);
    if (wait_for_w) lds_barrier();
    v4f sum[kSums][NB], total[kTotals][NB];
    auto clear = [&](auto& sums) {
#pragma unroll
        for (int a = 0; a < (int)(sizeof(sums) / sizeof(sums[0])); ++a)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) sums[a][nb] = (v4f){0.f, 0.f, 0.f, 0.f};
    };
    clear(sum);
    clear(total);
    const unsigned char* w_at = s_w + (first * 4 + q) * (NB * kPieces * 256) + i * 16;
#pragma unroll
    for (int m = 0; m < N; ++m, w_at += BY * 4 * NB * kPieces * 256) {
        if (BY > 1 && first + m * BY >= kSteps) break;  // (uniform)
        // (the weights of a piece or two at a time: registers)
        constexpr int kAtOnce = NB > 2 || !kHalf || (CIN == 32 && NB == 1) ? 1 : 2;
        v4u32 w[2][kAtOnce][NB];
        auto weights = [&](int p, v4u32 (&to)[kAtOnce][NB]) {
#pragma unroll
            for (int a = 0; a < kAtOnce; ++a)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) to[a][nb] = *reinterpret_cast<const v4u32*>(w_at + (nb * kPieces + p + a) * 256);
        };
        weights(0, w[0]);
#pragma unroll
        for (int p = 0; p < kPieces; p += kAtOnce) {
            if (p + kAtOnce < kPieces) weights(p + kAtOnce, w[p / kAtOnce % 2 ^ 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < kAtOnce; ++a) {
                const v4u32 &row = x[m % kDepth][p + a];
                if constexpr (kHalf) {
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        sum[0][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w[p / kAtOnce % 2][a][nb]), __builtin_bit_cast(v8h, row), sum[0][nb], 0, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            sum[e][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[p / kAtOnce % 2][a][nb][e]), __uint_as_float(row[e]), sum[e][nb], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (m + kDepth < N) request(m + kDepth);
        if constexpr (!kHalf) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                total[m % kTotals][nb] += (sum[0][nb] + sum[1][nb]) + (sum[2][nb] + sum[3][nb]);
                asm volatile("" : "+v"(total[m % kTotals][nb]));  // (here: left to the compiler the steps' sums wait in registers for the end)
            }
            clear(sum);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if constexpr (kHalf) acc[nb] = sum[0][nb];
        else if constexpr (kTotals == 2) acc[nb] = total[0][nb] + total[1][nb];
        else acc[nb] = (total[0][nb] + total[1][nb]) + (total[2][nb] + total[3][nb]);
    }
}

// lane (i, q) holds output channels 16nb+4q .. +3 of row i
template <int COUT, int COLS, typename TO>
__device__ __forceinline__ void put(const Tensors<TO>& t, int lane, int row0, int col0, const v4f (&acc)[COUT / 16], const float* s_epi, const DenseTarget& dt) {
    constexpr int NB = COUT / 16;
    const int i = lane & 15, q = lane >> 4;
    const int row = row0 + i;
    if (row >= t.n) return;
    bool to_dense = false;
    TO* d = nullptr;
    size_t plane = 0;
    if (dt.dense) {  // the sparse2Dense scatter of this row, fused (uniform branch)
        const int4 cc = reinterpret_cast<const int4*>(dt.coors)[row];  // (b,z,y,x)
        if (cc.x != 0 || cc.y < 0 || cc.y >= dt.D || cc.z < 0 || cc.z >= dt.H || cc.w < 0 || cc.w >= dt.W) {
            if (dt.status && q == 0 && col0 == 0) atomicOr(dt.status, SESSD_STATUS_BAD_COORD);
        } else {
            to_dense = true;
            d = static_cast<TO*>(dt.dense) + ((size_t)cc.y * dt.Hp + cc.z + dt.pad_top) * dt.Wp + cc.w + dt.pad_left;
            plane = (size_t)dt.D * dt.Hp * dt.Wp;
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int c4 = col0 + nb * 16 + q * 4;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = acc[nb][e];
            if (t.has_scale) s = s * s_epi[c4 + e];
            if (t.has_shift) s = s + s_epi[COLS + c4 + e];
            if (t.relu) s = s > 0.f ? s : 0.f;
            o[e] = s;
        }
        store4(t.out + (size_t)row * COLS + c4, o);
        if (to_dense) {
#pragma unroll
            for (int e = 0; e < 4; ++e) d[(size_t)(c4 + e) * plane] = (TO)o[e];
        }
    }
}

// Workgroup `group` of `groups`, of WAVES waves that multiply columns col0 .. col0 + COUT - 1 and PADS that write the rows beyond the active ones.
template <int CIN, int COUT, typename T, typename TO, int WAVES, int PADS, int COLS = COUT>
__device__ __forceinline__ void workgroup(const TallArgs& g, const DenseTarget& dt, int group, int groups, Lds<CIN, COUT, T, WAVES, COLS>& lds, int col0 = 0) {
    static_assert(COLS == COUT || (CIN * sizeof(T) == 64 && PADS == 0), "columns apart: packed as they are multiplied");
    constexpr int NB = COUT / 16, kThreads = (WAVES + PADS) * 64;
    constexpr int kOffsetBytes = CIN * COUT * (int)sizeof(T), kVectors = KC * kOffsetBytes / 16, kCopies = (kVectors + kThreads - 1) / kThreads;
    unsigned char* const s_w = lds.w;
    float* const s_epi = lds.epi;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    v4f copy[kCopies];
#pragma unroll
    for (int c = 0; c < kCopies; ++c) {
        const int v = c * kThreads + tid;
        const int in_w = COLS == COUT ? v : (v / (NB * 64) * (COLS / 16) + col0 / 16) * 64 + v % (NB * 64);  // (offset by offset)
        copy[c] = reinterpret_cast<const v4f*>(g.w)[v < kVectors ? in_w : 0];
    }
    int n = *g.num_out;
    n = n < 0 ? 0 : (n > g.max_voxels ? g.max_voxels : n);
    float by = 1.f, plus = 0.f;
    if (tid < COLS) {
        if (g.scale) by = g.scale[tid];
        if (g.shift) plus = g.shift[tid];
    }
    // a workgroup's share: `per` blocks of 16 rows; the workgroups of an XCD (dealt round robin over eight) take neighbouring ones
    const int blocks = (n + 15) >> 4, per = (blocks + groups - 1) / groups;
    const int share = groups % 8 ? group : (group & 7) * (groups >> 3) + (group >> 3);
    const int begin = share * per < blocks ? share * per : blocks, end = begin + per < blocks ? begin + per : blocks;
    Tensors<TO> t;
    t.in = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.in), 0, (int)((size_t)g.max_voxels * CIN * sizeof(T)), kRawBuffer);
    t.nbr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(g.nbr), 0, (int)((size_t)KC * g.max_voxels * sizeof(int32_t)), kRawBuffer);
    t.out = static_cast<TO*>(g.out);
    t.stride4 = (unsigned)g.max_voxels * 4u;
    t.n = n;
    t.relu = g.relu;
    t.has_scale = g.scale != nullptr;
    t.has_shift = g.shift != nullptr;
    auto publish = [&]() {  // the weights and the epilogue's factors; the barrier that makes them visible follows
#pragma unroll
        for (int c = 0; c < kCopies; ++c) {
            const int v = c * kThreads + tid;
            if (v >= kVectors) continue;
            if constexpr (CIN * sizeof(T) == 64) {
                reinterpret_cast<v4f*>(s_w)[v] = copy[c];
            } else if constexpr (sizeof(T) == 2) {  // (packed four channels of a column at a time: here eight)
                const int in_block = v & 31, h = in_block >> 3, i = (in_block & 7) * 2;  // of a column block: channels 4h .., columns i, i + 1
                unsigned char* to = s_w + (v >> 5) * 512 + (h >> 1) * 256 + i * 16 + (h & 1) * 8;
                *reinterpret_cast<v2f*>(to) = (v2f){copy[c][0], copy[c][1]};
                *reinterpret_cast<v2f*>(to + 16) = (v2f){copy[c][2], copy[c][3]};
            } else {  // (packed a channel of a column at a time: here four)
                float* to = reinterpret_cast<float*>(s_w + (v >> 4) * 256) + (v & 3) * 16 + (v >> 2 & 3);  // column block v / 16: channel v / 4 % 4, columns 4 (v % 4) ..
#pragma unroll
                for (int e = 0; e < 4; ++e) to[e * 4] = copy[c][e];
            }
        }
        if (tid < kOffsetBytes / 16) reinterpret_cast<v4f*>(s_w)[kVectors + tid] = (v4f){0.f, 0.f, 0.f, 0.f};
        if (tid < COLS) {
            s_epi[tid] = by;
            s_epi[COLS + tid] = plus;
        }
    };
    // BY waves a block
    auto walk = [&](auto by_c) {
        constexpr int BY = decltype(by_c)::value;
        if (PADS && wave >= WAVES) {
            publish();
            lds_barrier();
            write_pad_rows<TO, COLS>(t.out, n, g.max_voxels, group * (PADS * 64) + (tid - WAVES * 64), groups * (PADS * 64), s_epi, t.has_scale,
                                     t.has_shift, t.relu);
            if (BY > 1) {  // (the barriers below)
                lds_barrier();
                lds_barrier();
            }
            return;
        }
        const int part = wave % BY;
        int idx[kSteps];
        const int first_block = begin + wave / BY;
        if (first_block < end) ask_lists<BY>(t, tid & 63, first_block * 16, part, idx);
        publish();  // (in front of the rounds: inside, what it needs stays in registers over all of them)
        if (first_block >= end) lds_barrier();
        bool first = true;
        for (int at = begin; first || at < end; at += WAVES / BY) {
            const int block = at + wave / BY, row0 = block * 16;
            const bool work = block < end;  // (uniform)
            int lane = tid & 63;
            asm volatile("" : "+v"(lane));  // (or what a round reads from LDS is read in front of the rounds, into registers)
            v4f acc[NB];
            if (work && !first) ask_lists<BY>(t, lane, row0, part, idx);
            if (work) multiply<CIN, COUT, T, BY>(t, lane, idx, part, s_w, first, acc);
            if constexpr (BY > 1) {  // (there is one round: a workgroup has at most WAVES / BY blocks)
                float4* const sums = reinterpret_cast<float4*>(s_w);
                lds_barrier();
                if (work && part)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) sums[(wave * NB + nb) * 64 + lane] = make_float4(acc[nb][0], acc[nb][1], acc[nb][2], acc[nb][3]);
                lds_barrier();
                if (work && part == 0)
#pragma unroll
                    for (int o = BY - 1; o > 0; --o)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) {
                            const float4 v = sums[((wave + o) * NB + nb) * 64 + lane];
                            acc[nb][0] += v.x;
                            acc[nb][1] += v.y;
                            acc[nb][2] += v.z;
                            acc[nb][3] += v.w;
                        }
            }
            if (work && part == 0) put<COUT, COLS>(t, lane, row0, col0, acc, s_epi, dt);
            first = false;
        }
    };
    if (per <= WAVES / 4) walk(std::integral_constant<int, 4>{});
    else if (per <= WAVES / 2) walk(std::integral_constant<int, 2>{});
    else walk(std::integral_constant<int, 1>{});
}

}  // namespace tall
#endif

}  // namespace sessd
