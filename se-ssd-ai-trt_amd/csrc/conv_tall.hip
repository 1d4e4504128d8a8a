// conv_tall.hip -- gather-GEMM for FP16 3x3x3 layers with Cin 16 or 32: all of W in LDS, no barrier between the offsets.
//
//     out[o][:] = epilogue( sum_k  in[nbr[k][o]][:] @ W[k] )
//
// W is 14 to 110 KB and one workgroup a compute unit keeps all of it, so that its waves meet only once, in front of the first product.
//   * A workgroup owns a run of output rows, 16 at a time (a block) for each of its eight waves, and all columns; the accumulators stay
//     in registers over all offsets: no compaction, no partial tiles.  A row without a neighbour contributes a zero operand (a buffer
//     load that points out of range: zeros, no memory touched), so the matrix cores multiply about twice the useful pairs -- in FP16
//     they have the headroom.
//   * A step is four offsets.  Lane (i, q) of a wave requests all 32 or 64 bytes of the neighbour of row i at offset 4 step + q, and the inner
//     dimension of an MFMA is eight channels of each of the four offsets: the lane's own list entries are all that it needs, no other
//     lane's, and W is in LDS as the host has packed it (lane (i, q) reads the operand that holds these channels of W[4 step + q]).
//     Rows are requested two steps (eight offsets) ahead, with 16 channels three, all of them by straight-line code: the compiler's waits
//     are exact.
//   * With few rows (up to four blocks a workgroup, 16 384 rows on 256 units; up to two, 8 192) two or four waves share a block and take
//     every second or fourth step; their sums are added in LDS.
//   * W, the row count and, behind that, the lists are on their way together; the first rows are requested in front of the barrier.
//   * The rows beyond the active ones are written by four waves of their own.
// What bounds it from some 40 000 rows up are the requests for rows in four cache lookups a row (coalesced ones, with a 4 x 4
// transposition in registers, took longer: 49 874 rows 8.4 -> 9.5 us) and the reads of W from LDS (two blocks a wave: 8.4 -> 8.7), below
// the trips to memory: row count, lists, rows.
// Measured against the kernel with a barrier and 2 or 4 KB of W an offset that these layers ran on, launches back to back, 32 -> 32 and
// 32 -> 64: 801 rows 5.05 -> 3.5 us and 5.9 -> 4.8, 13 907 rows 5.3 -> 4.7 and 6.2 -> 6.25, 26 575 rows 7.1 -> 5.7 and 7.9 -> 7.3,
// 49 874 rows 11.2 -> 8.4 and 13.1 -> 10.9, 74 606 rows 13.9 -> 10.9 and 16.1 -> 13.4; frames of 60 000 points 229.6 -> 224.9.
// 16 -> 16 and 16 -> 32 against conv_wide.hip's pair lists (a quarter of the neighbours is there): 1 947 rows 5.0 -> 2.9 us and 5.2 -> 3.2,
// 16 198 rows 7.2 -> 3.3 and 8.1 -> 3.7, 60 000 rows 10.4 -> 4.9 and 11.9 -> 5.8; frames of 60 000 points 225.9 -> 215.7.
// The waves are eight because the coordinate passes beside them need registers (12: the same times, and 504 of 512 taken).
// Summation order per output element: a wave's steps ascending, in a step the channels eight at a time; where waves share a block, to the
// first one's sum those of the others, the last one's first.  Fixed for a row count and a grid, run-to-run identical; in a launch with more or
// fewer rows, or on another number of compute units, the same row may be summed in another of the three orders.
// (The ring of conv_tile.hip, faster from 64 channels up, has too little work per row here.)
#include <type_traits>

#include "pad_rows.h"

namespace sessd {

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned int v4u32 __attribute__((__vector_size__(16)));

constexpr int kWaves = 8;     // that multiply
constexpr int kPadWaves = 4;  // that write the rows beyond the active ones
constexpr int KC = 27;                  // kernel offsets: the 3x3x3 layers
constexpr int kSteps = (KC + 3) / 4;    // of four offsets
constexpr unsigned kOutOfRange = 0x80000000u;
constexpr int kRawBuffer = 0x00020000;
// steps whose rows are on their way (with 32 channels 3: the same times, 16 registers more)
constexpr int depth(int cin) { return cin == 32 ? 2 : 3; }

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

struct Tensors {
    __amdgpu_buffer_rsrc_t in, nbr;
    __half* out;
    unsigned stride4;  // bytes from offset to offset of the rulebook
    int n, relu;
    bool has_scale, has_shift;
};

// Where the neighbours of the lane's row are, at the lane's offset of steps first, first + BY, ... (-1: none)
template <int BY>
__device__ __forceinline__ void ask_lists(const Tensors& t, int lane, int row0, int first, int (&idx)[kSteps]) {
    const int row = row0 + (lane & 15), q = lane >> 4;
#pragma unroll
    for (int m = 0; m < (kSteps + BY - 1) / BY; ++m) {
        const int k = 4 * (first + m * BY) + q;
        const bool some = k < KC && row < t.n;
        idx[m] = (int)__builtin_amdgcn_raw_buffer_load_b32(t.nbr, some ? (unsigned)k * t.stride4 + (unsigned)row * 4u : kOutOfRange, 0, 0);
        idx[m] = some ? idx[m] : -1;
    }
}

// Steps first, first + BY, ... of the block
template <int CIN, int COUT, int BY>
__device__ __forceinline__ void multiply(const Tensors& t, int lane, const int (&idx)[kSteps], int first, const unsigned char* s_w, bool wait_for_w,
                                         v4f (&acc)[COUT / 16]) {
    constexpr int NB = COUT / 16, N = (kSteps + BY - 1) / BY, kPieces = CIN / 8;  // (16 bytes of a row each)
    constexpr int kDepth = depth(CIN) < N ? depth(CIN) : N;
    const int i = lane & 15, q = lane >> 4;
    v4u32 x[kDepth][kPieces];
    auto request = [&](int m) {  // (m < N)
        const unsigned at = idx[m] >= 0 ? (unsigned)idx[m] * (unsigned)(CIN * sizeof(__half)) : kOutOfRange;
#pragma unroll
        for (int p = 0; p < kPieces; ++p) x[m % kDepth][p] = __builtin_amdgcn_raw_buffer_load_b128(t.in, at + p * 16u, 0, 0);
    };
#pragma unroll
    for (int m = 0; m < kDepth; ++m) request(m);
    if (wait_for_w) lds_barrier();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = (v4f){0.f, 0.f, 0.f, 0.f};
    const unsigned char* w_at = s_w + (first * 4 + q) * (NB * kPieces * 256) + i * 16;
#pragma unroll
    for (int m = 0; m < N; ++m, w_at += BY * 4 * NB * kPieces * 256) {
        if (BY > 1 && first + m * BY >= kSteps) break;  // (uniform)
        // (the weights of a piece or two at a time: registers)
        constexpr int kAtOnce = NB > 2 ? 1 : 2;
        v8h w[2][kAtOnce][NB];
        auto weights = [&](int p, v8h (&to)[kAtOnce][NB]) {
#pragma unroll
            for (int a = 0; a < kAtOnce; ++a)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) to[a][nb] = *reinterpret_cast<const v8h*>(w_at + (nb * kPieces + p + a) * 256);
        };
        weights(0, w[0]);
#pragma unroll
        for (int p = 0; p < kPieces; p += kAtOnce) {
            if (p + kAtOnce < kPieces) weights(p + kAtOnce, w[p / kAtOnce % 2 ^ 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < kAtOnce; ++a)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[p / kAtOnce % 2][a][nb], __builtin_bit_cast(v8h, x[m % kDepth][p + a]), acc[nb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (m + kDepth < N) request(m + kDepth);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// lane (i, q) holds output channels 16nb+4q .. +3 of row i
template <int COUT>
__device__ __forceinline__ void put(const Tensors& t, int lane, int row0, const v4f (&acc)[COUT / 16], const float* s_epi, const DenseTarget& dt) {
    constexpr int NB = COUT / 16;
    const int i = lane & 15, q = lane >> 4;
    const int row = row0 + i;
    if (row >= t.n) return;
    bool to_dense = false;
    __half* d = nullptr;
    size_t plane = 0;
    if (dt.dense) {  // the sparse2Dense scatter of this row, fused (uniform branch)
        const int4 cc = reinterpret_cast<const int4*>(dt.coors)[row];  // (b,z,y,x)
        if (cc.x != 0 || cc.y < 0 || cc.y >= dt.D || cc.z < 0 || cc.z >= dt.H || cc.w < 0 || cc.w >= dt.W) {
            if (dt.status && q == 0) atomicOr(dt.status, SESSD_STATUS_BAD_COORD);
        } else {
            to_dense = true;
            d = static_cast<__half*>(dt.dense) + ((size_t)cc.y * dt.Hp + cc.z + dt.pad_top) * dt.Wp + cc.w + dt.pad_left;
            plane = (size_t)dt.D * dt.Hp * dt.Wp;
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int c4 = nb * 16 + q * 4;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = acc[nb][e];
            if (t.has_scale) s = s * s_epi[c4 + e];
            if (t.has_shift) s = s + s_epi[COUT + c4 + e];
            if (t.relu) s = s > 0.f ? s : 0.f;
            o[e] = s;
        }
        store4h(t.out + (size_t)row * COUT + c4, o);
        if (to_dense) {
#pragma unroll
            for (int e = 0; e < 4; ++e) d[(size_t)(c4 + e) * plane] = __float2half_rn(o[e]);
        }
    }
}

template <int CIN, int COUT, bool PAD>
__global__ void __launch_bounds__((kWaves + (PAD ? kPadWaves : 0)) * 64)
conv_tall(const int32_t* __restrict__ num_out, const int32_t* __restrict__ nbr, const __half* __restrict__ in,
          const void* __restrict__ Wp, int max_voxels, int relu, __half* __restrict__ out,
          const float* __restrict__ scale, const float* __restrict__ shift, DenseTarget dt) {
    constexpr int NB = COUT / 16, kThreads = (kWaves + (PAD ? kPadWaves : 0)) * 64;
    constexpr int kOffsetBytes = CIN * COUT * 2, kVectors = KC * kOffsetBytes / 16, kCopies = (kVectors + kThreads - 1) / kThreads;
    // (one offset more than there are, of zeros)
    __shared__ __align__(16) unsigned char s_w[kSteps * 4 * kOffsetBytes];
    __shared__ float s_epi[2 * COUT];
    static_assert(kSteps * 4 == KC + 1 && sizeof(s_w) >= kWaves * NB * 1024, "steps; the sums of waves that share a block");
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    v4f copy[kCopies];
#pragma unroll
    for (int c = 0; c < kCopies; ++c) {
        const int v = c * kThreads + tid;
        copy[c] = reinterpret_cast<const v4f*>(Wp)[v < kVectors ? v : 0];
    }
    int n = *num_out;
    n = n < 0 ? 0 : (n > max_voxels ? max_voxels : n);
    float by = 1.f, plus = 0.f;
    if (tid < COUT) {
        if (scale) by = scale[tid];
        if (shift) plus = shift[tid];
    }
    // a workgroup's share: `per` blocks of 16 rows; the workgroups of an XCD (dealt round robin over eight) take neighbouring ones
    const int blocks = (n + 15) >> 4, groups = gridDim.x, per = (blocks + groups - 1) / groups;
    const int share = groups % 8 ? (int)blockIdx.x : (int)(blockIdx.x & 7) * (groups >> 3) + (int)(blockIdx.x >> 3);
    const int begin = share * per < blocks ? share * per : blocks, end = begin + per < blocks ? begin + per : blocks;
    Tensors t;
    t.in = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half*>(in), 0, (int)((size_t)max_voxels * CIN * sizeof(__half)), kRawBuffer);
    t.nbr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(nbr), 0, (int)((size_t)KC * max_voxels * sizeof(int32_t)), kRawBuffer);
    t.out = out;
    t.stride4 = (unsigned)max_voxels * 4u;
    t.n = n;
    t.relu = relu;
    t.has_scale = scale != nullptr;
    t.has_shift = shift != nullptr;
    auto publish = [&]() {  // the weights and the epilogue's factors; the barrier that makes them visible follows
#pragma unroll
        for (int c = 0; c < kCopies; ++c) {
            const int v = c * kThreads + tid;
            if (v >= kVectors) continue;
            if constexpr (CIN == 32) {
                reinterpret_cast<v4f*>(s_w)[v] = copy[c];
            } else {  // (packed four channels of a column at a time: here eight)
                const int in_block = v & 31, g = in_block >> 3, i = (in_block & 7) * 2;  // of a column block: channels 4g .., columns i, i + 1
                unsigned char* to = s_w + (v >> 5) * 512 + (g >> 1) * 256 + i * 16 + (g & 1) * 8;
                *reinterpret_cast<v2f*>(to) = (v2f){copy[c][0], copy[c][1]};
                *reinterpret_cast<v2f*>(to + 16) = (v2f){copy[c][2], copy[c][3]};
            }
        }
        if (tid < kOffsetBytes / 16) reinterpret_cast<v4f*>(s_w)[kVectors + tid] = (v4f){0.f, 0.f, 0.f, 0.f};
        if (tid < COUT) {
            s_epi[tid] = by;
            s_epi[COUT + tid] = plus;
        }
    };
    // BY waves a block
    auto walk = [&](auto by_c) {
        constexpr int BY = decltype(by_c)::value;
        if (PAD && wave >= kWaves) {
            publish();
            lds_barrier();
            write_pad_rows<__half, COUT>(out, n, max_voxels, blockIdx.x * (kPadWaves * 64) + (tid - kWaves * 64), gridDim.x * (kPadWaves * 64), s_epi, t.has_scale,
                                         t.has_shift, relu);
            if (BY > 1) {  // (the barriers below)
                lds_barrier();
                lds_barrier();
            }
            return;
        }
        const int part = wave % BY;
        bool first = true;
        for (int at = begin; first || at < end; at += kWaves / BY) {
            const int block = at + wave / BY, row0 = block * 16;
            const bool work = block < end;  // (uniform)
            int lane = tid & 63;
            asm volatile("" : "+v"(lane));  // (or what a round reads from LDS is read in front of the rounds, into registers)
            int idx[kSteps];
            v4f acc[NB];
            if (work) ask_lists<BY>(t, lane, row0, part, idx);
            if (first) {
                publish();
                if (!work) lds_barrier();
            }
            if (work) multiply<CIN, COUT, BY>(t, lane, idx, part, s_w, first, acc);
            if constexpr (BY > 1) {  // (there is one round: a workgroup has at most kWaves / BY blocks)
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
            if (work && part == 0) put<COUT>(t, lane, row0, acc, s_epi, dt);
            first = false;
        }
    };
    if (per <= kWaves / 4) walk(std::integral_constant<int, 4>{});
    else if (per <= kWaves / 2) walk(std::integral_constant<int, 2>{});
    else walk(std::integral_constant<int, 1>{});
}

template <int CIN, int COUT>
int launch(const GemmArgs& a, hipStream_t stream) {
    if ((size_t)a.max_voxels * CIN * sizeof(__half) >= kOutOfRange) return SESSD_E_UNSUPPORTED;
    if ((size_t)a.max_voxels * (KC * sizeof(int32_t)) >= kOutOfRange) return SESSD_E_UNSUPPORTED;
    auto go = [&](auto pad) {
        hipLaunchKernelGGL((conv_tall<CIN, COUT, decltype(pad)::value>), dim3(gemm_compute_units()),
                           dim3((kWaves + (decltype(pad)::value ? kPadWaves : 0)) * 64), 0, stream, a.num_out, a.nbr,
                           static_cast<const __half*>(a.in_feat), a.w_packed, a.max_voxels, a.relu, static_cast<__half*>(a.out_feat), a.scale,
                           a.shift, a.dense);
    };
    a.write_pad_rows ? go(std::true_type{}) : go(std::false_type{});
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

}  // namespace

bool gemm_runs_tall(int K, int cin, int cout) { return K == KC && ((cin == 32 && (cout == 64 || cout == 32)) || (cin == 16 && (cout == 16 || cout == 32))); }

int launch_tall(const GemmArgs& a, hipStream_t stream) {
    // (FP32 layers stay on the pair lists: 4 -> 16 and 16 -> 16 are faster this way, at 16 198 rows 5.8 -> 3.6 and 6.6 -> 5.4 us, but what the
    // lists leave of a unit is what the coordinate passes of a frame run in: 20 000 points 263.0 -> 264.9 us, 80 000 408 -> 415)
    // (0 x infinity: with weights that are not finite an absent neighbour may not be a row of zeros)
    if (!a.w_packed || !a.halves_finite || a.K != KC || a.in_type != SESSD_HALF || a.out_type != SESSD_HALF) return SESSD_E_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(a.in_feat) | reinterpret_cast<uintptr_t>(a.out_feat)) & 15) return SESSD_E_UNSUPPORTED;
    if (a.cin == 32 && a.cout == 64) return launch<32, 64>(a, stream);
    if (a.cin == 32 && a.cout == 32) return launch<32, 32>(a, stream);
    if (a.cin == 16 && a.cout == 16) return launch<16, 16>(a, stream);
    if (a.cin == 16 && a.cout == 32) return launch<16, 32>(a, stream);
    return SESSD_E_UNSUPPORTED;
}

}  // namespace sessd
