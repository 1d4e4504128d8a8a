// conv_tile.hip -- gather-GEMM for FP16 layers with Cin and Cout of 64 or 128: one tile of output rows per compute unit,
// rows and weights through a ring of LDS buffers that memory fills directly.
//
//     out[o][:] = epilogue( sum_k  in[nbr[k][o]][:] @ W[k] )
//
// The layer is a dense product of the tile's rows with all K * Cin / 32 slices of W: a row without a neighbour at offset
// k contributes zeros (a request that points out of range: zeros arrive in LDS, no memory is touched), so the matrix
// cores multiply about twice the useful pairs -- in FP16 they have the headroom -- and the accumulators stay in registers
// from the first slice to the last: no compaction, no partial tiles, no reduction.
//   * A workgroup owns U * mf rows and all columns.  Four of its waves multiply: 16 mf rows and 64 columns each (Cout 128:
//     two waves deep, two wide; Cout 64: four deep).  mf is chosen on the device so that the launch is one round of tiles
//     over the compute units where that is possible: the weights, at 128 -> 128 with 884 KB more than the rows, are then
//     read once per unit.
//   * Four waves load, and do nothing else: a multiplying wave that also requests stalls on the requests' queue, and its
//     matrix core with it (128 -> 128 at 40 422 rows: 44.5 us, with loaders of their own 38.9).
//   * The inner dimension is walked in stages of 64 channels of one offset.  A stage's rows (128 bytes, a whole cache line;
//     eight lanes to a row) and its slice of W (host-packed in MFMA operand order) go into one of R buffers with buffer
//     loads that write LDS: no registers, one request per row and stage for the whole workgroup.  One barrier a stage:
//     at it the next stage is complete and the one in use has been read.
//   * The multiplying waves read their fragments one slice ahead, one LDS read behind each MFMA: reads in a row cost the
//     matrix core their issue time (measured on LDS alone: 993 cycles a stage for 640 of MFMAs, interleaved 710).
//   * A row's eight 16-byte pieces are stored rotated by its number (piece c of row r at c ^ (r / 2 % 8)), which lane
//     fetches which piece: the 16 rows of a fragment read lie in different banks (no conflicts counted).
//   * Tiles are dealt so that the workgroups of an XCD (dealt round robin over eight) take neighbouring ones.
// All vector-memory requests of a loading wave are of this one kind and are counted by hand (s_waitcnt vmcnt in issue
// order).  Summation order per output element: offsets ascending, channels inside the MFMA: fixed, run-to-run identical.
//
// Measured against a kernel with its operands in registers (64 or 128 rows, W read once for them), launches back to back: 128 -> 128 at 40 422 rows 47.0
// -> 34.2 us (1.05 PFLOP/s with the padding pairs; a large FP16 matrix product of the library reaches 1.13: under this
// load the clock falls to 1.4 .. 1.8 GHz), at 19 825 rows 37.9 -> 21.5, at 2 833 rows 21.5 -> 12.3; 64 -> 64 at 72 854 rows
// 29.9 -> 24.4, at 26 247 rows 14.9 -> 11.7, at 3 060 rows 9.0 -> 8.5.  Beyond 40 960 rows (Cout 128) the loads bound it.
#include <type_traits>

#include "pad_rows.h"

namespace sessd {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;    // that multiply
constexpr int kLoaders = 4;  // that fetch
constexpr int kThreads = (kWaves + kLoaders) * 64;
constexpr int kMaxRing = 4;  // (8 buffers where they fit: the same times)
constexpr unsigned kOutOfRange = 0x80000000u;
constexpr int kRawBuffer = 0x00020000;  // descriptor word 3: raw 32-bit data format, no swizzle
constexpr int kPool = 160 * 1024 - 2048;  // LDS for the row lists and the ring

template <int CIN, int COUT, int KC>
struct Shape {
    static constexpr int WN = COUT >= 128 ? 2 : 1;    // waves across the columns
    static constexpr int WM = kWaves / WN;            // ... and down the rows
    static constexpr int NB = COUT / 16 / WN;         // 16-column blocks of a wave
    static constexpr int U = WM * 16;                 // rows per unit of mf
    static constexpr int G = CIN / 64;                // stages per offset
    static constexpr int S = KC * G;                  // stages
    static constexpr int kWeightBytes = COUT * 128;   // ... of a stage
    static constexpr int stage_bytes(int mf) { return U * mf * 128 + kWeightBytes; }
    static constexpr int rows(int mf) { return U * mf / kLoaders; }  // that a loader fetches
    static constexpr int lists(int mf) { return (rows(mf) + 63) / 64; }       // its requests for an offset's neighbours
    static constexpr int requests(int mf) { return rows(mf) / 8 + COUT / 8 / kLoaders + lists(mf); }  // ... in a stage
    // an offset's neighbours are asked for so many offsets early that the wait for a stage covers them
    static constexpr int ahead(int ring) { return (ring - 1) / G + 3; }
    static constexpr int list_bytes(int mf, int ring) { return ahead(ring) * kLoaders * lists(mf) * 256; }
    static constexpr int ring(int mf) {
        int r = kMaxRing;
        while (r * stage_bytes(mf) + list_bytes(mf, r) > kPool || (r - 1) * requests(mf) > 63) --r;
        return r;
    }
    static constexpr int kMaxMf = COUT >= 128 ? 6 : 5;  // where the ring still has three buffers
};

__device__ __forceinline__ v4i make_rsrc(const void* p, unsigned bytes) {
    const unsigned long long a = (unsigned long long)p;
    v4i r;
    r.x = __builtin_amdgcn_readfirstlane((int)(a & 0xffffffffull));
    r.y = __builtin_amdgcn_readfirstlane((int)((a >> 32) & 0xffffull));
    r.z = __builtin_amdgcn_readfirstlane((int)bytes);
    r.w = kRawBuffer;
    return r;
}

// 16 bytes per lane from r[voff] to LDS bytes lds + 16 * lane.  (Written out: the compiler would wait for every such load
// before any LDS read that it cannot tell apart from its destination.  The compiler writes m0 itself; the nop is the wait
// state that a load to LDS needs behind that.)
__device__ __forceinline__ void load_to_lds(const v4i& r, unsigned voff, unsigned lds) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r) : "memory");
}
// 4 bytes per lane to lds + 4 * lane
__device__ __forceinline__ void load4_to_lds(const v4i& r, unsigned voff, unsigned lds) {
    asm volatile("s_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {  // all but the N youngest have arrived
    static_assert(N >= 0 && N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// this wave's LDS reads are done and everybody else's too
__device__ __forceinline__ void stage_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ void store4h(__half* dst, const float (&o)[4]) {
    union {
        __half2 h[2];
        uint2 u;
    } p;
    p.h[0] = __floats2half2_rn(o[0], o[1]);
    p.h[1] = __floats2half2_rn(o[2], o[3]);
    *reinterpret_cast<uint2*>(dst) = p.u;
}

template <int CIN, int COUT, int KC, int MF, typename Pads>
__device__ __forceinline__ void run_tile(const v4i& rs_in, const v4i& rs_w, const v4i& rs_nbr, unsigned nbr_stride,
                                         __half* __restrict__ out, int row0, int row_end, bool has_scale, bool has_shift, int relu,
                                         const DenseTarget& dt, unsigned char* pool, const float* s_epi, Pads& pads) {
    using C = Shape<CIN, COUT, KC>;
    constexpr int H = C::U * MF;
    constexpr int R = C::ring(MF);
    static_assert(R >= 3, "the ring needs a stage in use, one complete and one in flight");
    constexpr int NW = COUT / 8 / kLoaders;   // weight requests of a loader and stage (1 KB each)
    constexpr int NA = C::rows(MF) / 8;       // row requests (8 rows each)
    constexpr int NL = C::lists(MF);          // neighbour requests
    constexpr int D = NA + NW + NL;
    constexpr int P = C::ahead(R);
    static_assert(H % (8 * kLoaders) == 0 && COUT % (8 * kLoaders) == 0, "whole requests");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned char* ring = pool + C::list_bytes(MF, R);

    if (wave >= kWaves) {
        const int w = wave - kWaves;
        const unsigned pool_at = __builtin_amdgcn_readfirstlane(
            (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)pool);
        // the neighbours of this loader's rows: [P offsets][NL * 64], row w * 8 + e / 8 * 8 kLoaders + e % 8 at e
        const int* const lists = reinterpret_cast<const int*>(pool) + w * (P * NL * 64);
        const unsigned lists_at = pool_at + (unsigned)w * (P * NL * 256u);
        unsigned n_off = (unsigned)(row0 + w * 8 + (lane >> 3) * (8 * kLoaders) + (lane & 7)) * 4u;
        auto request_list = [&](unsigned slot) {
#pragma unroll
            for (int j = 0; j < NL; ++j) load4_to_lds(rs_nbr, n_off + j * (8 * 8 * kLoaders * 4u), lists_at + slot + j * 256u);
        };
#pragma unroll
        for (int k = 0; k < P; ++k) {
            request_list(k * (NL * 256u));
            n_off += nbr_stride;
        }
        wait_loads<0>();
        // lane l fetches for row l / 8 of its group of eight the piece that belongs at position l % 8
        const unsigned piece = ((lane & 7) ^ ((w & 1) * 4 + (lane >> 4))) * 16;
        unsigned row[NA], nxt[NA];
        auto look = [&](int slot, unsigned (&r)[NA]) {  // byte offsets of the neighbours' rows, or out of range
#pragma unroll
            for (int j = 0; j < NA; ++j) {
                const int idx = lists[slot + j * 8 + (lane >> 3)];
                r[j] = idx >= 0 ? (unsigned)idx * (unsigned)(CIN * 2) + piece : kOutOfRange;
            }
        };
        look(0, row);
        look(NL * 64, nxt);
        int at_list = 2 * NL * 64;   // of the offset behind nxt's
        unsigned to_list = 0;        // where the next list goes
        unsigned w_off = (unsigned)w * 1024u + lane * 16u;
        const unsigned ring_at = pool_at + C::list_bytes(MF, R) + w * 1024u;
        unsigned at = ring_at;
        // the requests of the next stage, which is part g of its offset (beyond the last offset they mean nothing)
        auto request = [&](int g) {
            request_list(to_list);
#pragma unroll
            for (int j = 0; j < NA; ++j) load_to_lds(rs_in, row[j] + (unsigned)g * 128u, at + j * (1024u * kLoaders));
#pragma unroll
            for (int j = 0; j < NW; ++j) load_to_lds(rs_w, w_off + j * (1024u * kLoaders), at + H * 128u + j * (1024u * kLoaders));
            w_off += C::kWeightBytes;
            at += C::stage_bytes(MF);
            at = at >= ring_at + (unsigned)(R * C::stage_bytes(MF)) ? ring_at : at;
            if (g == C::G - 1) {
#pragma unroll
                for (int j = 0; j < NA; ++j) row[j] = nxt[j];
                look(at_list, nxt);
                at_list = at_list == (P - 1) * NL * 64 ? 0 : at_list + NL * 64;
                to_list = to_list == (P - 1) * NL * 256u ? 0u : to_list + NL * 256u;
                n_off += nbr_stride;
            }
        };
#pragma unroll
        for (int s = 0; s < R; ++s) request(s % C::G);
        wait_loads<(R - 1) * D>();
        stage_barrier();
        for (int k = 0; k < KC; ++k) {
#pragma unroll
            for (int g = 0; g < C::G; ++g) {
                wait_loads<(R - 2) * D>();
                stage_barrier();
                request((g + R) % C::G);
            }
        }
        wait_loads<0>();
        __syncthreads();  // the next tile reuses the lists and the ring
        return;
    }

    const int wm = wave / C::WN, wn = wave % C::WN;
    const int i = lane & 15, q = lane >> 4;
    const unsigned char* frag_rows = ring + (wm * MF * 16 + i) * 128;
    const unsigned char* frag_w = ring + H * 128 + wn * C::NB * 1024 + lane * 16;
    const int piece_at[2] = {(q ^ (i >> 1)) << 4, ((4 + q) ^ (i >> 1)) << 4};
    struct Frags {
        v8h a[MF], w[C::NB];
    };
    auto read = [&](int at, int h, Frags& f) {
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) f.w[nb] = *reinterpret_cast<const v8h*>(frag_w + at + h * (COUT * 64) + nb * 1024);
#pragma unroll
        for (int b = 0; b < MF; ++b) f.a[b] = *reinterpret_cast<const v8h*>(frag_rows + at + piece_at[h] + b * 2048);
    };
    v4f acc[MF][C::NB];
#pragma unroll
    for (int b = 0; b < MF; ++b)
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) acc[b][nb] = (v4f){0.f, 0.f, 0.f, 0.f};
    // multiplies what is in `use` while slice h of the stage at `at` is read into `fill`: one LDS read behind each MFMA,
    // where it costs no time of the matrix core (all reads first: 1.4 times the time)
    auto step = [&](const Frags& use, Frags& fill, int at, int h) {
        read(at, h, fill);
#pragma unroll
        for (int b = 0; b < MF; ++b)
#pragma unroll
            for (int nb = 0; nb < C::NB; ++nb) acc[b][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(use.w[nb], use.a[b], acc[b][nb], 0, 0, 0);
        constexpr int kReads = MF + C::NB, kMfmas = MF * C::NB;
#pragma unroll
        for (int j = 0; j < kReads; ++j) {
            if (j < kMfmas) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if (kMfmas > kReads) __builtin_amdgcn_sched_group_barrier(0x008, kMfmas - kReads, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    Frags f0, f1;
    int at = 0;  // the stage in use
    stage_barrier();
    read(0, 0, f0);
    auto stage = [&](auto with_pads) {
        step(f0, f1, at, 1);
        if constexpr (decltype(with_pads)::value) pads.step();  // (these waves wait for no other request in the loop)
        stage_barrier();  // the stage in use is read, the next one complete
        at += C::stage_bytes(MF);
        at = at == R * C::stage_bytes(MF) ? 0 : at;
        step(f1, f0, at, 0);
    };
    int s = 0;
    if constexpr (KC > 3)  // (three offsets are unrolled, and the registers full)
        if (pads.left()) {
            pads.layer(s_epi, has_scale, has_shift, relu);
            for (; s < C::S && pads.left(); ++s) stage(std::true_type{});
        }
    for (; s < C::S; ++s) stage(std::false_type{});

    // epilogue: lane (i, q) holds output channels 16nb+4q .. +3 of row i of each of its blocks
#pragma unroll
    for (int b = 0; b < MF; ++b) {
        const int row = row0 + (wm * MF + b) * 16 + i;
        if (row >= row_end) continue;
        bool to_dense = false;
        __half* d = nullptr;
        size_t plane = 0;
        if (dt.dense) {  // the sparse2Dense scatter of this row, fused (uniform branch)
            const int4 cc = reinterpret_cast<const int4*>(dt.coors)[row];  // (b,z,y,x)
            if (cc.x != 0 || cc.y < 0 || cc.y >= dt.D || cc.z < 0 || cc.z >= dt.H || cc.w < 0 || cc.w >= dt.W) {
                if (dt.status && q == 0 && wn == 0) atomicOr(dt.status, SESSD_STATUS_BAD_COORD);
            } else {
                to_dense = true;
                d = static_cast<__half*>(dt.dense) + ((size_t)cc.y * dt.Hp + cc.z + dt.pad_top) * dt.Wp + cc.w + dt.pad_left;
                plane = (size_t)dt.D * dt.Hp * dt.Wp;
            }
        }
#pragma unroll
        for (int nb = 0; nb < C::NB; ++nb) {
            const int c4 = (wn * C::NB + nb) * 16 + q * 4;
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = acc[b][nb][e];
                if (has_scale) s = s * s_epi[c4 + e];
                if (has_shift) s = s + s_epi[COUT + c4 + e];
                if (relu) s = s > 0.f ? s : 0.f;
                o[e] = s;
            }
            store4h(out + (size_t)row * COUT + c4, o);
            if (to_dense) {
#pragma unroll
                for (int e = 0; e < 4; ++e) d[(size_t)(c4 + e) * plane] = __float2half_rn(o[e]);
            }
        }
    }
    __syncthreads();
}

// PAD: the rows beyond the active ones are written too.  A variant of its own: in the launches of a frame without, its registers are what
// the coordinate passes beside them run in (frames of 60 000 points 231 us, with one kernel for both 235).
template <int CIN, int COUT, int KC, bool PAD>
__global__ void __launch_bounds__(kThreads, 2)
conv_tile(const __half* __restrict__ in, __half* __restrict__ out, const void* __restrict__ Wp,
          const int32_t* __restrict__ nbr, const int32_t* __restrict__ num_out, int max_voxels,
          const float* __restrict__ scale, const float* __restrict__ shift, int relu, DenseTarget dt) {
    using C = Shape<CIN, COUT, KC>;
    static_assert(CIN % 64 == 0 && COUT % 16 == 0, "whole MFMA chunks");
    __shared__ __align__(1024) unsigned char pool[kPool];
    __shared__ float s_epi[2 * COUT];
    int n = *num_out;
    n = n < 0 ? 0 : (n > max_voxels ? max_voxels : n);
    const int tid = threadIdx.x;

    if (tid < COUT) {  // (published by the barrier behind the list staging)
        s_epi[tid] = scale ? scale[tid] : 1.f;
        s_epi[COUT + tid] = shift ? shift[tid] : 0.f;
    }
    // the smallest tile height at which the rows are whole rounds of tiles over the workgroups
    const int slots = gridDim.x;
    const int rounds = (n + slots * C::U * C::kMaxMf - 1) / (slots * C::U * C::kMaxMf);
    const int per = rounds ? (n + slots * rounds - 1) / (slots * rounds) : 0;
    const int mf = (per + C::U - 1) / C::U;
    const v4i rs_in = make_rsrc(in, (unsigned)((size_t)max_voxels * CIN * sizeof(__half)));
    const v4i rs_w = make_rsrc(Wp, (unsigned)(C::S * C::kWeightBytes));
    const v4i rs_nbr = make_rsrc(nbr, (unsigned)((size_t)KC * max_voxels * sizeof(int32_t)));
    const bool hs = scale != nullptr, hb = shift != nullptr;
    const unsigned wave = __builtin_amdgcn_readfirstlane((unsigned)tid >> 6);
    // Rows beyond the active ones: beside the products, in stages of their own until the wave's are written, where a quarter of the workgroups
    // have a tile, else behind them, by all waves.  128 -> 128 with 150 000 rows to write, behind / beside: 2 000 rows 17.0 / 17.3 us, 8 000
    // 20.9 / 18.9, 30 000 32.4 / 30.9; with none to write, 16 000 rows, 18.4 (19.6 when every stage asked).
    const bool beside = PAD && KC > 3 && n >= slots / 4 * C::U && PadRows<__half, COUT>::reach(n, max_voxels);
    std::conditional_t<PAD && (KC > 3), PadRows<__half, COUT>, NoPadRows> pads;
    if (beside) pads.begin(out, n, max_voxels, blockIdx.x * kWaves + wave, slots * kWaves);
    // the first tile's row: up to one round, tile t goes to workgroup t / each + 8 * (t % each)
    auto first = [&](int h) {
        const int t = (n + h - 1) / h, each = (t + 7) / 8, x = blockIdx.x & 7, j = blockIdx.x >> 3;
        return t > slots || slots % 8 ? (int)blockIdx.x * h : j < each ? (x * each + j) * h : n;
    };
    auto tiles = [&](auto mf_c) {
        constexpr int MF = decltype(mf_c)::value;
        if constexpr (MF <= C::kMaxMf)
            for (int row0 = first(C::U * MF); row0 < n; row0 += slots * (C::U * MF))
                run_tile<CIN, COUT, KC, MF>(rs_in, rs_w, rs_nbr, (unsigned)max_voxels * 4u, out, row0,
                                            row0 + C::U * MF < n ? row0 + C::U * MF : n, hs, hb, relu, dt, pool, s_epi, pads);
    };
    switch (mf) {
        case 1: tiles(std::integral_constant<int, 1>{}); break;
        case 2: tiles(std::integral_constant<int, 2>{}); break;
        case 3: tiles(std::integral_constant<int, 3>{}); break;
        case 4: tiles(std::integral_constant<int, 4>{}); break;
        case 5: tiles(std::integral_constant<int, 5>{}); break;
        case 6: tiles(std::integral_constant<int, 6>{}); break;
        default: break;  // no rows
    }
    if (PAD && n < max_voxels) {
        __syncthreads();  // (a workgroup may have had no tile)
        if (!beside) {
            write_pad_rows<__half, COUT>(out, n, max_voxels, blockIdx.x * kThreads + tid, slots * kThreads, s_epi, hs, hb, relu);
        } else if (wave < kWaves && pads.left()) {
            pads.layer(s_epi, hs, hb, relu);
            pads.rest();
        }
    }
}

template <int CIN, int COUT, int KC>
int launch(const GemmArgs& a, hipStream_t stream) {
    if ((size_t)a.max_voxels * (CIN * sizeof(__half)) >= kOutOfRange) return SESSD_E_UNSUPPORTED;
    if ((size_t)a.max_voxels * (KC * sizeof(int32_t)) >= kOutOfRange) return SESSD_E_UNSUPPORTED;
    auto go = [&](auto pad) {
        hipLaunchKernelGGL((conv_tile<CIN, COUT, KC, decltype(pad)::value>), dim3(gemm_compute_units()), dim3(kThreads), 0, stream,
                           static_cast<const __half*>(a.in_feat), static_cast<__half*>(a.out_feat), a.w_packed, a.nbr, a.num_out,
                           a.max_voxels, a.scale, a.shift, a.relu, a.dense);
    };
    a.write_pad_rows ? go(std::true_type{}) : go(std::false_type{});
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

}  // namespace

// (K 3: the (3,1,1) layer that ends the backbone)
bool gemm_runs_tile(int K, int cin, int cout) {
    return K == 3 ? cin == cout && (cin == 64 || cin == 128) : K == 27 && (cin == 64 || cin == 128) && (cout == 128 || cout == cin);
}

int launch_tile(const GemmArgs& a, hipStream_t stream) {
    // (0 x infinity: with weights that are not finite an absent neighbour may not be a row of zeros)
    if (!a.w_packed || !a.halves_finite || a.in_type != SESSD_HALF || a.out_type != SESSD_HALF) return SESSD_E_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(a.in_feat) | reinterpret_cast<uintptr_t>(a.out_feat)) & 15) return SESSD_E_UNSUPPORTED;
    if (a.K == 3) {
        if (a.cin == 128 && a.cout == 128) return launch<128, 128, 3>(a, stream);
        if (a.cin == 64 && a.cout == 64) return launch<64, 64, 3>(a, stream);
    } else if (a.K == 27) {
        if (a.cin == 128 && a.cout == 128) return launch<128, 128, 27>(a, stream);
        if (a.cin == 64 && a.cout == 128) return launch<64, 128, 27>(a, stream);
        if (a.cin == 64 && a.cout == 64) return launch<64, 64, 27>(a, stream);
    }
    return SESSD_E_UNSUPPORTED;
}

}  // namespace sessd
