// coord.hip -- the passes of the coordinate side (coord.h) and their launches.
//
//   vg_insert     point -> cell table, each cell keeping its smallest point index
//   vg_flags      "am I the first point of my cell" -> wave64 ballot words + counts per 256 points; the others are kept
//                 behind the first one, the S - 1 smallest of them
//   vg_finalize   prefix over the words = voxel row in first-appearance order; coordinate and mean
//   sp_insert     ticket (input row, candidate) -> table of output cells, each keeping its smallest ticket
//   sp_flags      "am I the first ticket of my cell" -> ballot words + counts per 256 tickets
//   sp_number     prefix over the words = output row in first-seen order; out coors + voxel_num
//   lookups       nbr[k][row] for all offsets of a row, and the rows' weights for the tile cuts
//   tile cuts     equal-work tile boundaries from those weights (tile_cut.hip describes them)
//
// A pass that creates rows (vg_finalize, sp_number) holds their coordinates and numbers in registers: it inserts the
// next strided layer's tickets right away, and what only needs finished tables (lookups, cuts) shares a launch with the
// next step of the chain.  For the reference's backbone that is 13 launches a frame in place of 35.
// Measured (frames without their GEMMs, us; 35 launches, 13, 13 as they are now): 2 000 points 141, 79, 62, 20 000 164, 97, 72, 80 000
// 231, 127, 95, 60 000 (FP16 configuration) 162, 111, 84, 150 000 221, 147, 111.  A pass is bound by its chain of dependent trips to
// memory (four to six of 0.7-1 us each) until some 40 000 rows, and by random accesses beyond.
#include "conv_tall.h"
#include "coord.h"
#include "fill.h"

namespace sessd {

namespace {

constexpr uint32_t kSlotBits = 26;
constexpr uint32_t kSlotMask = (1u << kSlotBits) - 1u;

// ---------------------------------------------------------------------------------------------
// voxelizer
// ---------------------------------------------------------------------------------------------
// -> key of the cell the point lies in, kEmpty when it lies in none
__device__ __forceinline__ uint32_t point_cell(const VgPart& p, float x, float y, float z, int& ix, int& iy, int& iz) {
    // voxelGenerator.cu:363-367: half-open range test
    if (!(x >= p.min_x && x < p.max_x && y >= p.min_y && y < p.max_y && z >= p.min_z && z < p.max_z)) return kEmpty;
    // voxelGenerator.cu:369-371: IEEE FP32 division (never a reciprocal multiply)
    ix = (int)floorf((x - p.min_x) / p.vx);
    iy = (int)floorf((y - p.min_y) / p.vy);
    iz = (int)floorf((z - p.min_z) / p.vz);
    // voxelGenerator.cu:375: a value just below max can still land on the grid size
    if (!(ix >= 0 && ix < p.gx && iy >= 0 && iy < p.gy && iz >= 0 && iz < p.gz)) return kEmpty;
    return ((uint32_t)iz * (uint32_t)p.gy + (uint32_t)iy) * (uint32_t)p.gx + (uint32_t)ix;
}

// cells that rows have taken -> empty
__device__ __forceinline__ void clean_pass(const CleanPart& P, int block) {
    const int n = clamp_rows(reinterpret_cast<const int32_t*>(P.taken), P.max_voxels);
    for (int row = block * kCoordBlock + (int)threadIdx.x; row < n; row += P.blocks * kCoordBlock) {
        const uint32_t key = P.taken[kCellListHead + row];
        if (key < P.t.cap) static_cast<uint32_t*>(P.t.base)[key] = kEmpty;
    }
}

struct Cleans {
    CleanPart c[kMaxCleans];
    int n;
};

template <int N>
__global__ void __launch_bounds__(kCoordBlock) vg_insert(VgPart p, Cleans cleans, FillPlan<N> also) {
    if ((int)blockIdx.x >= p.n_blocks) {
        int b = blockIdx.x - p.n_blocks;
        for (int i = 0; i < cleans.n; ++i) {
            if (b < cleans.c[i].blocks) return clean_pass(cleans.c[i], b);
            b -= cleans.c[i].blocks;
        }
        return fill_pass(also, b);
    }
    asm volatile("" :: "s"(p.points), "s"(p.points_size), "s"(p.max_points), "s"(p.pf), "s"(p.min_x), "s"(p.vz), "s"(p.gx), "s"(p.t.base), "s"(p.t.dense),
                 "s"(p.pt_slot), "s"(p.sums), "s"(p.status));
    const int i = blockIdx.x * kCoordBlock + threadIdx.x;
    const float* pt = p.points + (size_t)(i < p.max_points ? i : p.max_points - 1) * p.pf;  // (beside the number of points)
    const float x = pt[0], y = pt[1], z = pt[2];
    const int n = __builtin_amdgcn_readfirstlane(clamp_rows(p.points_size, p.max_points));
    if (p.sums && threadIdx.x == 0 && blockIdx.x % kCountsPerSum == 0) p.sums[blockIdx.x / kCountsPerSum] = 0;
    if (i >= n) return;
    int ix, iy, iz;
    const uint32_t key = point_cell(p, x, y, z, ix, iy, iz);
    int32_t slot = -1;
    if (key != kEmpty) {
        slot = insert_min(open_table(p.t, n), key, (uint32_t)i);
        if (slot < 0) atomicOr(&p.status[1], SESSD_STATUS_HASH_FULL);
    }
    p.pt_slot[i] = slot;
}

// The table names every cell's first point f now.  A later point of the cell is offered to the S - 1 places behind f,
// which keep the smallest indices in ascending order: every place ends up with the minimum of what was offered to it and
// passes the rest on, so the final state does not depend on the order in which the threads arrive.
template <int N>
__global__ void __launch_bounds__(kCoordBlock) vg_flags(VgPart p, FillPlan<N> also) {
    if ((int)blockIdx.x >= p.n_blocks) return fill_pass(also, blockIdx.x - p.n_blocks);
    __shared__ uint32_t lds4[4];
    asm volatile("" :: "s"(p.points_size), "s"(p.max_points), "s"(p.max_pts), "s"(p.t.base), "s"(p.t.dense), "s"(p.slots), "s"(p.pt_slot), "s"(p.words),
                 "s"(p.counts), "s"(p.sums));
    const int i = blockIdx.x * kCoordBlock + threadIdx.x;
    const int32_t slot = p.pt_slot[i < p.max_points ? i : p.max_points - 1];  // (beside the number of points)
    const int n = __builtin_amdgcn_readfirstlane(clamp_rows(p.points_size, p.max_points));
    bool first = false;
    if (i < n) {
        if (slot >= 0) {
            const uint32_t f = value_at(open_table(p.t, n), slot);
            first = f == (uint32_t)i;
            if (!first) {
                uint32_t* s = p.slots + (size_t)f * (p.max_pts - 1);
                uint32_t cur = (uint32_t)i;
                for (int q = 0; q < p.max_pts - 1; ++q) {
                    const uint32_t old = atomicMin(&s[q], cur);
                    if (old == kEmpty) break;
                    cur = old > cur ? old : cur;
                }
            }
        }
    }
    const uint64_t m = __ballot(first);
    if ((threadIdx.x & 63) == 0) {
        p.words[i >> 6] = m;
        lds4[threadIdx.x >> 6] = __popcll(m);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t c = lds4[0] + lds4[1] + lds4[2] + lds4[3];
        p.counts[blockIdx.x] = c;
        if (p.sums && c) atomicAdd(&p.sums[blockIdx.x / kCountsPerSum], c);
    }
}

// ---------------------------------------------------------------------------------------------
// strided layers: tickets
// ---------------------------------------------------------------------------------------------
// x / s truncating toward zero, s >= 1
__device__ __forceinline__ int div_trunc(int x, int s) {
    if (s == 1) return x;
    if (s == 2) return (x - (x >> 31)) >> 1;
    asm volatile("" : "+s"(s));  // (or the division's preparations are made in front of everything, whatever s is)
    return x / s;
}
// e / c for the short candidate lists (e < 27)
__device__ __forceinline__ int div_small(int e, int c) {
    return c == 1 ? e : (c == 2 ? e >> 1 : (c == 3 ? (e * 43) >> 7 : e / c));
}

// getValidOutPosKernel (sparseConv3dlayer.cu:310-386), one enumeration step: candidate `e` of the input cell c.  Integer
// divisions truncate toward zero exactly as in the reference; dilation is 1.
// -> false when e is past the enumeration or the output cell is outside the grid
__device__ __forceinline__ bool sp_candidate(const int c[3], const SpPart& P, int e, int o[3], int& offset) {
    int up[3], cs[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int lo = div_trunc(c[a] - (P.k[a] - 1) - 1 + P.s[a] + P.p[a], P.s[a]);
        up[a] = div_trunc(c[a] + P.p[a], P.s[a]);
        cs[a] = up[a] - lo + 1;
    }
    if (cs[0] <= 0 || cs[1] <= 0 || cs[2] <= 0 || e >= cs[0] * cs[1] * cs[2]) return false;
    const int e1 = div_small(e, cs[2]), e0 = div_small(e1, cs[1]);
    const int cnt[3] = {e0, e1 - e0 * cs[1], e - e1 * cs[2]};  // x fastest
    bool valid = true;
    int m = 1;
    offset = 0;
#pragma unroll
    for (int a = 2; a >= 0; --a) {
        o[a] = up[a] - cnt[a];
        if (o[a] < 0 || o[a] > P.os[a] - 1) valid = false;
        offset += m * (c[a] - o[a] * P.s[a] + P.p[a]);
        m *= P.k[a];
    }
    return valid;
}

// Rows that follow each other name the same output cells again and again (eight input cells share an output cell of a
// 3x3x3 stride-2 layer, and neighbours in space are mostly neighbours in the row order), and device-wide atomics are what
// this pass is made of.  A block therefore gathers the cells of kTicketsAtOnce tickets in an LDS table first (cell ->
// smallest ticket of the block), and one thread per distinct cell goes to the table in memory.
constexpr int kPerThread = 2;
constexpr int kTicketsAtOnce = kPerThread * kCoordBlock;
constexpr int kLocalBits = 10, kLocalSlots = 1 << kLocalBits;  // twice the tickets
struct alignas(16) InsertLds {
    uint32_t key[kLocalSlots], val[kLocalSlots];
};

// The same for kernels of 3 and strides of 2 on every axis, where an axis has one or two candidates; c >= 0.
__device__ __forceinline__ bool sp_candidate_halving(const int c[3], const SpPart& P, int e, int o[3], int& offset) {
    offset = 0;
    int m = 1;
    bool valid = true;
#pragma unroll
    for (int a = 2; a >= 0; --a) {
        const int at = c[a] + P.p[a], two = !(at & 1) && at > 0 ? 1 : 0, second = e & two;
        e >>= two;
        o[a] = (at >> 1) - second;
        valid = valid && (uint32_t)o[a] < (uint32_t)P.os[a];
        offset += m * ((at & 1) + 2 * second);
        m *= 3;
    }
    return valid && e == 0;
}

// the tickets of m rows (row, z, y, x) in LDS; the whole block takes part
template <bool HALVING>
__device__ __forceinline__ void sp_insert_rows(const SpPart& P, const CellView& t, const int4* rows, int m, InsertLds& L) {
    const int total = m * P.Kc;
    for (int base = 0; base < total; base += kTicketsAtOnce) {
        static_assert(kLocalSlots == 4 * kCoordBlock, "a store for each thread");
        reinterpret_cast<uint4*>(L.key)[threadIdx.x] = make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
        reinterpret_cast<uint4*>(L.val)[threadIdx.x] = make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
        __syncthreads();
        uint32_t key[kPerThread], tk[kPerThread];
        int local[kPerThread], offset[kPerThread];
        bool live[kPerThread], owner[kPerThread];
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) {
            const int item = base + j * kCoordBlock + threadIdx.x;
            live[j] = item < total;
            owner[j] = false;
            local[j] = -1;
            offset[j] = 0;
            key[j] = tk[j] = kEmpty;
            if (!live[j]) continue;
            int r = item >> 3, e = item & 7;
            if (!HALVING && P.Kc != 8) {
                int per = P.Kc;
                asm volatile("" : "+s"(per));
                r = item / per;
                e = item - r * per;
            }
            const int4 row = rows[r];
            const int c[3] = {row.y, row.z, row.w};
            tk[j] = (uint32_t)row.x * (uint32_t)P.Kc + (uint32_t)e;
            int o[3];
            // A negative coordinate makes the truncating divisions of getValidOutPos yield kernel offsets outside
            // [0, K) (c = -2, k = 3, s = 2, p = 1: o = 0, offset term -1), with which the reference indexes its
            // rulebook.  Such a row contributes nothing here and raises BAD_COORD; the offset is checked as well, so
            // that nothing a caller passes can make sp_scatter store outside the neighbour table.
            const bool bad = (c[0] | c[1] | c[2]) < 0;
            if (bad && e == 0) atomicOr(&P.meta[2], SESSD_STATUS_BAD_COORD);
            if (bad || !(HALVING ? sp_candidate_halving(c, P, e, o, offset[j]) : sp_candidate(c, P, e, o, offset[j])) || offset[j] < 0 ||
                offset[j] >= P.K)
                continue;
            key[j] = ((uint32_t)o[0] * (uint32_t)P.os[1] + (uint32_t)o[1]) * (uint32_t)P.os[2] + (uint32_t)o[2];
            uint32_t ls = (key[j] * 2654435769u) >> (32 - kLocalBits);
            for (;;) {  // (at most kTicketsAtOnce keys in twice as many slots: room is always found)
                const uint32_t prev = atomicCAS(&L.key[ls], kEmpty, key[j]);
                if (prev == kEmpty || prev == key[j]) {
                    owner[j] = prev == kEmpty;
                    break;
                }
                ls = (ls + 1) & (kLocalSlots - 1);
            }
            local[j] = (int)ls;
            atomicMin(&L.val[ls], tk[j]);
        }
        __syncthreads();
        // the thread that claimed a cell's LDS entry carries the block's smallest ticket to memory
        if (t.d) {
#pragma unroll
            for (int j = 0; j < kPerThread; ++j)
                if (owner[j]) atomicMin(&t.d[key[j]], L.val[local[j]]);
        } else {
            EntryGroup g[kPerThread];
            uint32_t at[kPerThread];
            unsigned long long prev[kPerThread];
#pragma unroll
            for (int j = 0; j < kPerThread; ++j)
                if (owner[j]) g[j] = load_group(t, first_slot(t, key[j]));
#pragma unroll
            for (int j = 0; j < kPerThread; ++j)
                if (owner[j]) {
                    at[j] = likely_slot(t, key[j], g[j]);
                    prev[j] = atomicCAS(&t.h[at[j]], kEmptyEntry, make_entry(key[j], L.val[local[j]]));
                }
#pragma unroll
            for (int j = 0; j < kPerThread; ++j)
                if (owner[j]) {
                    const int32_t slot = finish_insert_min(t, key[j], L.val[local[j]], at[j], prev[j]);
                    if (slot < 0) {
                        atomicOr(&P.meta[2], SESSD_STATUS_HASH_FULL);
                        L.key[local[j]] = kEmpty;  // (read below as "no slot")
                    } else {
                        L.val[local[j]] = (uint32_t)slot;
                    }
                }
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < kPerThread; ++j)
            if (live[j]) {
                uint32_t c = kEmpty;
                if (local[j] >= 0 && L.key[local[j]] != kEmpty)
                    c = ((uint32_t)offset[j] << kSlotBits) | (t.d ? key[j] : L.val[local[j]]);
                P.cand[tk[j]] = c;
            }
        if (base + kTicketsAtOnce < total) __syncthreads();
    }
}
__device__ __forceinline__ void sp_insert_rows(const SpPart& P, const CellView& t, const int4* rows, int m, InsertLds& L) {
    if (P.halving) sp_insert_rows<true>(P, t, rows, m, L);
    else sp_insert_rows<false>(P, t, rows, m, L);
}

// Points per block of vg_finalize: with a strided layer behind it, a wave of points gives the block's four waves about
// one round of tickets.
constexpr int kFinalPoints = 64;
constexpr int kBlocksAhead = 3;  // counts of 256-point blocks that a thread asks for at once (196 608 points)
constexpr int kAhead = 4;  // further points of a cell that are requested ahead (the reference averages five)

__global__ void __launch_bounds__(kCoordBlock) vg_finalize(VgPart p, SpPart next, int has_next) {
    __shared__ uint32_t lds[8];
    __shared__ int4 s_rows[kFinalPoints];
    __shared__ int s_m;
    __shared__ InsertLds L;
    asm volatile("" :: "s"(p.points), "s"(p.points_size), "s"(p.max_points), "s"(p.pf), "s"(p.max_voxels), "s"(p.max_pts), "s"(p.slots), "s"(p.pt_slot),
                 "s"(p.words), "s"(p.counts), "s"(p.sums), "s"(p.n_blocks), "s"(p.voxels), "s"(p.coors), "s"(p.taken), "s"(next.halving), "s"(next.t.base),
                 "s"(next.meta));
    // What the block's points need is requested beside the number of points, which says how much of it counts: their words, cells and
    // coordinates, the counts of the blocks in front of them and, for any that turns out to be its cell's first, the cell's further
    // points.
    const int first_point = blockIdx.x * kFinalPoints;
    const int i = first_point + (int)threadIdx.x;
    const int mine = first_point / kCoordBlock, in_block = (first_point / 64) & 3;
    uint64_t w[4];
    int32_t slot = -1;
    float x = 0.f, y = 0.f, z = 0.f, f = 0.f;
    uint32_t* more = p.slots + (size_t)i * (p.max_pts - 1);
    uint32_t idx[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) idx[q] = kEmpty;
    for (int q = 0; q < 4; ++q) w[q] = p.words[mine * 4 + q];
    if (threadIdx.x < kFinalPoints && i < p.max_points) {
        slot = p.pt_slot[i];
        const float* pt = p.points + (size_t)i * p.pf;
        x = pt[0];
        y = pt[1];
        z = pt[2];
        f = pt[3];
#pragma unroll
        for (int q = 0; q < kAhead; ++q)
            if (q < p.max_pts - 1) idx[q] = more[q];
    }
    uint32_t count[kBlocksAhead];
    if (!p.sums) {
#pragma unroll
        for (int q = 0; q < kBlocksAhead; ++q) {
            const int b = q * kCoordBlock + (int)threadIdx.x;
            count[q] = p.counts[b < p.n_blocks ? b : p.n_blocks - 1];
        }
    }
    const int n = __builtin_amdgcn_readfirstlane(clamp_rows(p.points_size, p.max_points));
    const int n_blocks = (n + kCoordBlock - 1) / kCoordBlock;  // 256-point blocks that hold points
    if (first_point >= n && blockIdx.x != 0) return;
    const bool point = threadIdx.x < kFinalPoints && i < n;
    uint64_t m = 0;
    for (int q = 0; q < 4; ++q)
        if (q == in_block) m = first_point < n ? w[q] : 0;
    const bool first = point && ((m >> threadIdx.x) & 1ull);
    float ahead[kAhead][4];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
        if (!first) idx[q] = kEmpty;
        const float* pt = p.points + (size_t)(idx[q] != kEmpty ? idx[q] : 0) * p.pf;
#pragma unroll
        for (int e = 0; e < 4; ++e) ahead[q][e] = idx[q] != kEmpty ? pt[e] : 0.f;
    }
    // the counts in front of the block's points and of all: each of them, or the sums over 64 and the own 64's
    uint32_t before = 0, total = 0;
    static_assert(kCountsPerSum <= kCoordBlock, "one count a thread");
    if (p.sums) {
        const int own = mine / kCountsPerSum, parts = (n_blocks + kCountsPerSum - 1) / kCountsPerSum;
        if ((int)threadIdx.x < mine - own * kCountsPerSum) before = p.counts[own * kCountsPerSum + (int)threadIdx.x];
        for (int j = threadIdx.x; j < parts; j += kCoordBlock) {
            const uint32_t c = p.sums[j];
            total += c;
            if (j < own) before += c;
        }
    } else {
#pragma unroll
        for (int q = 0; q < kBlocksAhead; ++q) {
            const int b = q * kCoordBlock + (int)threadIdx.x;
            total += b < n_blocks ? count[q] : 0;
            before += b < mine && b < n_blocks ? count[q] : 0;
        }
        for (int b = kBlocksAhead * kCoordBlock + (int)threadIdx.x; b < n_blocks; b += kCoordBlock) {
            const uint32_t c = p.counts[b];
            total += c;
            if (b < mine) before += c;
        }
    }
    block_sums(before, total, lds);
    const int rows = (int)(total > (uint32_t)p.max_voxels ? (uint32_t)p.max_voxels : total);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *p.voxel_num = rows;
        if (p.taken) p.taken[0] = (uint32_t)rows;
        p.status[0] = p.status[1] | (total > (uint32_t)p.max_voxels ? SESSD_STATUS_VOXEL_OVERFLOW : 0);
        p.status[1] = 0;
    }
    for (int q = 0; q < 4; ++q)
        if (q < in_block) before += __popcll(w[q]);
    const uint32_t rank = rank_in_wave(m), vid = before + rank;
    const bool kept = first && vid < (uint32_t)p.max_voxels;
    if (threadIdx.x < 64) {
        const int room = before >= (uint32_t)p.max_voxels ? 0 : (int)((uint32_t)p.max_voxels - before);
        const int here = __popcll(m);
        if (threadIdx.x == 0) s_m = here < room ? here : room;
        if (kept) {
            int ix, iy, iz;
            const uint32_t key = point_cell(p, x, y, z, ix, iy, iz);
            if (p.taken) p.taken[kCellListHead + vid] = key;
            reinterpret_cast<int4*>(p.coors)[vid] = make_int4(0, iz, iy, ix);  // voxelGenerator.cu:404-405
            s_rows[rank] = make_int4((int)vid, iz, iy, ix);
        }
        // the table now maps cell -> voxel row; cells first seen beyond the cap are dropped
        if (first) set_value(open_table(p.t, n), slot, kept ? vid : kEmpty);
    }
    if (has_next) {
        __syncthreads();
        sp_insert_rows(next, open_table(next.t, rows < next.max_voxels ? rows : next.max_voxels), s_rows, s_m, L);
    }
    // the places are left empty for the next frame
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
        if (idx[q] != kEmpty) more[q] = kEmpty;
    if (first && !kept)
        for (int q = kAhead; q < p.max_pts - 1; ++q) more[q] = kEmpty;
    if (!kept) return;
    // voxelGenerator.cu:274-296: all S slots are summed left to right, unfilled slots count as 0
    float sx = x, sy = y, sz = z, sw = f;
    int cnt = 1;
    for (int q = 0; q < p.max_pts - 1; ++q) {
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        if (q < kAhead) {
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (j == q) {
                    cnt += idx[j] != kEmpty ? 1 : 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[e] = ahead[j][e];
                }
        } else if (more[q] != kEmpty) {
            const float* pt = p.points + (size_t)more[q] * p.pf;
            for (int e = 0; e < 4; ++e) a[e] = pt[e];
            ++cnt;
            more[q] = kEmpty;
        }
        sx = sx + a[0];
        sy = sy + a[1];
        sz = sz + a[2];
        sw = sw + a[3];
    }
    const float c = (float)cnt;
    reinterpret_cast<float4*>(p.voxels)[vid] = make_float4(sx / c, sy / c, sz / c, sw / c);
}

// the tickets of a coors tensor (a strided layer on its own)
__global__ void __launch_bounds__(kCoordBlock) sp_insert(SpPart P) {
    __shared__ int4 s_rows[kTicketsAtOnce];
    __shared__ InsertLds L;
    const int n = clamp_rows(P.in_num, P.max_voxels);
    const int per = kTicketsAtOnce / P.Kc > 0 ? kTicketsAtOnce / P.Kc : 1;  // rows a block takes at a time
    const CellView t = open_table(P.t, n);
    for (int r0 = blockIdx.x * per; r0 < n; r0 += gridDim.x * per) {
        const int m = n - r0 < per ? n - r0 : per;
        __syncthreads();
        for (int r = threadIdx.x; r < m; r += kCoordBlock) {
            const int4 c = reinterpret_cast<const int4*>(P.in_coors)[r0 + r];
            s_rows[r] = make_int4(r0 + r, c.y, c.z, c.w);
        }
        __syncthreads();
        sp_insert_rows(P, t, s_rows, m, L);
    }
}

// A launch passes its arguments by value, and the compiler reads each of them where it is used: one trip to memory of 400-1 100
// cycles after the other, nine in a row in front of the first probe of a lookup.  The passes name all that they need in one place
// (an asm without instructions), so that it arrives together.
__device__ __forceinline__ void sp_flags_pass(const SpPart& a, int block, int blocks, uint32_t* lds4) {
    SpPart P = a;
    asm volatile("" :: "s"(P.in_num), "s"(P.max_voxels), "s"(P.Kc), "s"(P.t.base), "s"(P.t.dense), "s"(P.cand), "s"(P.words), "s"(P.counts));
    // (the first chunk's tickets beside the row count: in bounds, there are at most n_chunks blocks)
    uint32_t slot = P.cand[(uint32_t)block * kCoordBlock + threadIdx.x];
    const int64_t tickets = (int64_t)clamp_rows(P.in_num, P.max_voxels) * P.Kc;
    for (int c = block; (int64_t)c * kCoordBlock < tickets; c += blocks) {
        const uint32_t tk = (uint32_t)c * kCoordBlock + threadIdx.x;
        if (c != block) slot = P.cand[tk];
        bool first = false;
        if (tk < tickets && slot != kEmpty) {
            const uint32_t at = slot & kSlotMask;
            first = (P.t.dense ? static_cast<const uint32_t*>(P.t.base)[at] : static_cast<const uint32_t*>(P.t.base)[2 * (size_t)at]) == tk;
        }
        const uint64_t m = __ballot(first);
        __syncthreads();
        if ((threadIdx.x & 63) == 0) {
            P.words[tk >> 6] = m;
            lds4[threadIdx.x >> 6] = __popcll(m);
        }
        __syncthreads();
        if (threadIdx.x == 0) P.counts[c] = lds4[0] + lds4[1] + lds4[2] + lds4[3];
    }
}

// ---------------------------------------------------------------------------------------------
// lookups
// ---------------------------------------------------------------------------------------------
// A block takes 64 rows, a lane each; each of its four waves takes a quarter of the offsets, so that an offset's place in the kernel
// is the same for the whole wave, all probes of a lane are in flight at once, and stores are runs of 64 rows.
// A block of 64 rows at 17 262 rows: 11 900 cycles with four lanes a row (each lane a quarter of the offsets, their places found per
// lane: 2 000 for seven keys) and the arguments read as they came, 6 100 now; the SubM plugin 64 -> 64 40.3 -> 37.9 us, frames of 2 000
// points 205.5 -> 200.8, 20 000 306.9 -> 300.6, 60 000 (FP16) 250.7 -> 246.4.
// HASH: some of the launch's tables are hashes.  The probes of a hash take 106 registers, which leaves the blocks no room beside three
// workgroups of conv_wide<32,32> (3 x 144 of 512) or one of the 64-column kernels (2 x 216); dense tables alone take 48 and, with a row's
// counts in bytes, 272 B of LDS of the 576 or more that those leave.  Frames, one launch for both / so: FP32 5 000 points 211.5 -> 209.2 us,
// 40 000 332 -> 323, 80 000 418 -> 410, whose 61 440 rows and more in the second stage are two rounds of tiles; FP16 20 000 184.8 -> 181.0.
constexpr int kLookupRows = 64;                             // rows of a block
constexpr int kLookupDepth = (kGemmMaxOffsets + 3) / 4;     // offsets of a wave
struct LookupLds {
    uint8_t found[kCoordBlock];  // by each wave for each row (kLookupDepth at most)
    int32_t sum[4];              // ... for all of its rows
};

// What a wave finds for a row: val[j] = the row at the wave's j-th offset.  QUARTER 0 .. 3: of a 3x3x3 kernel on a dense table, where
// the offsets are constants; -1: any (`start`: the first offset, z << 16 | y << 8 | x, `mine`: how many).
template <int QUARTER, bool HASH>
__device__ __forceinline__ void look_up(const LookupPart& P, const int4& c, bool in_layer, int start, int mine, uint32_t (&val)[kLookupDepth]) {
    const int z0 = c.y * P.s[0] - P.p[0], y0 = c.z * P.s[1] - P.p[1], x0 = c.w * P.s[2] - P.p[2];
    const uint32_t origin = ((uint32_t)z0 * (uint32_t)P.t.gy + (uint32_t)y0) * (uint32_t)P.t.gx + (uint32_t)x0;
    uint32_t key[kLookupDepth];
    bool ok[kLookupDepth];
    auto probe = [&](int j, int kz, int ky, int kx) {
        ok[j] = in_layer && (uint32_t)(z0 + kz) < (uint32_t)P.t.gz && (uint32_t)(y0 + ky) < (uint32_t)P.t.gy && (uint32_t)(x0 + kx) < (uint32_t)P.t.gx;
        key[j] = origin + ((uint32_t)(kz * P.t.gy + ky) * (uint32_t)P.t.gx + (uint32_t)kx);
    };
    if constexpr (QUARTER >= 0) {
        const uint32_t* d = static_cast<const uint32_t*>(P.t.base);
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j) {
            constexpr int kFirst = QUARTER * kLookupDepth;
            const int k = kFirst + j;
            if (k >= 27) {
                val[j] = kEmpty;
                continue;
            }
            probe(j, k / 9, k / 3 % 3, k % 3);
            val[j] = d[ok[j] ? key[j] : 0];
        }
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j)
            if (QUARTER * kLookupDepth + j < 27) val[j] = ok[j] ? val[j] : kEmpty;
        return;
    }
    int kz = start >> 16, ky = (start >> 8) & 255, kx = start & 255;
#pragma unroll
    for (int j = 0; j < kLookupDepth; ++j) {
        probe(j, kz, ky, kx);
        ok[j] = ok[j] && j < mine;
        if (++kx == P.k[2]) {
            kx = 0;
            if (++ky == P.k[1]) {
                ky = 0;
                ++kz;
            }
        }
    }
    if (!HASH || P.t.dense) {
        const uint32_t* d = static_cast<const uint32_t*>(P.t.base);
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j) val[j] = d[ok[j] ? key[j] : 0];
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j) val[j] = ok[j] ? val[j] : kEmpty;
        return;
    }
    // All probe sequences advance together, a round of loads at a time, four entries per sequence and round: one
    // after the other the collisions of seven sequences were seven times the latency (15 us for 2 000 rows).
    const CellView t = open_table(P.t, clamp_rows(P.t_num, P.t_max));
    uint32_t slot[kLookupDepth];
    bool any = false;
#pragma unroll
    for (int j = 0; j < kLookupDepth; ++j) {
        slot[j] = first_slot(t, key[j]);
        val[j] = kEmpty;
        any |= ok[j];
    }
    for (uint32_t round = 0; any && round <= t.mask; round += kGroup) {
        EntryGroup g[kLookupDepth];
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j)
            if (ok[j]) g[j] = load_group(t, slot[j]);
        any = false;
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j) {
            if (ok[j]) {
#pragma unroll
                for (int e = 0; e < kGroup; ++e) {
                    if (e < (int)(slot[j] & (kGroup - 1))) continue;
                    if (entry_key(g[j].e[e]) == key[j]) {
                        val[j] = entry_val(g[j].e[e]);
                        ok[j] = false;
                    } else if (g[j].e[e] == kEmptyEntry) {
                        ok[j] = false;
                    }
                }
                slot[j] = ((slot[j] | (kGroup - 1)) + 1) & t.mask;
            }
            any |= ok[j];
        }
    }
}

// CUBE: a 3x3x3 kernel on a dense table
template <bool CUBE, bool HASH>
__device__ __forceinline__ void lookup_rows(const LookupPart& P, int block, int n, int start, int4 c, LookupLds& L) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int K = CUBE ? 27 : P.K, per = (K + 3) >> 2, k0 = wave * per, mine = K - k0 < per ? K - k0 : per;  // (mine may be negative: none)
    int row = block * kLookupRows + lane;
    for (int chunk = block; chunk * kLookupRows < n; chunk += P.blocks, row += P.blocks * kLookupRows) {
        if (chunk != block) c = reinterpret_cast<const int4*>(P.coors)[row < n ? row : n - 1];
        const bool in_layer = row < n && (uint32_t)c.y < (uint32_t)P.own[0] && (uint32_t)c.z < (uint32_t)P.own[1] && (uint32_t)c.w < (uint32_t)P.own[2];
        uint32_t val[kLookupDepth];
        if (!CUBE) look_up<-1, HASH>(P, c, in_layer, start, mine, val);
        else if (wave == 0) look_up<0, HASH>(P, c, in_layer, 0, 0, val);
        else if (wave == 1) look_up<1, HASH>(P, c, in_layer, 0, 0, val);
        else if (wave == 2) look_up<2, HASH>(P, c, in_layer, 0, 0, val);
        else look_up<3, HASH>(P, c, in_layer, 0, 0, val);
        int cnt = 0, sum = 0;
        int32_t* to = P.nbr + (size_t)k0 * P.max_voxels + row;
#pragma unroll
        for (int j = 0; j < kLookupDepth; ++j, to += P.max_voxels) {
            if (j >= (CUBE ? 27 - 3 * kLookupDepth : 0) && j >= mine) break;
            const bool hit = val[j] != kEmpty;
            cnt += hit ? 1 : 0;
            sum += __popcll(__ballot(hit));
            if (row < n) *to = (int32_t)val[j];
        }
        if (P.w) {
            __syncthreads();
            L.found[threadIdx.x] = (uint8_t)cnt;
            if (lane == 0) L.sum[wave] = sum;
            __syncthreads();
            if (wave == 0) {
                const int w = cnt + L.found[64 + lane] + L.found[128 + lane] + L.found[192 + lane] + P.row_weight;
                if (row < P.max_voxels) P.w[row] = row < n ? w : 0;
                const int rows = n - chunk * kLookupRows < kLookupRows ? n - chunk * kLookupRows : kLookupRows;
                if (lane == 0) P.wsum[chunk] = L.sum[0] + L.sum[1] + L.sum[2] + L.sum[3] + rows * P.row_weight;
            }
        }
    }
}

template <bool HASH>
__device__ __forceinline__ void lookup_pass(const LookupPart& a, int block, LookupLds& L) {
    const LookupPart P = a;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), start = a.first[wave];
    asm volatile("" :: "s"(P.coors), "s"(P.num), "s"(P.max_voxels), "s"(P.t.base), "s"(P.nbr), "s"(P.meta), "s"(P.w), "s"(P.K), "s"(start));
    const int row = block * kLookupRows + (threadIdx.x & 63);
    // (the first rows' coordinates beside the row count: in bounds, not used beyond the active ones)
    const int4 c = reinterpret_cast<const int4*>(P.coors)[row < P.max_voxels ? row : P.max_voxels - 1];
    const int n = __builtin_amdgcn_readfirstlane(clamp_rows(P.num, P.max_voxels));
    if (P.meta && block == 0 && threadIdx.x == 0) P.meta[1] = n;
    if (block * kLookupRows >= n) return;
    if (P.t.dense && P.k[0] == 3 && P.k[1] == 3 && P.k[2] == 3) lookup_rows<true, HASH>(P, block, n, start, c, L);
    else lookup_rows<false, HASH>(P, block, n, start, c, L);
}

struct FlagsLookups {
    SpPart flags;
    LookupPart look[kMaxLookups];
};

// Products of a layer that does not need what a pass makes, in the pass's launch (conv_tall.h, a workgroup of four waves for each compute
// unit): layer 0 beside the numbering of the first strided layer's rows, layer 1 beside the lookups on them.  On a branch of its own either
// side began 7 us after the other, and the first strided layer 8 to 10 us after the later one.  That layer's products begin, us after the
// frame: FP32 2 000 points 47.7 -> 41.1, 20 000 55.9 -> 49.9, FP16 60 000 61.8 -> 53.2.  Frames FP32 2 000 points 174.0 -> 167.1, 8 000 210.2 -> 202.8,
// 20 000 257.6 -> 254.9, 80 000 386 -> 378, FP16 8 000 161.9 -> 151.5, 60 000 196.1 -> 189.6, launched directly 20 000 286.7 -> 276.9.  Two
// workgroups a unit: the same times but 80 000 points, 1.008x.  The registers are held to what lets five blocks share a unit (lookups
// beside FP16 products seven, beside FP32 products four: held to five they need scratch, with which a launch begins 3 us later; frames of 2 000
// points 169.1 -> 167.2, 20 000 256.2 -> 254.8), so that a pass finds room for its blocks beside the products.  32 -> 32 in FP16 is
// multiplied by two workgroups of 16 columns each, which read the rows twice: with 54 KB of weights a unit would have room for two blocks (doubled
// widths, 30 000 points 284.9 -> 275.8 us, 150 000 0.997x, where the lookups are three rounds of blocks).
constexpr int kProductWaves = kCoordBlock / 64, kPadBlocks = 256;  // (those write the rows beyond the active ones, behind all others)
template <int CIN, int COUT, typename T>
constexpr int kProductCols = CIN == 32 ? 16 : COUT;
template <int CIN, int COUT, typename T>
using ProductLds = tall::Lds<CIN, kProductCols<CIN, COUT, T>, T, kProductWaves, COUT>;
static int product_blocks(const GemmArgs& a) { return gemm_compute_units() * (a.cin == 32 ? 2 : 1); }

template <int CIN, int COUT, typename T, typename TO>
__device__ __forceinline__ void products_pass(const TallArgs& g, int block, int blocks, ProductLds<CIN, COUT, T>& lds) {
    constexpr int kCols = kProductCols<CIN, COUT, T>;
    const int groups = blocks / (COUT / kCols), part = block / groups;
    tall::workgroup<CIN, kCols, T, TO, kProductWaves, 0, COUT>(g, DenseTarget(), block - part * groups, groups, lds, part * kCols);
}
template <int CIN, int COUT, typename T, typename TO>
__device__ __forceinline__ void products_pad_pass(const TallArgs& g, int block, ProductLds<CIN, COUT, T>& lds) {
    const int n = clamp_rows(g.num_out, g.max_voxels);
    if (threadIdx.x < COUT) {
        lds.epi[threadIdx.x] = g.scale ? g.scale[threadIdx.x] : 1.f;
        lds.epi[COUT + threadIdx.x] = g.shift ? g.shift[threadIdx.x] : 0.f;
    }
    __syncthreads();
    write_pad_rows<TO, COUT>(static_cast<TO*>(g.out), n, g.max_voxels, block * kCoordBlock + threadIdx.x, kPadBlocks * kCoordBlock, lds.epi, g.scale != nullptr,
                             g.shift != nullptr, g.relu);
}

// end1 .. end3: where the blocks of the lookups behind the first begin.  (Arguments of their own: those are in registers when the
// kernel starts.)
template <bool HASH>
__device__ __forceinline__ void flags_lookups_block(int b, int flag_blocks, int end1, int end2, int end3, const FlagsLookups& a, LookupLds& L) {
    if (b < flag_blocks) return sp_flags_pass(a.flags, b, flag_blocks, reinterpret_cast<uint32_t*>(L.sum));
    const int l = __builtin_amdgcn_readfirstlane((b >= end1 ? 1 : 0) + (b >= end2 ? 1 : 0) + (b >= end3 ? 1 : 0));
    static_assert(kMaxLookups == 4, "one argument for each lookup but the first");
    lookup_pass<HASH>(a.look[l], b - (l == 0 ? flag_blocks : (l == 1 ? end1 : (l == 2 ? end2 : end3))), L);
}
template <bool HASH>
__global__ void __launch_bounds__(kCoordBlock) flags_lookups(int flag_blocks, int end1, int end2, int end3, FlagsLookups a) {
    __shared__ LookupLds L;
    flags_lookups_block<HASH>(blockIdx.x, flag_blocks, end1, end2, end3, a, L);
}
template <int CIN, int COUT, typename T, typename TO>
__global__ void __launch_bounds__(kCoordBlock, (sizeof(T) == 4 ? 4 : CIN == 32 ? 5 : 7)) conv_tall_beside_flags_lookups(int gemm_blocks, int pads_at, int flag_blocks, int end1, int end2,
                                                                                              int end3, TallArgs g, FlagsLookups a) {
    __shared__ union {
        ProductLds<CIN, COUT, T> products;
        LookupLds lookups;
    } lds;
    const int b = blockIdx.x;
    if (b < gemm_blocks) return products_pass<CIN, COUT, T, TO>(g, b, gemm_blocks, lds.products);
    if (b >= pads_at) return products_pad_pass<CIN, COUT, T, TO>(g, b - pads_at, lds.products);
    flags_lookups_block<false>(b - gemm_blocks, flag_blocks, end1, end2, end3, a, lds.lookups);
}

// the flags alone (where the lookups on the rows behind them run on the other stream)
__global__ void __launch_bounds__(kCoordBlock) sp_flags(SpPart P) {
    __shared__ uint32_t lds4[4];
    sp_flags_pass(P, blockIdx.x, gridDim.x, lds4);
}

// ---------------------------------------------------------------------------------------------
// numbering, tile cuts
// ---------------------------------------------------------------------------------------------
// A block takes the chunks block, block + blocks, ...  All that its first chunk needs (words, cand, and the counts of the chunks in
// front of it) is requested before the row count is known, which says how many of the counts count: the pass is a chain of
// round trips to memory.  (A block at 45 874 input rows 15 000 -> 8 600 cycles: counts asked for one by one, two sums through LDS
// permutations, the divisions of a general stride prepared whatever the stride is.  The strided plugin 40.8 -> 36.9 us, frames of
// 60 000 points (FP16) 246 -> 240, 150 000 476 -> 461.)
constexpr int kCountsAhead = 8;  // counts that a thread asks for at a time: 2 048 chunks, 65 536 input rows of a 3x3x3 layer
__device__ __forceinline__ void sp_number_pass(const SpPart& a, const SpPart& next, bool has_next, int block, int blocks,
                                               uint32_t* lds, int4* s_rows, InsertLds& L) {
    const SpPart P = a;
    asm volatile("" :: "s"(P.words), "s"(P.cand), "s"(P.counts), "s"(P.in_num), "s"(P.max_voxels), "s"(P.Kc), "s"(P.t.base), "s"(P.t.dense), "s"(P.n_chunks),
                 "s"(P.out_coors), "s"(P.taken), "s"(P.nbr), "s"(next.halving), "s"(next.t.base), "s"(next.meta));
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint64_t w[4];
    uint32_t cand = 0, count[kCountsAhead];
    auto request = [&](int c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = P.words[c * 4 + q];
        cand = P.cand[(uint32_t)c * kCoordBlock + threadIdx.x];
    };
    auto request_counts = [&](int from, int end) {
#pragma unroll
        for (int q = 0; q < kCountsAhead; ++q) {
            const uint32_t j = (uint32_t)(from + q * kCoordBlock) + threadIdx.x;
            count[q] = P.counts[j < (uint32_t)end ? j : (uint32_t)end - 1];
        }
    };
    request(block);  // (in bounds: at most n_chunks blocks; not used where the chunk is beyond the active ones)
    request_counts(0, P.n_chunks);
    // Only the chunks that hold tickets of active input rows carry anything.
    const int n_in = __builtin_amdgcn_readfirstlane(clamp_rows(P.in_num, P.max_voxels));
    const int active = (int)(((int64_t)n_in * P.Kc + kCoordBlock - 1) / kCoordBlock);
    if (block >= active && block != 0) return;  // (no active input row at all: block 0 still owes the count)
    const CellView t = open_table(P.t, n_in);
    const uint32_t line = (uint32_t)P.os[2], plane = (uint32_t)P.os[1] * line;
    // the counts in front of the block's chunk: all of them for the first, then those it has stepped over (read anew for
    // every chunk they grew with the square of the rows: the strided plugin at 200 000 rows 146 -> 133 us, at 1 000 000
    // 800 -> 452)
    uint32_t before = 0;
    int n_out = 0, from = 0, to = active;
    for (int c = block; c < active || c == 0; c += blocks) {
        if (c != block) request(c);
        const bool first = c < active && ((w[wave] >> (threadIdx.x & 63)) & 1ull);
        const uint32_t slot = cand & kSlotMask;
        uint32_t key = 0;
        if (first) key = key_at(t, slot);
        uint32_t passed = 0, total = 0;
        for (int at = from; at < to; at += kCountsAhead * kCoordBlock) {
            if (c != block || at != 0) request_counts(at, to);
#pragma unroll
            for (int q = 0; q < kCountsAhead; ++q) {
                const int j = at + q * kCoordBlock + (int)threadIdx.x;
                const uint32_t v = j < to ? count[q] : 0;
                total += v;
                passed += j < c ? v : 0;
            }
        }
        from = c;
        to = c + blocks;
        block_sums(passed, total, lds);
        before += passed;
        if (c == block) n_out = (int)(total > (uint32_t)P.max_voxels ? (uint32_t)P.max_voxels : total);
        if (c == 0 && threadIdx.x == 0) {
            *P.out_num = n_out;
            if (P.taken) P.taken[0] = (uint32_t)n_out;
            P.meta[1] = n_out;
            // (the reference overflows its buffers; here the site is dropped)
            P.meta[0] = P.meta[2] | (total > (uint32_t)P.max_voxels ? SESSD_STATUS_VOXEL_OVERFLOW : 0);
            P.meta[2] = 0;
        }
        if (active == 0) return;
        uint32_t rank = rank_in_wave(w[wave]), here = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q < wave) rank += __popcll(w[q]);
            here += __popcll(w[q]);
        }
        if (first) {
            const uint32_t id = before + rank;
            if (id >= (uint32_t)P.max_voxels) {
                set_value(t, slot, kEmpty);
            } else {
                set_value(t, slot, id);  // from here on the table maps cell -> output row
                uint32_t rem, x;
                const uint32_t z = divide(key, plane, P.per_plane, rem), y = divide(rem, line, P.per_line, x);
                reinterpret_cast<int4*>(P.out_coors)[id] = make_int4(0, (int)z, (int)y, (int)x);  // sparseConv3dlayer.cu:438-441
                if (P.taken) P.taken[kCellListHead + id] = key;
                s_rows[rank] = make_int4((int)id, (int)z, (int)y, (int)x);
                // where sp_scatter fills the table in, the new row's entries start empty: clearing them here, row by
                // row, touches only the rows that exist
                if (P.nbr)
                    for (int k = 0; k < P.K; ++k) P.nbr[(size_t)k * P.max_voxels + id] = -1;
            }
        }
        if (has_next) {
            const int room = before >= (uint32_t)P.max_voxels ? 0 : (int)((uint32_t)P.max_voxels - before);
            __syncthreads();
            sp_insert_rows(next, open_table(next.t, n_out), s_rows, (int)here < room ? (int)here : room, L);
            __syncthreads();
        }
    }
}

// rows -> tile boundaries; 256 rows at a time
__device__ __forceinline__ void cut_pass(const CutPart& a, int block, uint32_t* lds) {
    const CutPart P = a;
    asm volatile("" :: "s"(P.num), "s"(P.max_voxels), "s"(P.w), "s"(P.wsum), "s"(P.hdr), "s"(P.num_cu), "s"(P.target), "s"(P.blocks));
    const int n = __builtin_amdgcn_readfirstlane(clamp_rows(P.num, P.max_voxels));
    if (n == 0) {
        if (block == 0 && threadIdx.x == 0) P.hdr[0] = 0;  // no cuts
        return;
    }
    const int groups = (n + 63) / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int tiles = tile_plan(n, P.wide ? P.num_cu >> wide_log2_split(n, P.K, P.num_cu) : P.num_cu, P.target).count;
    uint32_t* const s_wave = lds + 8;
    constexpr int kGroups = kCoordBlock / 64;  // sums of a chunk
    uint32_t before = 0, total = 0;  // weight before the chunk and of all rows
    for (int c = block; c * kCoordBlock < n; c += P.blocks) {
        const bool begin = c == block;
        uint32_t passed = 0, all = 0;
        for (int g = (begin ? 0 : (c - P.blocks) * kGroups) + (int)threadIdx.x; g < (begin ? groups : c * kGroups); g += kCoordBlock) {
            const uint32_t v = (uint32_t)P.wsum[g];
            all += v;
            if (g < c * kGroups) passed += v;
        }
        const int row = c * kCoordBlock + threadIdx.x;
        const int mine = row < n ? P.w[row] : 0;
        const int prev_w = row < n && row > 0 ? P.w[row - 1] : 0;
        block_sums(passed, all, lds);
        before += passed;
        if (begin) total = all;
        const uint32_t inc = wave_scan((uint32_t)mine);  // of the chunk's row weights, up to and with this one
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t excl = before + inc - (uint32_t)mine;  // weight of all rows before this one
        for (int v = 0; v < wave; ++v) excl += s_wave[v];
        // W is kept above the heaviest possible row: a row then advances the tile id by at most one, so every id
        // up to the last gets its start written (with few rows -- fewer than tiles -- total / tiles would fall
        // below a row's weight, ids would skip, and the skipped entries of the table would be read unwritten)
        uint32_t W = (total + (uint32_t)tiles - 1) / (uint32_t)tiles;
        W = W > (uint32_t)(kGemmMaxOffsets + P.row_weight) ? W : (uint32_t)(kGemmMaxOffsets + P.row_weight) + 1;
        if (row < n) {
            uint32_t rest;
            const int id = (int)divide(excl, W, reciprocal(W), rest);
            // the row before began in the tile before where its weight reaches back beyond this tile's first unit
            const int prev = row == 0 ? -1 : (rest >= (uint32_t)prev_w ? id : id - 1);
            int32_t* start = P.hdr + 4;
            if (id != prev) start[id] = row;  // ids grow by at most one per row (W exceeds every row weight)
            if (row == n - 1) {
                start[id + 1] = n;
                P.hdr[1] = (int)W;
                P.hdr[2] = (int)total;
                P.hdr[0] = id + 1;
            }
        }
        __syncthreads();
    }
}

template <int N>
struct NumberCuts {
    SpPart number, next;
    CutPart cut[kMaxCuts];
    CleanPart clean;
    FillPlan<N> also;
};

struct NumberLds {
    uint32_t sums[12];
    int4 rows[kCoordBlock];
    InsertLds insert;
};

// end0 .. end3: where the blocks of the cuts end, clean_end: those of the cleaning.
template <int N>
__device__ __forceinline__ void number_cuts_block(int b, int number_blocks, int has_next, int end0, int end1, int end2, int end3, int clean_end,
                                                  const NumberCuts<N>& a, NumberLds& L) {
    uint32_t* const lds = L.sums;
    if (b < number_blocks) return sp_number_pass(a.number, a.next, has_next != 0, b, number_blocks, lds, L.rows, L.insert);
    static_assert(kMaxCuts == 4, "an argument for each");
    if (b < end3) {
        const int l = __builtin_amdgcn_readfirstlane((b >= end0 ? 1 : 0) + (b >= end1 ? 1 : 0) + (b >= end2 ? 1 : 0));
        return cut_pass(a.cut[l], b - (l == 0 ? number_blocks : (l == 1 ? end0 : (l == 2 ? end1 : end2))), lds);
    }
    if (b < clean_end) return clean_pass(a.clean, b - end3);
    fill_pass(a.also, b - clean_end);
}
template <int N>
__global__ void __launch_bounds__(kCoordBlock) number_cuts(int number_blocks, int has_next, int end0, int end1, int end2, int end3, int clean_end,
                                                           NumberCuts<N> a) {
    __shared__ NumberLds L;
    number_cuts_block(blockIdx.x, number_blocks, has_next, end0, end1, end2, end3, clean_end, a, L);
}
// ... with a layer's products, whose blocks are the first of the grid (behind the numbering's instead: frames of 2 000 to 150 000 points, FP32
// and FP16, 0.994-1.004x)
template <int CIN, int COUT, typename T, typename TO>
__global__ void __launch_bounds__(kCoordBlock, 5) conv_tall_then_numbering(int gemm_blocks, int pads_at, int number_blocks, int has_next, int end0, int end1, int end2,
                                                                     int end3, int clean_end, TallArgs g, NumberCuts<1> a) {
    __shared__ union {
        ProductLds<CIN, COUT, T> products;
        NumberLds number;
    } lds;
    const int b = blockIdx.x;
    if (b < gemm_blocks) return products_pass<CIN, COUT, T, TO>(g, b, gemm_blocks, lds.products);
    if (b >= pads_at) return products_pad_pass<CIN, COUT, T, TO>(g, b - pads_at, lds.products);
    number_cuts_block(b - gemm_blocks, number_blocks, has_next, end0, end1, end2, end3, clean_end, a, lds.number);
}

// rulebook of a strided layer on its own: one store per ticket into the rows sp_number has initialised
__global__ void __launch_bounds__(kCoordBlock) sp_scatter(SpPart P) {
    const int n = clamp_rows(P.in_num, P.max_voxels);
    const CellView t = open_table(P.t, n);
    const int64_t tickets = (int64_t)n * P.Kc;
    for (int64_t tk = (int64_t)blockIdx.x * kCoordBlock + threadIdx.x; tk < tickets; tk += (int64_t)gridDim.x * kCoordBlock) {
        const uint32_t c = P.cand[tk];
        if (c == kEmpty) continue;
        const uint32_t id = value_at(t, c & kSlotMask);
        if (id == kEmpty) continue;
        P.nbr[(size_t)(c >> kSlotBits) * P.max_voxels + id] = (int32_t)(tk / P.Kc);  // unique (offset, out row): plain store
    }
}

// weights of the rows of a rulebook that was scattered: 256 rows per block, four threads per row (each sums every
// fourth offset)
constexpr int kSplit = 4;
__global__ void __launch_bounds__(kCoordBlock * kSplit)
tile_weights(const int32_t* __restrict__ nbr, const int32_t* __restrict__ num_out, int max_voxels, int K, int row_weight,
             int32_t* __restrict__ w, int32_t* __restrict__ wsum) {
    __shared__ int32_t s_cnt[kSplit][kCoordBlock];
    const int n = clamp_rows(num_out, max_voxels);
    if ((int)blockIdx.x * kCoordBlock >= n) return;
    const int r = threadIdx.x % kCoordBlock, kg = threadIdx.x / kCoordBlock;
    const int row = blockIdx.x * kCoordBlock + r;
    int c = 0;
    if (row < n) {
        constexpr int kPer = (kGemmMaxOffsets + kSplit - 1) / kSplit;
        int32_t e[kPer];  // all loads of the thread are requested before the first is used
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int k = kg + j * kSplit;
            e[j] = k < K ? nbr[(size_t)k * max_voxels + row] : -1;
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j) c += e[j] >= 0 ? 1 : 0;
    }
    s_cnt[kg][r] = c;
    __syncthreads();
    if (kg != 0) return;
    int v = 0;
    if (row < n) {
        v = row_weight;
#pragma unroll
        for (int g = 0; g < kSplit; ++g) v += s_cnt[g][r];
    }
    if (row < max_voxels) w[row] = v;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    if ((r & 63) == 0 && row < n) wsum[row >> 6] = v;
}

}  // namespace

int sp_pass_blocks(const SpPart& s) { return s.n_chunks < kMaxPassBlocks ? s.n_chunks : kMaxPassBlocks; }
int lookup_blocks(int max_voxels) {
    const int b = ceil_div(max_voxels, kLookupRows);
    return b < kMaxPassBlocks ? b : kMaxPassBlocks;
}

static int clean_blocks(int max_voxels) {
    const int b = ceil_div(max_voxels, kCoordBlock);
    return b < 128 ? b : 128;
}

template <int N>
static int vg_insert_n(const VgPart& v, const Cleans& cleans, int n_clean_blocks, const FillArgs& also, hipStream_t stream) {
    FillPlan<N> plan;
    const int blocks = make_fill_plan(also, plan);
    if (blocks < 0) return fail(SESSD_E_INVALID, "fill: a region is not 16-byte aligned");
    hipLaunchKernelGGL(vg_insert<N>, dim3(v.n_blocks + n_clean_blocks + blocks), dim3(kCoordBlock), 0, stream, v, cleans, plan);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}
int launch_vg_insert(const VgPart& v, const CleanPart* cleans, int n_cleans, const FillArgs& also, hipStream_t stream) {
    if (n_cleans < 0 || n_cleans > kMaxCleans) return fail(SESSD_E_INVALID, "vg_insert: at most %d tables are cleaned beside it", kMaxCleans);
    Cleans c;
    c.n = n_cleans;
    int total = 0;
    for (int i = 0; i < n_cleans; ++i) {
        c.c[i] = cleans[i];
        c.c[i].blocks = clean_blocks(cleans[i].max_voxels);
        total += c.c[i].blocks;
    }
    return also.n <= kFewRegions ? vg_insert_n<kFewRegions>(v, c, total, also, stream)
                                 : vg_insert_n<FillArgs::kMaxRegions>(v, c, total, also, stream);
}

template <int N>
static int vg_flags_n(const VgPart& v, const FillArgs& also, hipStream_t stream) {
    FillPlan<N> plan;
    const int blocks = make_fill_plan(also, plan);
    if (blocks < 0) return fail(SESSD_E_INVALID, "fill: a region is not 16-byte aligned");
    hipLaunchKernelGGL(vg_flags<N>, dim3(v.n_blocks + blocks), dim3(kCoordBlock), 0, stream, v, plan);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}
int launch_vg_flags(const VgPart& v, const FillArgs& also, hipStream_t stream) {
    return also.n <= kFewRegions ? vg_flags_n<kFewRegions>(v, also, stream) : vg_flags_n<FillArgs::kMaxRegions>(v, also, stream);
}

int launch_vg_finalize(const VgPart& v, const SpPart* next, hipStream_t stream) {
    hipLaunchKernelGGL(vg_finalize, dim3(ceil_div(v.max_points, kFinalPoints)), dim3(kCoordBlock), 0, stream, v,
                       next ? *next : SpPart(), next ? 1 : 0);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

int launch_sp_insert(const SpPart& s, hipStream_t stream) {
    const int per = kTicketsAtOnce / s.Kc > 0 ? kTicketsAtOnce / s.Kc : 1;
    const int blocks = ceil_div(s.max_voxels, per);
    hipLaunchKernelGGL(sp_insert, dim3(blocks < 2 * kMaxPassBlocks ? blocks : 2 * kMaxPassBlocks), dim3(kCoordBlock), 0, stream, s);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

// (finite weights, 32-bit offsets, ... : tall_takes())
bool number_takes_products(const GemmArgs& a) { return a.cin == 4 && !a.dense.dense && tall_takes(a); }
bool lookups_take_products(const GemmArgs& a, const LookupPart* lookups, int n) {
    for (int l = 0; l < n; ++l)
        if (!lookups[l].t.dense) return false;
    return n <= kMaxLookups && a.cin == a.cout && (a.cin == 16 || (a.cin == 32 && a.in_type == SESSD_HALF)) && !a.dense.dense && tall_takes(a);
}

static int flags_lookups_launch(const SpPart* flags, const LookupPart* lookups, int n, const GemmArgs* products, hipStream_t stream) {
    if (n < 0 || n > kMaxLookups) return fail(SESSD_E_INVALID, "lookups: at most %d in one launch", kMaxLookups);
    FlagsLookups a;
    int flag_blocks = 0;
    if (flags) {
        a.flags = *flags;
        flag_blocks = sp_pass_blocks(*flags);
    }
    int blocks = flag_blocks, end[kMaxLookups];
    for (int l = 0; l < kMaxLookups; ++l) {
        if (l < n) {
            LookupPart& p = a.look[l];
            p = lookups[l];
            p.blocks = lookup_blocks(p.max_voxels);
            const int per = (p.K + 3) >> 2;  // (offsets of a wave)
            for (int w = 0; w < 4; ++w) {
                const int k = w * per;
                p.first[w] = (k / (p.k[1] * p.k[2])) << 16 | (k / p.k[2] % p.k[1]) << 8 | k % p.k[2];
            }
            blocks += p.blocks;
        }
        end[l] = blocks;
    }
    if (!blocks && !products) return SESSD_OK;
    if (products) {
        if (!lookups_take_products(*products, lookups, n)) return fail(SESSD_E_UNSUPPORTED, "lookups: a layer's products cannot share this launch");
        const TallArgs g = tall_args(*products);
        const int gemm_blocks = product_blocks(*products), pads_at = gemm_blocks + blocks;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(pads_at + (products->write_pad_rows ? kPadBlocks : 0)), dim3(kCoordBlock), 0, stream, gemm_blocks, pads_at, flag_blocks, end[0],
                               end[1], end[2], g, a);
        };
        if (products->cin == 32) go(conv_tall_beside_flags_lookups<32, 32, __half, __half>);
        else products->in_type == SESSD_HALF ? go(conv_tall_beside_flags_lookups<16, 16, __half, __half>) : go(conv_tall_beside_flags_lookups<16, 16, float, float>);
        SESSD_HIP_TRY(hipGetLastError());
        return SESSD_OK;
    }
    bool hash = false;  // (the flags read either kind of table)
    for (int l = 0; l < n; ++l) hash = hash || !lookups[l].t.dense;
    if (hash) hipLaunchKernelGGL(flags_lookups<true>, dim3(blocks), dim3(kCoordBlock), 0, stream, flag_blocks, end[0], end[1], end[2], a);
    else hipLaunchKernelGGL(flags_lookups<false>, dim3(blocks), dim3(kCoordBlock), 0, stream, flag_blocks, end[0], end[1], end[2], a);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

int launch_flags_lookups(const SpPart* flags, const LookupPart* lookups, int n, hipStream_t stream) {
    return flags_lookups_launch(flags, lookups, n, nullptr, stream);
}
int launch_flags_lookups_products(const SpPart* flags, const LookupPart* lookups, int n, const GemmArgs& products, hipStream_t stream) {
    return flags_lookups_launch(flags, lookups, n, &products, stream);
}

int launch_sp_flags(const SpPart& s, hipStream_t stream) {
    hipLaunchKernelGGL(sp_flags, dim3(sp_pass_blocks(s)), dim3(kCoordBlock), 0, stream, s);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

static int number_launch(const SpPart* number, const SpPart* next, const CutPart* cuts, int n_cuts, const CleanPart* clean, const FillArgs* also,
                         const GemmArgs* products, hipStream_t stream) {
    if (n_cuts < 0 || n_cuts > kMaxCuts) return fail(SESSD_E_INVALID, "tile cuts: at most %d in one launch", kMaxCuts);
    NumberCuts<1> a;
    int number_blocks = 0, has_next = 0;
    if (number) {
        a.number = *number;
        a.number.per_line = reciprocal((uint32_t)number->os[2]);
        a.number.per_plane = reciprocal((uint32_t)number->os[1] * (uint32_t)number->os[2]);
        number_blocks = sp_pass_blocks(*number);
        if (next) {
            a.next = *next;
            has_next = 1;
        }
    }
    int blocks = number_blocks, end[kMaxCuts];
    for (int l = 0; l < kMaxCuts; ++l) {
        if (l < n_cuts) {
            a.cut[l] = cuts[l];
            blocks += a.cut[l].blocks;
        }
        end[l] = blocks;
    }
    if (clean) {
        a.clean = *clean;
        a.clean.blocks = clean_blocks(clean->max_voxels);
        blocks += a.clean.blocks;
    }
    const int clean_end = blocks;
    FillArgs none;
    if (also && also->n > 1) return fail(SESSD_E_INVALID, "numbering: one region can be cleared beside it");
    const int fill_blocks = make_fill_plan(also ? *also : none, a.also);
    if (fill_blocks < 0) return fail(SESSD_E_INVALID, "fill: a region is not 16-byte aligned");
    blocks += fill_blocks;
    if (!blocks && !products) return SESSD_OK;
    if (products) {
        if (!number_takes_products(*products)) return fail(SESSD_E_UNSUPPORTED, "numbering: a layer's products cannot share this launch");
        const TallArgs g = tall_args(*products);
        const int gemm_blocks = product_blocks(*products), pads_at = gemm_blocks + blocks;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(pads_at + (products->write_pad_rows ? kPadBlocks : 0)), dim3(kCoordBlock), 0, stream, gemm_blocks, pads_at, number_blocks,
                               has_next, end[0], end[1], end[2], end[3], clean_end, g, a);
        };
        const bool half = products->out_type == SESSD_HALF, narrow = products->cout == 16;
        if (half) narrow ? go(conv_tall_then_numbering<4, 16, float, __half>) : go(conv_tall_then_numbering<4, 32, float, __half>);
        else narrow ? go(conv_tall_then_numbering<4, 16, float, float>) : go(conv_tall_then_numbering<4, 32, float, float>);
    } else {
        hipLaunchKernelGGL(number_cuts<1>, dim3(blocks), dim3(kCoordBlock), 0, stream, number_blocks, has_next, end[0], end[1], end[2], end[3], clean_end, a);
    }
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}
int launch_number(const SpPart* number, const SpPart* next, const CutPart* cuts, int n_cuts, const CleanPart* clean, const FillArgs* also,
                  hipStream_t stream) {
    return number_launch(number, next, cuts, n_cuts, clean, also, nullptr, stream);
}
int launch_number_products(const SpPart* number, const SpPart* next, const CutPart* cuts, int n_cuts, const CleanPart* clean, const FillArgs* also,
                           const GemmArgs& products, hipStream_t stream) {
    return number_launch(number, next, cuts, n_cuts, clean, also, &products, stream);
}

int launch_sp_scatter(const SpPart& s, hipStream_t stream) {
    hipLaunchKernelGGL(sp_scatter, dim3(sp_pass_blocks(s)), dim3(kCoordBlock), 0, stream, s);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

int launch_tile_weights(const int32_t* nbr, const int32_t* num_out, int K, int max_voxels, int row_weight, void* region, hipStream_t stream) {
    hipLaunchKernelGGL(tile_weights, dim3(ceil_div(max_voxels, kCoordBlock)), dim3(kCoordBlock * kSplit), 0, stream, nbr, num_out,
                       max_voxels, K, row_weight, tile_weight_array(region, max_voxels), tile_weight_sums(region, max_voxels));
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

}  // namespace sessd
