// coord.h -- the coordinate side of the path: cell tables, and the passes over points, tickets and rows that turn a
// frame's points into voxels, a layer's sites and its rulebook.  Each pass is a device function over "its" blocks, so
// that a plugin can launch it alone and the frame pipeline can put independent passes into one launch (coord.hip).
//
// A frame's coordinate work is a chain of small dependent steps; at 20 000 points a launch that does one of them takes
// 3-8 us, of which 2 are the launch itself.  The chain is therefore as short as its dependences allow:
//     insert(points) | flags | number + insert(stage 2) | flags + lookups | number + insert(stage 3) | ...
#pragma once

#include "kernels.h"

namespace sessd {

// ---------------------------------------------------------------------------------------------
// cell tables
// ---------------------------------------------------------------------------------------------
// cell key (z*gy + y)*gx + x -> 32-bit value (a point index or ticket while rows are being found, the row afterwards).
// Two forms:
//   hash   open addressing over 64-bit entries (key << 32 | value), all ones = empty: one atomic inserts a cell with its
//          value, one load answers a probe.  Only the slots that `rows` input rows can need are used (per_row16), so
//          a table allocated for a large capacity still fits the L2 of an XCD when the frame is small.
//   dense  one word per cell: no probing, and the three x-neighbours of a cell lie in one line.
// Multiplicative hashing spreads the strongly correlated keys of neighbouring cells; linear probing keeps a probe
// sequence inside one or two cache lines.  Every loop is bounded by the table: a full one is reported, never spun on.
struct CellTable {
    void* base = nullptr;
    uint32_t cap = 0;       // hash: slots allocated (a power of two); dense: cells
    int32_t dense = 0;
    int32_t per_row16 = 0;  // hash: slots per input row, in sixteenths
    int32_t gx = 0, gy = 0, gz = 0;
    size_t words() const { return dense ? cap : (size_t)cap * 2; }
};

// A table that an enqueue clears anew: one word per cell where that is at most twice the hash's bytes, or 8 MB (a fill of
// 1.2 us).  An insert is then one atomic without an answer and a lookup one load: at 17 000 rows 2 + 6 us where the
// probing of the hash takes 4 + 12.
inline bool dense_pays(uint64_t volume, uint64_t hash_bytes) {
    const uint64_t most = 2 * hash_bytes > (8u << 20) ? 2 * hash_bytes : (8u << 20);
    return volume * 4 <= most;
}

#ifdef __HIPCC__
constexpr int kCoordBlock = 256;  // threads of every pass

struct CellView {
    unsigned long long* h;  // hash entries, or null
    uint32_t* d;            // dense cells, or null
    uint32_t mask;
    int32_t shift;
};

__device__ __forceinline__ CellView open_table(const CellTable& t, int rows) {
    CellView v;
    v.h = t.dense ? nullptr : static_cast<unsigned long long*>(t.base);
    v.d = t.dense ? static_cast<uint32_t*>(t.base) : nullptr;
    unsigned long long need = (unsigned long long)rows * (unsigned)t.per_row16 / 16u;
    need = need < 32 ? 32 : need;  // (whole groups)
    int lg = 64 - __clzll(need - 1);
    const int most = 31 - __clz((int)t.cap);
    lg = lg < most ? lg : most;
    v.mask = (1u << lg) - 1u;
    v.shift = 32 - lg;
    return v;
}

constexpr unsigned long long kEmptyEntry = ~0ull;
__device__ __forceinline__ unsigned long long make_entry(uint32_t key, uint32_t val) {
    return ((unsigned long long)key << 32) | val;
}
__device__ __forceinline__ uint32_t entry_key(unsigned long long e) { return (uint32_t)(e >> 32); }
__device__ __forceinline__ uint32_t entry_val(unsigned long long e) { return (uint32_t)e; }
__device__ __forceinline__ uint32_t first_slot(const CellView& t, uint32_t key) { return (key * 2654435769u) >> t.shift; }

// Four entries that lie in one 32-byte sector; a probe sequence walks through its first group from its first slot on.
constexpr int kGroup = 4;
struct EntryGroup {
    unsigned long long e[kGroup];
};
__device__ __forceinline__ EntryGroup load_group(const CellView& t, uint32_t slot) {
    const ulonglong2* p = reinterpret_cast<const ulonglong2*>(t.h + (slot & ~(uint32_t)(kGroup - 1)));
    const ulonglong2 a = p[0], b = p[1];
    return {{a.x, a.y, b.x, b.y}};
}
// Where an insert of `key` should try first: the key itself or an empty entry in the group of its first slot, else the
// slot behind the group.  The group may be older than the table: an entry it shows as taken is taken, one it shows as
// empty may no longer be, which the atomic then says.
__device__ __forceinline__ uint32_t likely_slot(const CellView& t, uint32_t key, const EntryGroup& g) {
    const uint32_t first = first_slot(t, key), base = first & ~(uint32_t)(kGroup - 1);
    uint32_t at = (base + kGroup) & t.mask;
#pragma unroll
    for (int e = kGroup - 1; e >= 0; --e)
        if (e >= (int)(first & (kGroup - 1)) && (g.e[e] == kEmptyEntry || entry_key(g.e[e]) == key)) at = base + e;
    return at;
}

// slot of `key` with the smaller of its old value and `val`, -1 when the table is full; `prev` = what an
// atomicCAS(empty -> entry) on slot `at` has returned (issued by the caller, so that several can be in flight)
__device__ __forceinline__ int32_t finish_insert_min(const CellView& t, uint32_t key, uint32_t val, uint32_t at, unsigned long long prev) {
    const unsigned long long e = make_entry(key, val);
    for (uint32_t probe = 0; probe <= t.mask; ++probe) {
        if (prev == kEmptyEntry) return (int32_t)at;
        if (entry_key(prev) == key) {
            if (entry_val(prev) > val) atomicMin(&t.h[at], e);
            return (int32_t)at;
        }
        at = (at + 1) & t.mask;
        prev = atomicCAS(&t.h[at], kEmptyEntry, e);
    }
    return -1;
}
__device__ __forceinline__ int32_t insert_min(const CellView& t, uint32_t key, uint32_t val) {
    if (t.d) {
        atomicMin(&t.d[key], val);
        return (int32_t)key;
    }
    const uint32_t at = likely_slot(t, key, load_group(t, first_slot(t, key)));
    return finish_insert_min(t, key, val, at, atomicCAS(&t.h[at], kEmptyEntry, make_entry(key, val)));
}

// a slot (hash) or cell (dense) that an insert returned
__device__ __forceinline__ uint32_t value_at(const CellView& t, uint32_t slot) {
    return t.d ? t.d[slot] : reinterpret_cast<const uint32_t*>(t.h)[2 * (size_t)slot];
}
__device__ __forceinline__ uint32_t key_at(const CellView& t, uint32_t slot) {
    return t.d ? slot : reinterpret_cast<const uint32_t*>(t.h)[2 * (size_t)slot + 1];
}
__device__ __forceinline__ void set_value(const CellView& t, uint32_t slot, uint32_t val) {
    if (t.d) t.d[slot] = val;
    else reinterpret_cast<uint32_t*>(t.h)[2 * (size_t)slot] = val;
}

__device__ __forceinline__ int clamp_rows(const int32_t* p, int cap) {
    const int n = *p;
    return n < 0 ? 0 : (n > cap ? cap : n);
}
// Sum over the lanes up to and with this one.  (Data-parallel moves between lanes: six additions, where a sum by __shfl is six trips
// through LDS, some 700 cycles.)
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1, 2, 4, 8: sums in rows of 16
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15: the row before, into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31: both rows before, into rows 2 and 3
    return v;
}
// sums of a and b over the block, returned to every thread; lds: eight words
__device__ __forceinline__ void block_sums(uint32_t& a, uint32_t& b, uint32_t* lds) {
    a = wave_scan(a);
    b = wave_scan(b);
    __syncthreads();
    if ((threadIdx.x & 63) == 63) {
        lds[threadIdx.x >> 6] = a;
        lds[4 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    a = lds[0] + lds[1] + lds[2] + lds[3];
    b = lds[4] + lds[5] + lds[6] + lds[7];
}
// n / d for inv = reciprocal(d): off by one at most before the correction, as d * inv is within d of 2^32
__host__ __device__ inline uint32_t reciprocal(uint32_t d) { return 0xffffffffu / d; }
__device__ __forceinline__ uint32_t divide(uint32_t n, uint32_t d, uint32_t inv, uint32_t& rest) {
    uint32_t q = __umulhi(n, inv);
    rest = n - q * d;
    if (rest >= d) {
        rest -= d;
        ++q;
    }
    return q;
}
#endif

// ---------------------------------------------------------------------------------------------
// what the passes work on (kernel arguments)
// ---------------------------------------------------------------------------------------------
// The cells that a frame's rows have taken in a table that is kept for the next frame: what empties the table goes by
// this list.  The coors tensor names the same cells, but callers get pointers to it.
// One pointer (kernels that pass two layers are short of scalar registers): [0] the number of cells, [kCellListHead ..]
// their keys.  Null: no list is kept.
typedef uint32_t* CellList;
constexpr int kCellListHead = 64;

// Every 64 points of vg_finalize need the counts of all 256-point blocks.  Beyond a million points the blocks read their
// sums over 64 instead: reading them all grows with the square of the points (the plugin at
// 2 400 000 points 452 -> 353 us, at 1 200 000 189 -> 176); below, the atomics that make the sums cost more than they
// save (at 600 000 97 -> 101).
constexpr int kCountsPerSum = 64, kSumsFromPoints = 1 << 20;
struct VgPart {
    const float* points = nullptr;
    const int32_t* points_size = nullptr;
    int max_points = 0, pf = 0;
    float min_x, max_x, min_y, max_y, min_z, max_z, vx, vy, vz;
    int gx, gy, gz;
    int max_voxels;
    int max_pts;  // S: points averaged per voxel
    CellTable t;  // cell -> smallest point index, then voxel row
    uint32_t* slots = nullptr;  // [max_points][S - 1], all kEmpty between enqueues: the smallest later points of the cell
                                // whose first point this is, ascending
    int32_t* pt_slot = nullptr;
    uint64_t* words = nullptr;
    uint32_t* counts = nullptr;
    uint32_t* sums = nullptr;  // null, or the sums of the counts of kCountsPerSum blocks
    int n_blocks = 0;
    float* voxels = nullptr;
    int32_t* coors = nullptr;
    int32_t* voxel_num = nullptr;
    CellList taken = nullptr;
    int32_t* status = nullptr;  // [0] status, [1] what vg_insert has met (folded into [0] and cleared by vg_finalize)
};

// A strided layer.  Ticket t = input row * Kc + candidate.
struct SpPart {
    int k[3], s[3], p[3], os[3];  // z,y,x
    int Kc = 0;                   // enumeration slots per input row
    int halving = 0;              // kernels of 3 and strides of 2 on every axis (Kc = 8)
    int max_voxels = 0;           // rows of the input and of the output tensors
    int K = 0;
    CellTable t;  // output cell -> smallest ticket, then output row
    uint32_t* cand = nullptr;
    uint64_t* words = nullptr;
    uint32_t* counts = nullptr;
    int n_chunks = 0;  // 256-ticket chunks at capacity
    uint32_t per_plane = 0, per_line = 0;  // reciprocal() of the output grid's cells a plane and a line (launch_number())
    const int32_t* in_coors = nullptr;
    const int32_t* in_num = nullptr;
    int32_t* out_coors = nullptr;
    int32_t* out_num = nullptr;
    CellList taken = nullptr;
    int32_t* nbr = nullptr;   // null: the rulebook is looked up (LookupPart), sp_number has nothing to initialise
    int32_t* meta = nullptr;  // [0] status, [1] output rows, [2] what sp_insert has met (folded into [0] by sp_number)
};

// Rulebook by lookup: nbr[k][row] = row of the input cell  out*s - p + k  in `t`.  SubM layers (s = 1, t = the table of
// their own rows) and, in the pipeline, strided layers (t = the table of their input rows).
struct LookupPart {
    const int32_t* coors = nullptr;  // of the output rows
    const int32_t* num = nullptr;
    int max_voxels = 0;
    int k[3], s[3], p[3];  // z,y,x
    int K = 0;
    int first[4];  // first offset of each quarter: z << 16 | y << 8 | x (launch_flags_lookups())
    int own[3];  // the layer's grid (z,y,x): a row outside it has no neighbours
    CellTable t;
    const int32_t* t_num = nullptr;  // rows the table was opened with
    int t_max = 0;
    int32_t* nbr = nullptr;
    int32_t* meta = nullptr;  // null, or [1] <- rows
    int32_t* w = nullptr;     // null, or the rows' weights for the tile cuts and their sums over 64 rows
    int32_t* wsum = nullptr;
    int row_weight = 0;
    int blocks = 0;
};

struct CutPart {
    const int32_t* num = nullptr;
    int max_voxels = 0, K = 0, num_cu = 0, target = 0, row_weight = 0, wide = 0;
    const int32_t* w = nullptr;
    const int32_t* wsum = nullptr;
    int32_t* hdr = nullptr;
    int blocks = 0;
};

// the weight arrays inside a rulebook's tile region (tile_cut_bytes())
int32_t* tile_weight_array(void* region, int max_voxels);
int32_t* tile_weight_sums(void* region, int max_voxels);
CutPart make_cut_part(const int32_t* num_out, int K, int max_voxels, int target_rows, int row_weight, int wide, void* region);

// A dense table that stays from frame to frame: emptied cell by cell instead of by a fill of its whole volume.
struct CleanPart {
    CellList taken = nullptr;
    int max_voxels = 0;
    CellTable t;
    int blocks = 0;
};

constexpr int kMaxLookups = 4, kMaxCuts = 4, kMaxCleans = 4;
constexpr int kMaxPassBlocks = 1024;  // blocks of a pass over tickets or rows; each takes several chunks beyond that
int sp_pass_blocks(const SpPart& s);
int lookup_blocks(int max_voxels);

// launches (coord.hip)
int launch_vg_insert(const VgPart& v, const CleanPart* cleans, int n_cleans, const FillArgs& also,
                     hipStream_t stream);  // `also`: regions cleared beside it
int launch_vg_flags(const VgPart& v, const FillArgs& also, hipStream_t stream);
int launch_vg_finalize(const VgPart& v, const SpPart* next, hipStream_t stream);  // next: its tickets are inserted
int launch_sp_insert(const SpPart& s, hipStream_t stream);
int launch_flags_lookups(const SpPart* flags, const LookupPart* lookups, int n, hipStream_t stream);
int launch_number(const SpPart* number, const SpPart* next, const CutPart* cuts, int n_cuts, const CleanPart* clean, const FillArgs* also,
                  hipStream_t stream);
// ... the same passes with a layer's products in the launch: whether it can be so, and the launches
bool number_takes_products(const GemmArgs& a);
bool lookups_take_products(const GemmArgs& a, const LookupPart* lookups, int n);
int launch_flags_lookups_products(const SpPart* flags, const LookupPart* lookups, int n, const GemmArgs& products, hipStream_t stream);
int launch_number_products(const SpPart* number, const SpPart* next, const CutPart* cuts, int n_cuts, const CleanPart* clean, const FillArgs* also,
                           const GemmArgs& products, hipStream_t stream);
int launch_sp_flags(const SpPart& s, hipStream_t stream);
int launch_sp_scatter(const SpPart& s, hipStream_t stream);
int launch_tile_weights(const int32_t* nbr, const int32_t* num_out, int K, int max_voxels, int row_weight, void* region, hipStream_t stream);

}  // namespace sessd
