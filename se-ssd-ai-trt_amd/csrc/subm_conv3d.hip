// subm_conv3d.hip -- SubmConv3dLayerPlugin: submanifold 3-D convolution.
//
// Replaces submConv3dlayer.cu:271-641.  The reference memsets a dense int grid over the whole volume
// (369 MB at 41x1600x1408), materialises 27 candidate positions per voxel, appends rulebook pairs
// with atomicAdd and then launches the GEMM kernel 27 times.  Here:
//
//   subm_insert      one thread per active voxel: cell key -> hash table (value = voxel row)
//   lookups          nbr[k][o] = the row in cell o - padding + k, all offsets of a row at once (coord.hip)
//   gather-GEMM      one launch for all offsets
//
// nbr[k][o] is the rulebook: the pair (i, o) is in the reference's list of offset k exactly when
// nbr[k][o] == i.  sessd_submconv3d_export_rulebook compacts it into the reference's layout.
#include "coord.h"
#include "plugins.h"

namespace sessd {

namespace {

constexpr int kBlock = 256;

struct Grid3 {
    int X, Y, Z;
};

// submConv3dlayer.cu:441-459 (prepareSubMGridKernel) with the dense grid replaced by a hash
__global__ void __launch_bounds__(kBlock)
subm_insert(const int32_t* __restrict__ coors, const int32_t* __restrict__ voxel_num, int max_voxels,
            Grid3 g, CellTable table, int32_t* meta) {
    const int v = blockIdx.x * kBlock + threadIdx.x;
    const int n = clamp_rows(voxel_num, max_voxels);
    if (v >= n) return;
    const int4 c = reinterpret_cast<const int4*>(coors)[v];  // (b,z,y,x)
    if (c.y < 0 || c.y >= g.Z || c.z < 0 || c.z >= g.Y || c.w < 0 || c.w >= g.X) {
        atomicOr(&meta[0], SESSD_STATUS_BAD_COORD);  // the reference would write outside its grid
        return;
    }
    const uint32_t key = ((uint32_t)c.y * (uint32_t)g.Y + (uint32_t)c.z) * (uint32_t)g.X + (uint32_t)c.w;
    if (insert_min(open_table(table, n), key, (uint32_t)v) < 0) atomicOr(&meta[0], SESSD_STATUS_HASH_FULL);
}

// The whole rulebook of a layer of few rows in one launch: every workgroup keeps the cells of all rows in a hash table of its own,
// in LDS, and looks up the neighbours of 64 rows.  Clearing, filling and reading a table in memory are three launches, which is what
// a small layer spends its time on.  For each hash value the table holds the first row that has it and a list of the rows of other
// cells: a row enters with one minimum and, where cells collide, one exchange (the probes of an open table, each waiting for the one
// before, took 8 us for 2 000 rows).  Rows that name one cell are in no list: as one, which each of them walked, 8 192 of them were
// a layer of 882 us, 17 now.  What bounds it are two trips to memory and the launch.  Layer 4 -> 16, three launches before and this: 300 rows 19.0 -> 11.4
// us, 2 000 18.6 -> 11.5, 8 000 19.5 -> 13.0 (then with a launch for the products); 64 -> 64 with 8 000 rows 26.4 -> 22.  The line lies where the table still fits LDS: 8 192 rows and
// their lists, 128 KB.  It is drawn at the tensors' capacity, which is what the host knows when it launches.
constexpr int kSmallRows = 8192;
constexpr int kSmallHeads = 16384;
constexpr int kSmallBlock = 1024;
constexpr int kSmallWaves = kSmallBlock / 64;
constexpr int kSmallOwn = kSmallRows / kSmallBlock;                                 // rows that a thread enters
constexpr int kSmallDepth = (kGemmMaxOffsets + kSmallWaves - 1) / kSmallWaves;  // offsets that it looks up
static_assert(kSmallRows < 0xffff, "rows in 16 bits beside kNoRow");

// The layer behind such a rulebook where its products are plain FP32 and few: the workgroup that has looked up the neighbours of its 64
// rows multiplies them as well.  What bounds a call of two launches is the host, which takes 3.4 us for each, from 2 000 rows up the
// GPU, where the second one's trips to memory (row count, lists, rows) are gone but for the rows.  A wave takes 16 of the rows and a
// quarter of the offsets, whose weights it has asked for in front of everything else; an absent neighbour's product is left out behind
// the MFMA (0 x infinity).  An offset's products are summed by themselves, the sums of offsets and of the four quarters two by two.
// Two launches / one, a call: 4 -> 16 at 300 rows 10.9 / 8.1 us, 2 000 10.9 / 7.8, 8 000 13.9 / 11.0; 4 -> 32 10.8 / 7.7, 11.9 / 8.5,
// 15.9 / 11.6; 16 -> 16 11.0 / 8.2, 11.0 / 9.1, 14.7 / 12.0.  Not 16 -> 32, 10.9 / 11.7, 11.5 / 12.8, 15.9 / 16.2: every 64 rows wait for 54 KB
// of weights, and the registers spill.  Distance from 64-bit sums at 2 000 rows 3.58e-8 / 3.58e-8, 3.53e-8 / 3.53e-8, 6.04e-8 / 6.04e-8.
struct SmallGemm {
    const float* in = nullptr;
    float* out = nullptr;
    const float* w = nullptr;  // operand order (pack_weights())
    const float* scale = nullptr;
    const float* shift = nullptr;
    int relu = 0, write_pad = 0;
};
constexpr int kSmallQuarters = 4, kSmallQuarter = (kGemmMaxOffsets + kSmallQuarters - 1) / kSmallQuarters;  // offsets of a quarter
static_assert(kSmallWaves == 4 * kSmallQuarters, "a wave for each 16 rows and quarter");

__device__ __forceinline__ void small_operand(const float* from, float (&v)[1]) { v[0] = from[0]; }
__device__ __forceinline__ void small_operand(const float* from, float (&v)[4]) {
    const float4 t = *reinterpret_cast<const float4*>(from);
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
}

// four output elements of a row
__device__ __forceinline__ float4 small_epilogue(const SmallGemm& g, float4 v, const float4& scale, const float4& shift) {
    float o[4] = {v.x, v.y, v.z, v.w};
    const float sc[4] = {scale.x, scale.y, scale.z, scale.w}, sh[4] = {shift.x, shift.y, shift.z, shift.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (g.scale) o[e] = o[e] * sc[e];
        if (g.shift) o[e] = o[e] + sh[e];
        if (g.relu) o[e] = o[e] > 0.f ? o[e] : 0.f;
    }
    return make_float4(o[0], o[1], o[2], o[3]);
}

// CIN 0: the rulebook alone
template <int CIN, int COUT>
__global__ void __launch_bounds__(kSmallBlock)
subm_small(LookupPart P, int32_t* __restrict__ tiles, SmallGemm G) {
    constexpr uint32_t kNoRow = 0xffffu;
    constexpr bool kGemm = CIN > 0;
    constexpr int E = kGemm ? CIN / 4 : 1, NB = kGemm ? COUT / 16 : 1, kVecs = kGemm ? COUT / 4 : 1;
    __shared__ __align__(16) uint32_t s_head[kSmallHeads];  // of a hash value: first row << 16 | first row of the list of others
    __shared__ uint2 s_cell[kSmallRows];                    // a row's cell, the next row of its list
    __shared__ int32_t s_pairs[64];
    __shared__ int32_t s_found[kGemm ? kSmallQuarters * kSmallQuarter * 64 : 1];  // [offset][row]
    static_assert(kSmallQuarters * 64 * 32 <= kSmallHeads, "the quarters' sums take the heads' place");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int4* coors = reinterpret_cast<const int4*>(P.coors);  // (b,z,y,x)
    const int heads_lg = P.max_voxels <= kSmallHeads / 8 ? 32 - __clz(P.max_voxels * 4) : 14;  // (four and more a row, up to the room there is)
    const int shift = 32 - (heads_lg < 6 ? 6 : heads_lg);
    // (all of it requested before the row count is known)
    int4 c[kSmallOwn];
#pragma unroll
    for (int j = 0; j < kSmallOwn; ++j) {
        const int v = j * kSmallBlock + tid;
        c[j] = make_int4(0, 0, 0, 0);
        if (v < P.max_voxels) c[j] = coors[v];
    }
    const int row = blockIdx.x * 64 + lane;  // whose neighbours this lane looks up, at offsets wave, wave + kSmallWaves, ...
    const int4 own = coors[row < P.max_voxels ? row : 0];
    const int quarter = wave >> 2, rows16 = (wave & 3) * 16 + (lane & 15);  // of the products: the wave's offsets, the lane's row
    const int vec = (tid % kVecs) * 4;                                      // of the epilogue: the thread's columns
    float w[kSmallQuarter][NB][E];
    float4 epi_scale = make_float4(1.f, 1.f, 1.f, 1.f), epi_shift = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (kGemm) {
#pragma unroll
        for (int j = 0; j < kSmallQuarter; ++j) {
            const int k = quarter * kSmallQuarter + j;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) small_operand(G.w + (((k < P.K ? k : 0) * NB + nb) * 64 + lane) * E, w[j][nb]);
        }
        if (G.scale) epi_scale = *reinterpret_cast<const float4*>(G.scale + vec);
        if (G.shift) epi_shift = *reinterpret_cast<const float4*>(G.shift + vec);
    }
    for (int t = tid; t < (1 << (32 - shift)) / 4; t += kSmallBlock) reinterpret_cast<uint4*>(s_head)[t] = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (tid < 64) s_pairs[tid] = 0;
    const int n = clamp_rows(P.num, P.max_voxels);
    // (a layer without rows ends here as well: a captured call 16 -> 16 7.6 -> 3.1 us, 4 -> 16 6.0 -> 2.8; two launches 5.9)
    if ((int)blockIdx.x * 64 >= n && (kGemm || blockIdx.x)) {
        if (blockIdx.x == 0 && tid < 4) P.meta[tid] = tiles[tid] = 0;
        const int r = blockIdx.x * 64 + tid / kVecs;
        if (kGemm && G.write_pad && tid < 64 * kVecs && r < P.max_voxels)
            *reinterpret_cast<float4*>(G.out + (size_t)r * COUT + vec) = small_epilogue(G, make_float4(0.f, 0.f, 0.f, 0.f), epi_scale, epi_shift);
        return;
    }
    __syncthreads();
    auto cell = [&](int z, int y, int x) { return ((uint32_t)z * (uint32_t)P.t.gy + (uint32_t)y) * (uint32_t)P.t.gx + (uint32_t)x; };
    auto list = [&](uint32_t key) { return (key * 2654435769u) >> shift; };
    bool bad = false;
    uint32_t mine[kSmallOwn], hash[kSmallOwn];  // (of rows that are in the layer)
#pragma unroll
    for (int j = 0; j < kSmallOwn; ++j) {
        const int v = j * kSmallBlock + tid;
        hash[j] = ~0u;
        if (v < n) {
            if (c[j].y < 0 || c[j].y >= P.t.gz || c[j].z < 0 || c[j].z >= P.t.gy || c[j].w < 0 || c[j].w >= P.t.gx) {
                bad = true;  // the reference would write outside its grid
            } else {
                mine[j] = cell(c[j].y, c[j].z, c[j].w);
                hash[j] = list(mine[j]);
                s_cell[v].x = mine[j];
                atomicMin(&s_head[hash[j]], (uint32_t)v << 16 | kNoRow);
            }
        }
    }
    const bool any_bad = __syncthreads_or(bad);
#pragma unroll
    for (int j = 0; j < kSmallOwn; ++j) {
        const int v = j * kSmallBlock + tid;
        if (hash[j] == ~0u) continue;
        const uint32_t first = s_head[hash[j]] >> 16;
        if (s_cell[first].x != mine[j]) s_cell[v].y = atomicExch(&s_head[hash[j]], first << 16 | (uint32_t)v) & 0xffffu;
    }
    __syncthreads();
    if (blockIdx.x == 0 && tid < 4) {
        P.meta[tid] = tid == 0 ? (any_bad ? SESSD_STATUS_BAD_COORD : 0) : (tid == 1 ? n : 0);
        tiles[tid] = 0;
    }
    const bool in_layer = row < n && own.y >= 0 && own.y < P.t.gz && own.z >= 0 && own.z < P.t.gy && own.w >= 0 && own.w < P.t.gx;
    uint32_t key[kSmallDepth], at[kSmallDepth], found[kSmallDepth];
    int open = 0;
#pragma unroll
    for (int j = 0; j < kSmallDepth; ++j) {
        const int k = wave + j * kSmallWaves;
        const int z = own.y - P.p[0] + k / (P.k[1] * P.k[2]), y = own.z - P.p[1] + k / P.k[2] % P.k[1], x = own.w - P.p[2] + k % P.k[2];
        const bool ok = in_layer && k < P.K && z >= 0 && z < P.t.gz && y >= 0 && y < P.t.gy && x >= 0 && x < P.t.gx;
        key[j] = cell(z, y, x);
        const uint32_t head = ok ? s_head[list(key[j])] : ~0u;
        const uint32_t first = head >> 16;
        const bool here = first != kNoRow && s_cell[first != kNoRow ? first : 0].x == key[j];
        found[j] = here ? first : kEmpty;
        at[j] = here ? kNoRow : head & 0xffffu;
        open |= at[j] != kNoRow ? 1 : 0;
    }
    while (open) {  // (lists end: a row is in one of them, in front of the rows that were in it before)
        open = 0;
#pragma unroll
        for (int j = 0; j < kSmallDepth; ++j) {
            if (at[j] == kNoRow) continue;
            const uint2 e = s_cell[at[j]];
            if (e.x == key[j]) found[j] = found[j] < at[j] ? found[j] : at[j];  // (a cell that two rows name belongs to the first)
            at[j] = e.y;
            open |= e.y != kNoRow ? 1 : 0;
        }
    }
    int pairs = 0;
#pragma unroll
    for (int j = 0; j < kSmallDepth; ++j) {
        const int k = wave + j * kSmallWaves;
        pairs += found[j] != kEmpty ? 1 : 0;
        if (k < P.K && row < n) P.nbr[(size_t)k * P.max_voxels + row] = (int32_t)found[j];
        if (kGemm && k < kSmallQuarters * kSmallQuarter) s_found[k * 64 + lane] = k < P.K ? (int32_t)found[j] : -1;
    }
    if constexpr (kGemm) {
        typedef float v4f __attribute__((ext_vector_type(4)));
        static_assert(kSmallDepth * kSmallWaves >= kSmallQuarters * kSmallQuarter, "an entry for each offset");
        const int q = lane >> 4;  // channels of an MFMA's operands, columns of its results
        __syncthreads();
        float x[kSmallQuarter][E];
        int idx[kSmallQuarter];
#pragma unroll
        for (int j = 0; j < kSmallQuarter; ++j) idx[j] = s_found[(quarter * kSmallQuarter + j) * 64 + rows16];
#pragma unroll
        for (int j = 0; j < kSmallQuarter; ++j)
            small_operand(G.in + (idx[j] >= 0 ? idx[j] : 0) * CIN + q * E, x[j]);
        v4f sum[kSmallQuarter][NB];
#pragma unroll
        for (int j = 0; j < kSmallQuarter; ++j)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < E; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][nb][e], x[j][e], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[j][nb][r] = idx[j] >= 0 ? acc[r] : 0.f;
            }
#pragma unroll
        for (int m = kSmallQuarter; m > 1; m = (m + 1) / 2)
#pragma unroll
            for (int j = 0; j < m / 2; ++j)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[j][nb][r] += sum[m - 1 - j][nb][r];
        float4* const part = reinterpret_cast<float4*>(s_head);  // [quarter][row][column / 4]
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            part[(quarter * 64 + rows16) * kVecs + nb * 4 + q] = make_float4(sum[0][nb][0], sum[0][nb][1], sum[0][nb][2], sum[0][nb][3]);
        __syncthreads();
        const int r = blockIdx.x * 64 + tid / kVecs;
        if (tid < 64 * kVecs && r < (G.write_pad ? P.max_voxels : n)) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r < n) {
                float4 p[kSmallQuarters];
#pragma unroll
                for (int g = 0; g < kSmallQuarters; ++g) p[g] = part[g * 64 * kVecs + tid];
                v = make_float4((p[0].x + p[3].x) + (p[1].x + p[2].x), (p[0].y + p[3].y) + (p[1].y + p[2].y),
                                (p[0].z + p[3].z) + (p[1].z + p[2].z), (p[0].w + p[3].w) + (p[1].w + p[2].w));
            }
            *reinterpret_cast<float4*>(G.out + (size_t)r * COUT + vec) = small_epilogue(G, v, epi_scale, epi_shift);
        }
    }
    if (!P.w) return;  // (uniform)
    atomicAdd(&s_pairs[lane], pairs);
    __syncthreads();
    if (wave == 0) {  // as lookup_pass() leaves them
        int w = row < n ? s_pairs[lane] + P.row_weight : 0;
        if (row < P.max_voxels) P.w[row] = w;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) w += __shfl_xor(w, d, 64);
        if (lane == 0 && (int)blockIdx.x * 64 < n) P.wsum[blockIdx.x] = w;
    }
}

}  // namespace

struct SubmConv3dLayerPlugin::Layout {
    void* cells;  // cell table: cell -> row
    int32_t* nbr;
    void* export_scratch;
    int32_t* tiles;  // equal-work tile cuts of the rulebook (tile_cut.hip); first word 0 = none
    int32_t* meta;  // [0] status word, [1] active rows of the last enqueue
    uint32_t cap;
    bool dense;
    size_t meta_offset;
    size_t total;
};

SubmConv3dLayerPlugin::Layout SubmConv3dLayerPlugin::carve(void* workspace) const {
    Layout L;
    WorkspaceCarver c(workspace);
    L.cap = next_pow2((uint64_t)(max_voxels_ < 32 ? 32 : max_voxels_) * 2);
    const uint64_t volume = (uint64_t)out_shape_x_ * out_shape_y_ * out_shape_z_;
    L.dense = dense_pays(volume, (uint64_t)L.cap * 8);
    if (L.dense) L.cap = (uint32_t)volume;
    L.cells = c.take<uint32_t>(L.dense ? (size_t)L.cap : (size_t)L.cap * 2);
    L.nbr = c.take<int32_t>((size_t)kernel_volume_ * max_voxels_);
    L.export_scratch = c.take<uint8_t>(export_scratch_bytes(kernel_volume_, max_voxels_));
    L.tiles = reinterpret_cast<int32_t*>(c.take<uint8_t>(tile_cut_bytes(max_voxels_)));
    L.meta_offset = c.offset;
    L.meta = c.take<int32_t>(4);
    L.total = c.total();
    return L;
}

int SubmConv3dLayerPlugin::validate() const {
    if (in_channel_ <= 0 || out_channel_ <= 0 || max_voxels_ <= 0)
        return fail(SESSD_E_INVALID, "submconv3d: channels/max_voxels must be positive");
    if (ksize_ != 1 && ksize_ != 3)
        return fail(SESSD_E_UNSUPPORTED, "submconv3d: ksize %d (the rulebook holds at most 27 offsets)", ksize_);
    if (stride_ != 1 || dilation_ != 1)
        return fail(SESSD_E_UNSUPPORTED, "submconv3d: stride and dilation must be 1");
    if (padding_ != ksize_ / 2)
        return fail(SESSD_E_UNSUPPORTED, "submconv3d: padding must be ksize/2 (output sites == input sites)");
    if (out_shape_x_ <= 0 || out_shape_y_ <= 0 || out_shape_z_ <= 0 ||
        (int64_t)out_shape_x_ * out_shape_y_ * out_shape_z_ >= (int64_t)kEmpty)
        return fail(SESSD_E_UNSUPPORTED, "submconv3d: out_shape volume must fit a 32-bit cell key");
    return SESSD_OK;
}

int SubmConv3dLayerPlugin::create(const sessd_submconv3d_desc& d, const float* weights,
                                  SubmConv3dLayerPlugin** out) {
    auto* p = new SubmConv3dLayerPlugin();
    p->in_channel_ = d.in_channel;
    p->out_channel_ = d.out_channel;
    p->max_voxels_ = d.max_voxels;
    p->feature_num_ = d.feature_num;
    p->out_shape_x_ = d.out_shape[0];
    p->out_shape_y_ = d.out_shape[1];
    p->out_shape_z_ = d.out_shape[2];
    p->spatial_shape_x_ = d.spatial_shape[0];
    p->spatial_shape_y_ = d.spatial_shape[1];
    p->spatial_shape_z_ = d.spatial_shape[2];
    p->ksize_ = d.ksize;
    p->stride_ = d.stride;
    p->padding_ = d.padding;
    p->dilation_ = d.dilation;
    p->out_padding_ = d.out_padding;
    p->kernel_volume_ = d.ksize * d.ksize * d.ksize;
    int rc = p->validate();
    if (rc == SESSD_OK)
        rc = p->uploadWeights(weights, (size_t)p->kernel_volume_ * d.in_channel * d.out_channel);
    if (rc != SESSD_OK) {
        delete p;
        return rc;
    }
    *out = p;
    return SESSD_OK;
}

// 16 ints + FP32 weights, submConv3dlayer.cu:684-714 (+ optional epilogue trailer, conv_base.hip)
size_t SubmConv3dLayerPlugin::getSerializationSize() const {
    return (size_t)weights_size_ * sizeof(float) + 16 * sizeof(int) + conv_epilogue_trailer_size(epi_);
}

void SubmConv3dLayerPlugin::serialize(void* buffer) const {
    char* d = static_cast<char*>(buffer);
    writeToBuffer<int>(d, in_channel_);
    writeToBuffer<int>(d, out_channel_);
    writeToBuffer<int>(d, max_voxels_);
    writeToBuffer<int>(d, feature_num_);
    writeToBuffer<int>(d, out_shape_x_);
    writeToBuffer<int>(d, out_shape_y_);
    writeToBuffer<int>(d, out_shape_z_);
    writeToBuffer<int>(d, spatial_shape_x_);
    writeToBuffer<int>(d, spatial_shape_y_);
    writeToBuffer<int>(d, spatial_shape_z_);
    writeToBuffer<int>(d, ksize_);
    writeToBuffer<int>(d, stride_);
    writeToBuffer<int>(d, padding_);
    writeToBuffer<int>(d, dilation_);
    writeToBuffer<int>(d, out_padding_);
    writeToBuffer<int>(d, weights_size_);
    for (int i = 0; i < weights_size_; ++i) writeToBuffer<float>(d, weights_data_[i]);
    conv_write_epilogue_trailer(d, epi_);
}

// The reference's deserialising ctor leaves the device weights unset and relies on TensorRT calling
// clone() (submConv3dlayer.cu:154-196); here the plugin is usable right away.
int SubmConv3dLayerPlugin::deserialize(const void* data, size_t length, SubmConv3dLayerPlugin** out) {
    if (!data || length < 16 * sizeof(int)) return fail(SESSD_E_INVALID, "submconv3d: blob too short");
    const char* d = static_cast<const char*>(data);
    sessd_submconv3d_desc desc;
    desc.in_channel = readFromBuffer<int>(d);
    desc.out_channel = readFromBuffer<int>(d);
    desc.max_voxels = readFromBuffer<int>(d);
    desc.feature_num = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.out_shape[a] = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.spatial_shape[a] = readFromBuffer<int>(d);
    desc.ksize = readFromBuffer<int>(d);
    desc.stride = readFromBuffer<int>(d);
    desc.padding = readFromBuffer<int>(d);
    desc.dilation = readFromBuffer<int>(d);
    desc.out_padding = readFromBuffer<int>(d);
    const int wsize = readFromBuffer<int>(d);
    const int64_t expect = (int64_t)desc.ksize * desc.ksize * desc.ksize * desc.in_channel * desc.out_channel;
    if (wsize < 0 || wsize != expect || length < 16 * sizeof(int) + (size_t)wsize * sizeof(float))
        return fail(SESSD_E_INVALID, "submconv3d: weights_size %d does not match the layer shape", wsize);
    std::vector<float> w((size_t)wsize);
    std::memcpy(w.data(), d, (size_t)wsize * sizeof(float));
    d += (size_t)wsize * sizeof(float);
    SubmConv3dLayerPlugin* p = nullptr;
    SESSD_TRY(create(desc, w.data(), &p));
    const int rc = read_epilogue_trailer(d, length - 16 * sizeof(int) - (size_t)wsize * sizeof(float), p);
    if (rc != SESSD_OK) {
        delete p;
        return rc;
    }
    *out = p;
    return SESSD_OK;
}

int SubmConv3dLayerPlugin::configurePlugin(const sessd_tensor_desc* in, int nbInputs,
                                           const sessd_tensor_desc* out, int nbOutputs) {
    return configureTypes(in, nbInputs, out, nbOutputs);
}

size_t SubmConv3dLayerPlugin::getWorkspaceSize(const sessd_tensor_desc*, int, const sessd_tensor_desc*,
                                               int) const {
    return carve(nullptr).total;
}

size_t SubmConv3dLayerPlugin::statusOffset() const { return carve(nullptr).meta_offset; }

CellTable SubmConv3dLayerPlugin::ownTable(void* workspace) const {
    const Layout L = carve(workspace);
    CellTable t;
    t.base = L.cells;
    t.cap = L.cap;
    t.dense = L.dense ? 1 : 0;
    t.per_row16 = 32;  // at most half full
    t.gx = out_shape_x_;
    t.gy = out_shape_y_;
    t.gz = out_shape_z_;
    return t;
}

LookupPart SubmConv3dLayerPlugin::lookupPart(void* workspace, const int32_t* coors, const int32_t* voxel_num, const CellTable& cells,
                                             const int32_t* cells_num, int cells_max) const {
    const Layout L = carve(workspace);
    LookupPart p;
    p.coors = coors;
    p.num = voxel_num;
    p.max_voxels = max_voxels_;
    for (int a = 0; a < 3; ++a) {
        p.k[a] = ksize_;
        p.s[a] = 1;
        p.p[a] = padding_;
    }
    p.K = kernel_volume_;
    p.own[0] = out_shape_z_;
    p.own[1] = out_shape_y_;
    p.own[2] = out_shape_x_;
    p.t = cells;
    p.t_num = cells_num;
    p.t_max = cells_max;
    p.nbr = L.nbr;
    p.meta = L.meta;
    if (wantTileCuts()) {
        p.w = tile_weight_array(L.tiles, max_voxels_);
        p.wsum = tile_weight_sums(L.tiles, max_voxels_);
        p.row_weight = tileRowWeight();
    }
    return p;
}

CutPart SubmConv3dLayerPlugin::cutPart(void* workspace, const int32_t* voxel_num) const {
    return make_cut_part(voxel_num, kernel_volume_, max_voxels_, tileRows(), tileRowWeight(), tilesWide(), carve(workspace).tiles);
}

void SubmConv3dLayerPlugin::collectHeaderFill(void* workspace, FillArgs& f) const {
    const Layout L = carve(workspace);
    f.add(L.tiles, 4, 0);
    f.add(L.meta, 4, 0);
}

// The two halves of enqueue.  The rulebook depends only on the coordinates, the GEMM only on the
// rulebook and the features: a pipeline may run the halves of different layers on different streams.
int SubmConv3dLayerPlugin::enqueueBuild(const int32_t* coors, const int32_t* voxel_num, void* workspace, hipStream_t stream) {
    if (!coors || !voxel_num || !workspace) return fail(SESSD_E_INVALID, "submconv3d.build: null pointer");
    const Layout L = carve(workspace);
    const Grid3 g{out_shape_x_, out_shape_y_, out_shape_z_};
    const CellTable t = ownTable(workspace);
    const LookupPart look = lookupPart(workspace, coors, voxel_num, t, voxel_num, max_voxels_);
    if (max_voxels_ <= kSmallRows) {
        hipLaunchKernelGGL((subm_small<0, 0>), dim3(ceil_div(max_voxels_, 64)), dim3(kSmallBlock), 0, stream, look, L.tiles, SmallGemm());
        SESSD_HIP_TRY(hipGetLastError());
    } else {
        FillArgs f;
        f.add(L.cells, t.words(), kEmpty);
        collectHeaderFill(workspace, f);
        SESSD_TRY(launch_fill(f, stream));
        hipLaunchKernelGGL(subm_insert, dim3(ceil_div(max_voxels_, kBlock)), dim3(kBlock), 0, stream, coors, voxel_num, max_voxels_, g, t,
                           L.meta);
        SESSD_HIP_TRY(hipGetLastError());
        SESSD_TRY(launch_flags_lookups(nullptr, &look, 1, stream));
    }
    if (!wantTileCuts()) return SESSD_OK;
    const CutPart cut = cutPart(workspace, voxel_num);
    return launch_number(nullptr, nullptr, &cut, 1, nullptr, nullptr, stream);
}

// Rulebook and products in one launch (subm_small): layers of few rows on plain FP32 products.  Where a caller times the products
// they are a launch of their own.
bool SubmConv3dLayerPlugin::runsInOne() const {
    const bool shape = out_channel_ == 16 ? in_channel_ == 4 || in_channel_ == 16 : out_channel_ == 32 && in_channel_ == 4;
    return max_voxels_ <= kSmallRows && shape && in_type_ == SESSD_FLOAT && out_type_ == SESSD_FLOAT && gemmOnMatrixCores() && !wantTileCuts() &&
           !ev_gemm_begin_ && !ev_gemm_end_;
}

int SubmConv3dLayerPlugin::enqueueInOne(const void* in_feat, const int32_t* coors, const int32_t* voxel_num, void* out_feat, void* workspace,
                                        hipStream_t stream) {
    const Layout L = carve(workspace);
    const LookupPart look = lookupPart(workspace, coors, voxel_num, ownTable(workspace), voxel_num, max_voxels_);
    SmallGemm g;
    g.in = static_cast<const float*>(in_feat);
    g.out = static_cast<float*>(out_feat);
    g.w = static_cast<const float*>(weights_packed_dev_);
    g.scale = epi_.scale_dev;
    g.shift = epi_.shift_dev;
    g.relu = epi_.relu;
    g.write_pad = (flags_ & SESSD_FLAG_SKIP_PAD_ROWS) ? 0 : 1;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(ceil_div(max_voxels_, 64)), dim3(kSmallBlock), 0, stream, look, L.tiles, g); };
    if (in_channel_ == 16) go(subm_small<16, 16>);
    else out_channel_ == 16 ? go(subm_small<4, 16>) : go(subm_small<4, 32>);
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

int SubmConv3dLayerPlugin::enqueueGemm(const void* in_feat, void* out_feat, const int32_t* voxel_num,
                                       const void* rulebook_workspace, hipStream_t stream,
                                       const DenseTarget* dense) {
    if (!in_feat || !out_feat || !voxel_num || !rulebook_workspace)
        return fail(SESSD_E_INVALID, "submconv3d.gemm: null pointer");
    const Layout L = carve(const_cast<void*>(rulebook_workspace));
    return runGemm(in_feat, out_feat, L.nbr, L.tiles, voxel_num, stream, dense);
}

GemmArgs SubmConv3dLayerPlugin::sharedGemmArgs(const void* in_feat, void* out_feat, const int32_t* voxel_num, void* rulebook_workspace) const {
    const Layout L = carve(rulebook_workspace);
    return gemmArgs(in_feat, out_feat, L.nbr, L.tiles, voxel_num);
}

int SubmConv3dLayerPlugin::enqueue(const sessd_tensor_desc* inputDesc, const sessd_tensor_desc* outputDesc,
                                   const void* const* inputs, void* const* outputs, void* workspace,
                                   hipStream_t stream) {
    SESSD_TRY(conv_check_io(inputDesc, outputDesc, inputs, outputs, in_type_, out_type_, max_voxels_,
                            in_channel_, out_channel_, "submconv3d.enqueue"));
    if (!workspace) return fail(SESSD_E_INVALID, "submconv3d.enqueue: workspace is null");
    const int32_t *coors = static_cast<const int32_t*>(inputs[1]), *voxel_num = static_cast<const int32_t*>(inputs[2]);
    if (runsInOne()) return enqueueInOne(inputs[0], coors, voxel_num, outputs[0], workspace, stream);
    SESSD_TRY(enqueueBuild(coors, voxel_num, workspace, stream));
    return enqueueGemm(inputs[0], outputs[0], voxel_num, workspace, stream);
}

int SubmConv3dLayerPlugin::enqueueShared(const sessd_tensor_desc* inputDesc, const sessd_tensor_desc* outputDesc,
                                         const void* const* inputs, void* const* outputs,
                                         const void* rulebook_workspace, hipStream_t stream) {
    SESSD_TRY(conv_check_io(inputDesc, outputDesc, inputs, outputs, in_type_, out_type_, max_voxels_,
                            in_channel_, out_channel_, "submconv3d.enqueue_shared"));
    if (!rulebook_workspace) return fail(SESSD_E_INVALID, "submconv3d.enqueue_shared: rulebook workspace is null");
    return enqueueGemm(inputs[0], outputs[0], static_cast<const int32_t*>(inputs[2]), rulebook_workspace, stream);
}

int SubmConv3dLayerPlugin::exportRulebook(const void* workspace, int32_t* indice_pairs, uint32_t* indice_num,
                                          hipStream_t stream) const {
    if (!workspace) return fail(SESSD_E_INVALID, "submconv3d.export_rulebook: workspace is null");
    const Layout L = carve(const_cast<void*>(workspace));
    return ConvPluginBase::exportRulebook(L.nbr, L.meta + 1, L.export_scratch, indice_pairs, indice_num, stream);
}

int SubmConv3dLayerPlugin::countPairs(const void* workspace, uint32_t* indice_num, hipStream_t stream) const {
    if (!workspace) return fail(SESSD_E_INVALID, "submconv3d.count_pairs: workspace is null");
    const Layout L = carve(const_cast<void*>(workspace));
    return launch_count_pairs(L.nbr, L.meta + 1, kernel_volume_, max_voxels_, L.export_scratch, indice_num, stream);
}

}  // namespace sessd
