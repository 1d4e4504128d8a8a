// sparse_conv3d.hip -- SparseConv3dLayerPlugin: strided sparse 3-D convolution.
//
// Replaces sparseConv3dlayer.cu:310-813.  The reference marks candidate output cells in a dense
// grid, numbers them by scanning the WHOLE grid with atomicAdd (fillGridKernel2: 46 200 blocks at
// 21x800x704) and appends rulebook pairs with atomics.  Here every (input row, candidate) pair is
// a "ticket" t = row*Kc + e, e being the position in getValidOutPos' enumeration order:
//
//   sp_insert   one thread per ticket: output cell key -> hash, value = min ticket that names it
//   sp_flags    one thread per ticket: "am I the first ticket of my cell" -> wave64 ballot words
//   sp_number   exclusive prefix over the ballot words = output row in first-seen order (the order
//               of a sequential walk, sparseConv3dlayer.cu:738-757); writes out coors + voxel_num
//   sp_scatter  one thread per ticket: nbr[offset][out row] = input row  (in the pipeline, which has the table of the
//               input rows at hand, the rulebook is looked up instead: LookupPart)
//   gather-GEMM one launch for all offsets
// (kernels: coord.hip)
//
// No pass touches anything larger than O(active sites); numbering is deterministic.
#include "coord.h"
#include "plugins.h"

namespace sessd {

// cand[] keeps a ticket's table slot in 26 bits
constexpr uint32_t kSlotBits = 26;

struct SparseConv3dLayerPlugin::Layout {
    void* cells;  // table of output cells
    int32_t* nbr;
    uint32_t* cand;
    uint64_t* words;
    uint32_t* counts;
    void* export_scratch;
    int32_t* tiles;  // equal-work tile cuts of the rulebook (tile_cut.hip); first word 0 = none
    int32_t* meta;
    uint32_t cap;
    bool dense;
    int Kc;
    int n_chunks;
    size_t meta_offset;
    size_t total;
};

// slots of the candidate hash beyond the worst-case number of distinct candidates: 1/kHashSlack of it
constexpr uint64_t kHashSlack = 16;

int SparseConv3dLayerPlugin::maxCandidates() const {
    const int k[3] = {ksize0_, ksize1_, ksize2_}, s[3] = {stride0_, stride1_, stride2_};
    int kc = 1;
    for (int a = 0; a < 3; ++a) kc *= (k[a] + s[a] - 1) / s[a];
    return kc;
}

SparseConv3dLayerPlugin::Layout SparseConv3dLayerPlugin::carve(void* workspace) const {
    Layout L;
    WorkspaceCarver c(workspace);
    L.Kc = maxCandidates();
    const uint64_t volume = (uint64_t)out_shape_x_ * out_shape_y_ * out_shape_z_;
    uint64_t distinct = (uint64_t)L.Kc * max_voxels_;  // upper bound on distinct candidate cells
    if (distinct > volume) distinct = volume;
    if (distinct < 32) distinct = 32;
    // every distinct candidate cell gets a slot (the cap on output rows applies after numbering).  The bound is
    // the worst case -- every input row with Kc candidates of its own -- of which a real frame uses a few per
    // cent, so the table is sized just above it rather than at twice it: half the bytes to clear per frame.
    L.cap = next_pow2(distinct + distinct / kHashSlack);
    L.dense = dense_pays(volume, (uint64_t)L.cap * 8) && volume < (1ull << kSlotBits);
    if (L.dense) L.cap = (uint32_t)volume;
    const int64_t tickets = (int64_t)L.Kc * max_voxels_;
    L.n_chunks = ceil_div(tickets, 256);
    L.cells = c.take<uint32_t>(L.dense ? (size_t)L.cap : (size_t)L.cap * 2);
    L.nbr = c.take<int32_t>((size_t)kernel_volume_ * max_voxels_);
    L.cand = c.take<uint32_t>((size_t)L.n_chunks * 256);
    L.words = c.take<uint64_t>((size_t)L.n_chunks * 4);
    L.counts = c.take<uint32_t>((size_t)L.n_chunks);
    L.export_scratch = c.take<uint8_t>(export_scratch_bytes(kernel_volume_, max_voxels_));
    L.tiles = reinterpret_cast<int32_t*>(c.take<uint8_t>(tile_cut_bytes(max_voxels_)));
    L.meta_offset = c.offset;
    L.meta = c.take<int32_t>(4);
    L.total = c.total();
    return L;
}

int SparseConv3dLayerPlugin::validate() const {
    if (in_channel_ <= 0 || out_channel_ <= 0 || max_voxels_ <= 0)
        return fail(SESSD_E_INVALID, "sparseconv3d: channels/max_voxels must be positive");
    const int k[3] = {ksize0_, ksize1_, ksize2_}, s[3] = {stride0_, stride1_, stride2_},
              p[3] = {padding0_, padding1_, padding2_};
    for (int a = 0; a < 3; ++a)
        if (k[a] <= 0 || s[a] <= 0 || p[a] < 0)
            return fail(SESSD_E_INVALID, "sparseconv3d: bad ksize/stride/padding on axis %d", a);
    if (kernel_volume_ > 27 || maxCandidates() > 27)
        return fail(SESSD_E_UNSUPPORTED, "sparseconv3d: more than 27 kernel offsets (the reference's limit)");
    if (dilation_ != 1) return fail(SESSD_E_UNSUPPORTED, "sparseconv3d: dilation must be 1");
    if (out_shape_x_ <= 0 || out_shape_y_ <= 0 || out_shape_z_ <= 0 ||
        (int64_t)out_shape_x_ * out_shape_y_ * out_shape_z_ >= (int64_t)kEmpty)
        return fail(SESSD_E_UNSUPPORTED, "sparseconv3d: out_shape volume must fit a 32-bit cell key");
    if ((uint64_t)next_pow2((uint64_t)maxCandidates() * max_voxels_ * 2) > (1ull << kSlotBits))
        return fail(SESSD_E_UNSUPPORTED, "sparseconv3d: max_voxels too large for the candidate table");
    if ((int64_t)maxCandidates() * max_voxels_ >= (int64_t)kEmpty)
        return fail(SESSD_E_UNSUPPORTED, "sparseconv3d: ticket space exceeds 32 bits");
    return SESSD_OK;
}

int SparseConv3dLayerPlugin::create(const sessd_sparseconv3d_desc& d, const float* weights,
                                    SparseConv3dLayerPlugin** out) {
    auto* p = new SparseConv3dLayerPlugin();
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
    p->ksize0_ = d.ksize[0]; p->ksize1_ = d.ksize[1]; p->ksize2_ = d.ksize[2];
    p->stride0_ = d.stride[0]; p->stride1_ = d.stride[1]; p->stride2_ = d.stride[2];
    p->padding0_ = d.padding[0]; p->padding1_ = d.padding[1]; p->padding2_ = d.padding[2];
    p->dilation_ = d.dilation;
    p->out_padding_ = d.out_padding;
    p->kernel_volume_ = d.ksize[0] * d.ksize[1] * d.ksize[2];
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

// 22 ints + FP32 weights, sparseConv3dlayer.cu:863-899 (+ optional epilogue trailer)
size_t SparseConv3dLayerPlugin::getSerializationSize() const {
    return (size_t)weights_size_ * sizeof(float) + 22 * sizeof(int) + conv_epilogue_trailer_size(epi_);
}

void SparseConv3dLayerPlugin::serialize(void* buffer) const {
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
    writeToBuffer<int>(d, ksize0_);
    writeToBuffer<int>(d, ksize1_);
    writeToBuffer<int>(d, ksize2_);
    writeToBuffer<int>(d, stride0_);
    writeToBuffer<int>(d, stride1_);
    writeToBuffer<int>(d, stride2_);
    writeToBuffer<int>(d, padding0_);
    writeToBuffer<int>(d, padding1_);
    writeToBuffer<int>(d, padding2_);
    writeToBuffer<int>(d, dilation_);
    writeToBuffer<int>(d, out_padding_);
    writeToBuffer<int>(d, weights_size_);
    for (int i = 0; i < weights_size_; ++i) writeToBuffer<float>(d, weights_data_[i]);
    conv_write_epilogue_trailer(d, epi_);
}

int SparseConv3dLayerPlugin::deserialize(const void* data, size_t length, SparseConv3dLayerPlugin** out) {
    if (!data || length < 22 * sizeof(int)) return fail(SESSD_E_INVALID, "sparseconv3d: blob too short");
    const char* d = static_cast<const char*>(data);
    sessd_sparseconv3d_desc desc;
    desc.in_channel = readFromBuffer<int>(d);
    desc.out_channel = readFromBuffer<int>(d);
    desc.max_voxels = readFromBuffer<int>(d);
    desc.feature_num = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.out_shape[a] = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.spatial_shape[a] = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.ksize[a] = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.stride[a] = readFromBuffer<int>(d);
    for (int a = 0; a < 3; ++a) desc.padding[a] = readFromBuffer<int>(d);
    desc.dilation = readFromBuffer<int>(d);
    desc.out_padding = readFromBuffer<int>(d);
    const int wsize = readFromBuffer<int>(d);
    const int64_t expect = (int64_t)desc.ksize[0] * desc.ksize[1] * desc.ksize[2] * desc.in_channel * desc.out_channel;
    if (wsize < 0 || wsize != expect || length < 22 * sizeof(int) + (size_t)wsize * sizeof(float))
        return fail(SESSD_E_INVALID, "sparseconv3d: weights_size %d does not match the layer shape", wsize);
    std::vector<float> w((size_t)wsize);
    std::memcpy(w.data(), d, (size_t)wsize * sizeof(float));
    d += (size_t)wsize * sizeof(float);
    SparseConv3dLayerPlugin* p = nullptr;
    SESSD_TRY(create(desc, w.data(), &p));
    const int rc = read_epilogue_trailer(d, length - 22 * sizeof(int) - (size_t)wsize * sizeof(float), p);
    if (rc != SESSD_OK) {
        delete p;
        return rc;
    }
    *out = p;
    return SESSD_OK;
}

int SparseConv3dLayerPlugin::configurePlugin(const sessd_tensor_desc* in, int nbInputs,
                                             const sessd_tensor_desc* out, int nbOutputs) {
    if (nbOutputs < 3) return fail(SESSD_E_INVALID, "sparseconv3d.configure: expected 3 outputs");
    return configureTypes(in, nbInputs, out, nbOutputs);
}

size_t SparseConv3dLayerPlugin::getWorkspaceSize(const sessd_tensor_desc*, int, const sessd_tensor_desc*,
                                                 int) const {
    return carve(nullptr).total;
}

size_t SparseConv3dLayerPlugin::statusOffset() const { return carve(nullptr).meta_offset; }

CellTable SparseConv3dLayerPlugin::cellTable(void* workspace) const {
    const Layout L = carve(workspace);
    CellTable t;
    t.base = L.cells;
    t.cap = L.cap;
    t.dense = L.dense ? 1 : 0;
    t.per_row16 = L.Kc * (16 + 16 / (int)kHashSlack);
    t.gx = out_shape_x_;
    t.gy = out_shape_y_;
    t.gz = out_shape_z_;
    return t;
}

SpPart SparseConv3dLayerPlugin::part(const int32_t* coors, const int32_t* voxel_num, int32_t* out_coors, int32_t* out_num,
                                     void* workspace, bool scattered) const {
    const Layout L = carve(workspace);
    SpPart P;
    P.k[0] = ksize0_; P.k[1] = ksize1_; P.k[2] = ksize2_;
    P.s[0] = stride0_; P.s[1] = stride1_; P.s[2] = stride2_;
    P.p[0] = padding0_; P.p[1] = padding1_; P.p[2] = padding2_;
    P.os[0] = out_shape_z_; P.os[1] = out_shape_y_; P.os[2] = out_shape_x_;
    P.Kc = L.Kc;
    P.halving = L.Kc == 8;
    for (int x = 0; x < 3; ++x) P.halving = P.halving && P.k[x] == 3 && P.s[x] == 2;
    P.max_voxels = max_voxels_;
    P.K = kernel_volume_;
    P.t = cellTable(workspace);
    P.cand = L.cand;
    P.words = L.words;
    P.counts = L.counts;
    P.n_chunks = L.n_chunks;
    P.in_coors = coors;
    P.in_num = voxel_num;
    P.out_coors = out_coors;
    P.out_num = out_num;
    P.nbr = scattered ? L.nbr : nullptr;
    P.meta = L.meta;
    return P;
}

LookupPart SparseConv3dLayerPlugin::lookupPart(void* workspace, const int32_t* out_coors, const int32_t* out_num, const CellTable& cells,
                                               const int32_t* cells_num, int cells_max) const {
    const Layout L = carve(workspace);
    LookupPart p;
    p.coors = out_coors;
    p.num = out_num;
    p.max_voxels = max_voxels_;
    p.k[0] = ksize0_; p.k[1] = ksize1_; p.k[2] = ksize2_;
    p.s[0] = stride0_; p.s[1] = stride1_; p.s[2] = stride2_;
    p.p[0] = padding0_; p.p[1] = padding1_; p.p[2] = padding2_;
    p.K = kernel_volume_;
    p.own[0] = out_shape_z_; p.own[1] = out_shape_y_; p.own[2] = out_shape_x_;
    p.t = cells;
    p.t_num = cells_num;
    p.t_max = cells_max;
    p.nbr = L.nbr;
    if (wantTileCuts()) {
        p.w = tile_weight_array(L.tiles, max_voxels_);
        p.wsum = tile_weight_sums(L.tiles, max_voxels_);
        p.row_weight = tileRowWeight();
    }
    return p;
}

CutPart SparseConv3dLayerPlugin::cutPart(void* workspace, const int32_t* out_num) const {
    return make_cut_part(out_num, kernel_volume_, max_voxels_, tileRows(), tileRowWeight(), tilesWide(), carve(workspace).tiles);
}

void SparseConv3dLayerPlugin::collectTableFill(void* workspace, FillArgs& f) const {
    f.add(carve(workspace).cells, cellTable(workspace).words(), kEmpty);
}
void SparseConv3dLayerPlugin::collectHeaderFill(void* workspace, FillArgs& f) const {
    const Layout L = carve(workspace);
    f.add(L.tiles, 4, 0);
    f.add(L.meta, 4, 0);
}
void SparseConv3dLayerPlugin::collectPadFill(int32_t* out_coors, FillArgs& f) const {
    if (!(flags_ & SESSD_FLAG_SKIP_PAD_ROWS)) f.add(out_coors, (uint64_t)max_voxels_ * 4, 0);  // :668
}

// The two halves of enqueue (see SubmConv3dLayerPlugin::enqueueBuild): output sites + rulebook from the
// coordinates, then the GEMM over the features.
int SparseConv3dLayerPlugin::enqueueBuild(const int32_t* coors, const int32_t* voxel_num, int32_t* out_coors,
                                          int32_t* out_num, void* workspace, hipStream_t stream) {
    if (!coors || !voxel_num || !out_coors || !out_num || !workspace)
        return fail(SESSD_E_INVALID, "sparseconv3d.build: null pointer");
    if (reinterpret_cast<uintptr_t>(out_coors) & 15)
        return fail(SESSD_E_INVALID, "sparseconv3d.build: output coors must be 16-byte aligned");
    const Layout L = carve(workspace);
    const SpPart P = part(coors, voxel_num, out_coors, out_num, workspace, true);
    FillArgs f;
    collectTableFill(workspace, f);
    collectHeaderFill(workspace, f);
    collectPadFill(out_coors, f);
    SESSD_TRY(launch_fill(f, stream));
    SESSD_TRY(launch_sp_insert(P, stream));
    SESSD_TRY(launch_flags_lookups(&P, nullptr, 0, stream));
    SESSD_TRY(launch_number(&P, nullptr, nullptr, 0, nullptr, nullptr, stream));
    SESSD_TRY(launch_sp_scatter(P, stream));
    if (!wantTileCuts()) return SESSD_OK;
    SESSD_TRY(launch_tile_weights(L.nbr, out_num, kernel_volume_, max_voxels_, tileRowWeight(), L.tiles, stream));
    const CutPart cut = cutPart(workspace, out_num);
    return launch_number(nullptr, nullptr, &cut, 1, nullptr, nullptr, stream);
}

int SparseConv3dLayerPlugin::enqueueGemm(const void* in_feat, void* out_feat, const int32_t* out_num,
                                         const void* workspace, hipStream_t stream, const DenseTarget* dense) {
    if (!in_feat || !out_feat || !out_num || !workspace) return fail(SESSD_E_INVALID, "sparseconv3d.gemm: null pointer");
    const Layout L = carve(const_cast<void*>(workspace));
    return runGemm(in_feat, out_feat, L.nbr, L.tiles, out_num, stream, dense);
}

int SparseConv3dLayerPlugin::enqueue(const sessd_tensor_desc* inputDesc, const sessd_tensor_desc* outputDesc,
                                     const void* const* inputs, void* const* outputs, void* workspace,
                                     hipStream_t stream) {
    SESSD_TRY(conv_check_io(inputDesc, outputDesc, inputs, outputs, in_type_, out_type_, max_voxels_,
                            in_channel_, out_channel_, "sparseconv3d.enqueue"));
    if (!workspace || !outputs[1] || !outputs[2]) return fail(SESSD_E_INVALID, "sparseconv3d.enqueue: null pointer");
    int32_t* out_num = static_cast<int32_t*>(outputs[2]);
    SESSD_TRY(enqueueBuild(static_cast<const int32_t*>(inputs[1]), static_cast<const int32_t*>(inputs[2]),
                           static_cast<int32_t*>(outputs[1]), out_num, workspace, stream));
    return enqueueGemm(inputs[0], outputs[0], out_num, workspace, stream);
}

int SparseConv3dLayerPlugin::exportRulebook(const void* workspace, int32_t* indice_pairs, uint32_t* indice_num,
                                            hipStream_t stream) const {
    if (!workspace) return fail(SESSD_E_INVALID, "sparseconv3d.export_rulebook: workspace is null");
    const Layout L = carve(const_cast<void*>(workspace));
    return ConvPluginBase::exportRulebook(L.nbr, L.meta + 1, L.export_scratch, indice_pairs, indice_num, stream);
}

int SparseConv3dLayerPlugin::countPairs(const void* workspace, uint32_t* indice_num, hipStream_t stream) const {
    if (!workspace) return fail(SESSD_E_INVALID, "sparseconv3d.count_pairs: workspace is null");
    const Layout L = carve(const_cast<void*>(workspace));
    return launch_count_pairs(L.nbr, L.meta + 1, kernel_volume_, max_voxels_, L.export_scratch, indice_num, stream);
}

}  // namespace sessd
