// voxel_generator.hip -- VoxelGeneratorPlugin: points -> voxels with mean VFE.
//
// Replaces voxelGenerator.cu:255-542 of the reference.  The reference keeps a dense
// [Z*Y*X][2] slot table (721 MB, memset every frame) and hands out voxel ids and point slots with
// atomicAdd, so which points are kept and how voxels are numbered depends on scheduling.  Here:
//
//   vg_insert    one thread per point: cell key -> open-addressing hash (a few MB, L2 resident), or a table with a word
//                per cell where the pipeline keeps one; each cell keeps its smallest point index
//   vg_flags     one thread per point: "am I the first point of my cell" -> wave64 ballot words + per-block counts;
//                the later points of a cell go through a chain of atomicMin "comparators" behind its first one, whose
//                final state is independent of the order in which threads arrive
//   vg_finalize  exclusive prefix over the ballot words = voxel id in first-appearance order;
//                that thread writes the coordinate and the mean of the (<= S) kept points
// (kernels: coord.hip)
//
// The result equals a sequential walk over the points: ids in first-appearance order, the first S
// points of a cell kept, cells first seen after max_voxels dropped.  All traffic is O(points):
// 16 B/point read + 32 B/voxel written, plus the hash clear.
#include <mutex>

#include "coord.h"
#include "plugins.h"

namespace sessd {

namespace {

constexpr int kBlock = 256;

// np.round as in spconv's voxel generator (voxelGenerator.cu:61-68): half to even
int np_round(float x) {
    int x2 = int(x * 2.0f);
    if (x != int(x) && x2 == x * 2.0f) return int(x / 2.0f + 0.5f) * 2;
    return int(x + 0.5f);
}

}  // namespace

struct VoxelGeneratorPlugin::Layout {
    uint64_t* entries;  // cell table; its value is the voxel row after vg_finalize (kEmpty for dropped cells)
    uint32_t* slots;
    int32_t* pt_slot;
    uint64_t* words;
    uint32_t* counts;
    uint32_t* sums;
    int32_t* status;
    uint32_t cap;
    uint64_t slot_words;
    int n_blocks;
    size_t total;
};

VoxelGeneratorPlugin::Layout VoxelGeneratorPlugin::carve(void* workspace, int max_points, int slots_per_point) const {
    Layout L;
    WorkspaceCarver c(workspace);
    L.status = c.take<int32_t>(4);
    L.cap = next_pow2((uint64_t)(max_points < 32 ? 32 : max_points) * slots_per_point);
    L.n_blocks = ceil_div(max_points, kBlock);
    // entries and slots are adjacent so that one fill region clears both
    L.slot_words = (uint64_t)max_points * (pointNum_ - 1);
    L.entries = reinterpret_cast<uint64_t*>(c.take<uint32_t>((uint64_t)L.cap * 2 + L.slot_words));
    L.slots = L.entries ? reinterpret_cast<uint32_t*>(L.entries + L.cap) : nullptr;
    L.pt_slot = c.take<int32_t>((size_t)L.n_blocks * kBlock);
    L.words = c.take<uint64_t>((size_t)L.n_blocks * 4);
    L.counts = c.take<uint32_t>((size_t)L.n_blocks);
    L.sums = max_points > kSumsFromPoints ? c.take<uint32_t>((size_t)ceil_div(L.n_blocks, kCountsPerSum)) : nullptr;
    L.total = c.total();
    return L;
}

CellTable VoxelGeneratorPlugin::cellTable(void* workspace, int max_points, int slots_per_point) const {
    const Layout L = carve(workspace, max_points, slots_per_point);
    CellTable t;
    t.base = L.entries;
    t.cap = L.cap;
    t.per_row16 = 16 * slots_per_point;
    t.gx = grid_x_size_;
    t.gy = grid_y_size_;
    t.gz = grid_z_size_;
    return t;
}

VgPart VoxelGeneratorPlugin::part(const float* points, const int32_t* points_size, int max_points, int pf, float* voxels,
                                  int32_t* coors, int32_t* voxel_num, void* workspace, int slots_per_point) const {
    const Layout L = carve(workspace, max_points, slots_per_point);
    VgPart v;
    v.points = points;
    v.points_size = points_size;
    v.max_points = max_points;
    v.pf = pf;
    v.min_x = min_x_range_;
    v.max_x = max_x_range_;
    v.min_y = min_y_range_;
    v.max_y = max_y_range_;
    v.min_z = min_z_range_;
    v.max_z = max_z_range_;
    v.vx = voxel_x_size_;
    v.vy = voxel_y_size_;
    v.vz = voxel_z_size_;
    v.gx = grid_x_size_;
    v.gy = grid_y_size_;
    v.gz = grid_z_size_;
    v.max_voxels = voxelNum_;
    v.max_pts = pointNum_;
    v.t = cellTable(workspace, max_points, slots_per_point);
    v.slots = L.slots;
    v.pt_slot = L.pt_slot;
    v.words = L.words;
    v.counts = L.counts;
    v.sums = L.sums;
    v.n_blocks = L.n_blocks;
    v.voxels = voxels;
    v.coors = coors;
    v.voxel_num = voxel_num;
    v.status = L.status;
    return v;
}

void VoxelGeneratorPlugin::collectTableFill(void* workspace, int max_points, bool table_only, FillArgs& f, int slots_per_point) const {
    const Layout L = carve(workspace, max_points, slots_per_point);
    f.add(L.entries, (uint64_t)L.cap * 2 + (table_only ? 0 : L.slot_words), kEmpty);
}
void VoxelGeneratorPlugin::collectPadFill(float* voxels, int32_t* coors, FillArgs& f) const {
    if (flags_ & SESSD_FLAG_SKIP_PAD_ROWS) return;
    f.add(voxels, (uint64_t)voxelNum_ * 4, 0);  // voxelGenerator.cu:524-525
    f.add(coors, (uint64_t)voxelNum_ * 4, 0);
}

void VoxelGeneratorPlugin::deriveGrid() {
    // voxelGenerator.cu:232-234
    grid_x_size_ = np_round((max_x_range_ - min_x_range_) / voxel_x_size_);
    grid_y_size_ = np_round((max_y_range_ - min_y_range_) / voxel_y_size_);
    grid_z_size_ = np_round((max_z_range_ - min_z_range_) / voxel_z_size_);
}

int VoxelGeneratorPlugin::create(const sessd_voxelgen_desc& d, VoxelGeneratorPlugin** out) {
    if (d.max_voxels <= 0 || d.max_num_points_per_voxel <= 0 || d.max_num_points_per_voxel > 64)
        return fail(SESSD_E_INVALID, "voxelgen: max_voxels=%d max_num_points_per_voxel=%d", d.max_voxels,
                    d.max_num_points_per_voxel);
    if (d.voxel_feature_num != 4)
        return fail(SESSD_E_UNSUPPORTED, "voxelgen: voxel_feature_num must be 4 (x,y,z,i), got %d",
                    d.voxel_feature_num);
    for (int a = 0; a < 3; ++a)
        if (!(d.voxel_size[a] > 0.f) || !(d.point_cloud_range[a + 3] > d.point_cloud_range[a]))
            return fail(SESSD_E_INVALID, "voxelgen: empty range or non-positive voxel size on axis %d", a);
    auto* p = new VoxelGeneratorPlugin();
    // argument order of the reference creator call (voxelGenerator.cu:697-699)
    p->voxelNum_ = d.max_voxels;
    p->pointNum_ = d.max_num_points_per_voxel;
    p->featureNum_ = d.voxel_feature_num;
    p->min_x_range_ = d.point_cloud_range[0];
    p->max_x_range_ = d.point_cloud_range[3];
    p->min_y_range_ = d.point_cloud_range[1];
    p->max_y_range_ = d.point_cloud_range[4];
    p->min_z_range_ = d.point_cloud_range[2];
    p->max_z_range_ = d.point_cloud_range[5];
    p->voxel_x_size_ = d.voxel_size[0];
    p->voxel_y_size_ = d.voxel_size[1];
    p->voxel_z_size_ = d.voxel_size[2];
    p->deriveGrid();
    if ((int64_t)p->grid_x_size_ * p->grid_y_size_ * p->grid_z_size_ >= (int64_t)kEmpty) {
        delete p;
        return fail(SESSD_E_UNSUPPORTED, "voxelgen: grid volume does not fit a 32-bit cell key");
    }
    *out = p;
    return SESSD_OK;
}

size_t VoxelGeneratorPlugin::getSerializationSize() const { return 9 * sizeof(float) + 7 * sizeof(int); }

void VoxelGeneratorPlugin::serialize(void* buffer) const {
    char* d = static_cast<char*>(buffer);
    writeToBuffer<int>(d, voxelNum_);
    writeToBuffer<int>(d, pointNum_);
    writeToBuffer<int>(d, featureNum_);
    writeToBuffer<float>(d, min_x_range_);
    writeToBuffer<float>(d, max_x_range_);
    writeToBuffer<float>(d, min_y_range_);
    writeToBuffer<float>(d, max_y_range_);
    writeToBuffer<float>(d, min_z_range_);
    writeToBuffer<float>(d, max_z_range_);
    writeToBuffer<float>(d, voxel_x_size_);
    writeToBuffer<float>(d, voxel_y_size_);
    writeToBuffer<float>(d, voxel_z_size_);
    writeToBuffer<int>(d, pointFeatureNum_);
    writeToBuffer<int>(d, grid_x_size_);
    writeToBuffer<int>(d, grid_y_size_);
    writeToBuffer<int>(d, grid_z_size_);
}

int VoxelGeneratorPlugin::deserialize(const void* data, size_t length, VoxelGeneratorPlugin** out) {
    if (!data || length < 9 * sizeof(float) + 7 * sizeof(int))
        return fail(SESSD_E_INVALID, "voxelgen: serialized blob too short (%zu bytes)", length);
    const char* d = static_cast<const char*>(data);
    auto* p = new VoxelGeneratorPlugin();
    p->voxelNum_ = readFromBuffer<int>(d);
    p->pointNum_ = readFromBuffer<int>(d);
    p->featureNum_ = readFromBuffer<int>(d);
    p->min_x_range_ = readFromBuffer<float>(d);
    p->max_x_range_ = readFromBuffer<float>(d);
    p->min_y_range_ = readFromBuffer<float>(d);
    p->max_y_range_ = readFromBuffer<float>(d);
    p->min_z_range_ = readFromBuffer<float>(d);
    p->max_z_range_ = readFromBuffer<float>(d);
    p->voxel_x_size_ = readFromBuffer<float>(d);
    p->voxel_y_size_ = readFromBuffer<float>(d);
    p->voxel_z_size_ = readFromBuffer<float>(d);
    p->pointFeatureNum_ = readFromBuffer<int>(d);
    p->grid_x_size_ = readFromBuffer<int>(d);
    p->grid_y_size_ = readFromBuffer<int>(d);
    p->grid_z_size_ = readFromBuffer<int>(d);
    if (p->voxelNum_ <= 0 || p->pointNum_ <= 0 || p->pointNum_ > 64 || p->featureNum_ != 4) {
        delete p;
        return fail(SESSD_E_INVALID, "voxelgen: serialized fields out of range");
    }
    *out = p;
    return SESSD_OK;
}

int VoxelGeneratorPlugin::configurePlugin(const sessd_tensor_desc* in, int nbInputs,
                                          const sessd_tensor_desc*, int) {
    if (!in || nbInputs < 1 || in[0].nbDims != 3)
        return fail(SESSD_E_INVALID, "voxelgen.configure: expected points desc [1,max_points,F]");
    if (in[0].d[2] < 4) return fail(SESSD_E_INVALID, "voxelgen.configure: need >= 4 point features");
    pointFeatureNum_ = in[0].d[2];  // voxelGenerator.cu:231
    lastMaxPoints_ = in[0].d[1];
    deriveGrid();
    return SESSD_OK;
}

size_t VoxelGeneratorPlugin::getWorkspaceSize(const sessd_tensor_desc* inputs, int nbInputs,
                                              const sessd_tensor_desc*, int) const {
    if (!inputs || nbInputs < 1 || inputs[0].nbDims != 3 || inputs[0].d[1] <= 0) return 0;
    return carve(nullptr, inputs[0].d[1], kSlotsPerPoint).total;
}

int VoxelGeneratorPlugin::enqueue(const sessd_tensor_desc* inputDesc, const sessd_tensor_desc*,
                                  const void* const* inputs, void* const* outputs, void* workspace,
                                  hipStream_t stream) {
    return enqueueOn(inputDesc, inputs, outputs, workspace, kSlotsPerPoint, stream);
}

int VoxelGeneratorPlugin::enqueueOn(const sessd_tensor_desc* inputDesc, const void* const* inputs, void* const* outputs,
                                    void* workspace, int slots_per_point, hipStream_t stream) {
    if (!inputDesc || !inputs || !outputs || !workspace)
        return fail(SESSD_E_INVALID, "voxelgen.enqueue: null argument");
    if (inputDesc[0].nbDims != 3 || inputDesc[0].d[0] != 1)
        return fail(SESSD_E_UNSUPPORTED, "voxelgen.enqueue: points must be [1,max_points,F]");
    if (inputDesc[0].type != SESSD_FLOAT) return fail(SESSD_E_UNSUPPORTED, "voxelgen.enqueue: points must be FP32");
    const int max_points = inputDesc[0].d[1];
    const int pf = inputDesc[0].d[2];
    if (max_points <= 0 || pf < 4) return fail(SESSD_E_INVALID, "voxelgen.enqueue: bad points shape");
    if (grid_x_size_ <= 0) return fail(SESSD_E_INVALID, "voxelgen.enqueue: configure() was not called");
    const float* points = static_cast<const float*>(inputs[0]);
    const int32_t* points_size = static_cast<const int32_t*>(inputs[1]);
    float* voxels = static_cast<float*>(outputs[0]);
    int32_t* coors = static_cast<int32_t*>(outputs[1]);
    int32_t* voxel_num = static_cast<int32_t*>(outputs[2]);
    if (!points || !points_size || !voxels || !coors || !voxel_num)
        return fail(SESSD_E_INVALID, "voxelgen.enqueue: null tensor pointer");
    if ((reinterpret_cast<uintptr_t>(voxels) | reinterpret_cast<uintptr_t>(coors)) & 15)
        return fail(SESSD_E_INVALID, "voxelgen.enqueue: outputs must be 16-byte aligned");

    lastMaxPoints_ = max_points;
    const VgPart v = part(points, points_size, max_points, pf, voxels, coors, voxel_num, workspace, slots_per_point);
    FillArgs f;
    collectTableFill(workspace, max_points, false, f, slots_per_point);
    f.add(v.status, 4, 0);
    SESSD_TRY(launch_fill(f, stream));
    FillArgs pads;
    collectPadFill(voxels, coors, pads);
    SESSD_TRY(launch_vg_insert(v, nullptr, 0, pads, stream));
    SESSD_TRY(launch_vg_flags(v, FillArgs(), stream));
    return launch_vg_finalize(v, nullptr, stream);
}

int read_status_word(const void* workspace, size_t offset, hipStream_t stream, int32_t* status) {
    if (!workspace || !status) return fail(SESSD_E_INVALID, "status: null argument");
    SESSD_HIP_TRY(hipMemcpyAsync(status, static_cast<const uint8_t*>(workspace) + offset, sizeof(int32_t),
                                 hipMemcpyDeviceToHost, stream));
    SESSD_HIP_TRY(hipStreamSynchronize(stream));
    return SESSD_OK;
}

// ---------------------------------------------------------------------------------------------
// The enqueue that allocates nothing and takes no workspace: its scratch memory is a file-scope device
// array.  Every GPU the library runs on holds its own copy of the array (8 MiB, until the process ends)
// at its own address; `scratch` below is only the host-side name of the symbol, never a device pointer,
// so host code asks the runtime for the address once per device and hands THAT to the kernels.
// ---------------------------------------------------------------------------------------------
constexpr size_t kStaticScratchBytes = 8u << 20;  // fits the reference's 80000-point tensor (5.8 MB)
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {nullptr};  // device address of `scratch`, per device
}  // namespace

// -> address of the current device's copy of `scratch` (resolved on the first call per device)
int voxelgen_static_scratch(void** out) {
    int dev = -1;
    SESSD_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(SESSD_E_UNSUPPORTED, "voxelgen: device index %d is beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        SESSD_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(SESSD_E_HIP, "voxelgen: the static scratch array has no address on device %d", dev);
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return SESSD_OK;
}

int VoxelGeneratorPlugin::enqueueStatic(const sessd_tensor_desc* inputDesc, const sessd_tensor_desc*,
                                        const void* const* inputs, void* const* outputs, hipStream_t stream) {
    if (!inputDesc || inputDesc[0].nbDims != 3 || inputDesc[0].d[1] <= 0)
        return fail(SESSD_E_INVALID, "voxelgen.enqueue_static: points must be [1,max_points,F]");
    // the size check comes before any runtime call: a request that does not fit touches nothing
    // With one point per voxel the hash is all that grows with the points: half as many slots double the rows that fit.
    // (With more, the places of the later points grow too, and 131 072 rows remain the limit.)
    int slots = kSlotsPerPoint;
    if (pointNum_ == 1 && carve(nullptr, inputDesc[0].d[1], slots).total > kStaticScratchBytes) slots = kSlotsPerPointDense;
    const size_t need = carve(nullptr, inputDesc[0].d[1], slots).total;
    if (need > kStaticScratchBytes)
        return fail(SESSD_E_INVALID,
                    "voxelgen.enqueue_static: a points tensor of %d rows with %d points per voxel needs %zu bytes of "
                    "scratch, the static buffer holds %zu; use sessd_voxelgen_enqueue with a workspace of your own",
                    inputDesc[0].d[1], pointNum_, need, kStaticScratchBytes);
    void* ws = nullptr;
    SESSD_TRY(voxelgen_static_scratch(&ws));
    return enqueueOn(inputDesc, inputs, outputs, ws, slots, stream);
}

}  // namespace sessd
