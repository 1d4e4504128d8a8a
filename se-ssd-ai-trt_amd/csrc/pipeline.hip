// pipeline.hip -- frame pipeline: VoxelGenerator -> conv stack -> Sparse2Dense on one stream.
//
// Counterpart of the graph the reference wires in createEngine (se-ssd-ai-trt.cpp:1138-1252) and of
// what TensorRT's executor does at run time: it owns every intermediate tensor and workspace and
// calls each plugin's enqueue in order.  BatchNorm1d + ReLU (se-ssd-ai-trt.cpp:808-856) is folded
// into each conv's epilogue.  Everything is allocated in create(); enqueue only launches kernels,
// optionally by replaying a hipGraph captured from the same enqueue sequence.
#include <memory>

#include "plugins.h"

namespace sessd {

namespace {

sessd_tensor_desc make_desc(std::initializer_list<int> dims, int type) {
    sessd_tensor_desc t;
    std::memset(&t, 0, sizeof(t));
    t.nbDims = (int)dims.size();
    int i = 0;
    for (int v : dims) t.d[i++] = v;
    t.type = type;
    t.scale = 1.0f;
    return t;
}

struct DeviceBuffer {
    void* p = nullptr;
    size_t bytes = 0;
    int alloc(size_t n) {
        SESSD_HIP_TRY(hipMalloc(&p, n ? n : 16));
        bytes = n;
        return SESSD_OK;
    }
    ~DeviceBuffer() {
        if (p) (void)hipFree(p);
    }
};

// A cell table that stays from frame to frame: a word per cell of the grid and, behind it, the list of the cells that
// the rows of the last frame have taken.  Nothing of it is handed out.
struct KeptTable {
    DeviceBuffer mem;
    uint32_t cells = 0;  // 0: none
    int alloc(uint64_t volume, int rows) {
        SESSD_TRY(mem.alloc(listAt(volume) + ((size_t)kCellListHead + rows) * sizeof(uint32_t)));
        cells = (uint32_t)volume;
        return SESSD_OK;
    }
    static size_t listAt(uint64_t volume) { return align_up(volume * sizeof(uint32_t)); }
    CellList taken() const {
        return cells ? reinterpret_cast<CellList>(static_cast<uint8_t*>(mem.p) + listAt(cells)) : nullptr;
    }
    void replace(CellTable& t) const {  // t: the table of the workspace, for the same grid
        if (!cells) return;
        t.base = mem.p;
        t.cap = cells;
        t.dense = 1;
    }
    CleanPart clean(const CellTable& t, int max_rows) const {
        CleanPart c;
        c.taken = taken();
        c.max_voxels = max_rows;
        c.t = t;
        return c;
    }
    void collectFill(FillArgs& f) const {
        if (!cells) return;
        f.add(mem.p, cells, kEmpty);
        f.add(taken(), 1, 0);
    }
};

}  // namespace

struct ConvStage {
    sessd_layer_spec spec;
    std::unique_ptr<SubmConv3dLayerPlugin> subm;
    std::unique_ptr<SparseConv3dLayerPlugin> sparse;
    DeviceBuffer ws, feat, coors, num;  // coors/num only for sparse layers (they produce new ones)
    // Sparse layers: output cell -> row (47 MB for 21 x 800 x 704); none where the grid or the device's memory does not
    // allow it (the workspace's table then)
    KeptTable cells;
    int rulebook_from = -1;             // SubM layer whose workspace holds this layer's rulebook
    sessd_tensor_desc in_desc[3], out_desc[3];
    void* coors_ptr = nullptr;  // coordinates valid AFTER this layer
    void* num_ptr = nullptr;
};

// a captured enqueue sequence, replayed while the pointers it was captured with stay the same
struct CapturedGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    const void* points = nullptr;
    const void* size = nullptr;
    void* dense = nullptr;
    int nodes = -1;
    void reset() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }
    ~CapturedGraph() { reset(); }
};

struct Pipeline {
    sessd_pipeline_desc desc;
    std::unique_ptr<VoxelGeneratorPlugin> vg;
    std::unique_ptr<Sparse2DensePlugin> s2d;
    std::vector<std::unique_ptr<ConvStage>> stages;
    DeviceBuffer vg_ws, vg_voxels, vg_coors, vg_num, s2d_ws;
    KeptTable vg_cells;  // the voxelizer's cell table (360 MB for 40 x 1600 x 1408), as ConvStage::cells
    sessd_tensor_desc vg_in[2], vg_out[3], s2d_in[3], s2d_out[1];
    int max_voxels = 0;
    size_t device_bytes = 0;
    CapturedGraph captured;  // graph replay

    // Frames in flight (desc.frames_in_flight = R >= 2): R complete replicas of this pipeline (tensors, workspaces,
    // graph), used in turn, each on a stream of its own: frame t + 1 starts on the next replica while frame t is
    // still running on its own, so that the head of one frame and the launch gaps between its kernels fill with the
    // other frames' work.  `ev_in` / `ev_frame_done` tie a replica's frame to the caller's streams.
    std::vector<std::unique_ptr<Pipeline>> replicas;
    hipStream_t frame_stream = nullptr;  // (replica) the stream its frames run on
    hipEvent_t ev_in = nullptr, ev_frame_done = nullptr;
    int64_t next_ticket = 0;
    int last_replica = 0;                       // replica of the last submitted frame (layer_io, status, stats)

    // two-stream schedule: the voxelizer, the lookups on its voxels and the feature chain on the caller's stream, the
    // coordinate passes behind them on `aux`; ev_pass[i] = "coordinate pass i is done" (CoordPass)
    hipStream_t aux = nullptr;
    hipEvent_t ev_head = nullptr;
    std::vector<hipEvent_t> ev_pass;
    // The voxelizer's cell table is empty at the start of a frame: a pass behind its last reader empties it for the next
    // one (a clear at the head of a frame was 4-6 us of every frame).  The strided layers' dense tables hold the rows
    // of the frame before, which their lists name.  create() clears all of them, and so does a frame that has run
    // plugin by plugin (behind its end) and a call that has failed (recover()): a frame that a caller has captured holds
    // no clear of its own.  False: that clear failed as well, the next frame begins with it.
    bool tables_ready = false;

    // profiling: one event per segment boundary (see sessd_pipeline_enqueue_timed)
    std::vector<hipEvent_t> events;
    DeviceBuffer stats;  // u32[32] scratch for per-offset pair counts

    ~Pipeline() {
        replicas.clear();
        for (hipEvent_t e : {ev_in, ev_frame_done})
            if (e) (void)hipEventDestroy(e);
        if (frame_stream) (void)hipStreamDestroy(frame_stream);
        for (hipEvent_t e : events) (void)hipEventDestroy(e);
        for (hipEvent_t e : ev_pass)
            if (e) (void)hipEventDestroy(e);
        if (ev_head) (void)hipEventDestroy(ev_head);
        if (aux) (void)hipStreamDestroy(aux);
    }

    // Whether the last layer's gather-GEMM scatters into the dense tensor itself (matrix-core kernel, same element
    // type).  The tensor is then cleared beside the voxelizer's first pass and nothing follows the last GEMM; the
    // plugin's own cell-major pass writes fewer bytes but puts two more launches at the end of the critical path
    // (measured: frames 20-40 us longer).
    bool denseByEpilogue() const {
        if (stages.empty()) return false;
        const ConvStage& st = *stages.back();
        const ConvPluginBase* cp = st.subm ? static_cast<const ConvPluginBase*>(st.subm.get()) : st.sparse.get();
        return cp->out_type_ == s2d->out_type_ && cp->out_channel_ == s2d->feature_map_channel_ && cp->gemmOnMatrixCores();
    }

    CellTable cellTable(const ConvStage& st) const {
        CellTable t = st.sparse->cellTable(st.ws.p);
        st.cells.replace(t);
        return t;
    }
    CellTable voxelTable() const {
        CellTable t = vg->cellTable(vg_ws.p, desc.max_points);
        vg_cells.replace(t);
        return t;
    }
    int clearTables(hipStream_t stream) {
        FillArgs f;
        vg->collectTableFill(vg_ws.p, desc.max_points, false, f);
        vg_cells.collectFill(f);
        for (auto& st : stages) {
            if (f.n + 2 > FillArgs::kMaxRegions) {
                SESSD_TRY(launch_fill(f, stream));
                f = FillArgs();
            }
            st->cells.collectFill(f);
        }
        return launch_fill(f, stream);
    }

    // everything that a frame has to find as the one before leaves it, as for the first frame
    int resetState(hipStream_t stream) {
        FillArgs f;
        f.add(static_cast<uint8_t*>(vg_ws.p) + vg->statusOffset(), 4, 0);
        for (auto& st : stages) {
            if (!st->ws.p) continue;
            if (f.n + 2 > FillArgs::kMaxRegions) {
                SESSD_TRY(launch_fill(f, stream));
                f = FillArgs();
            }
            if (st->subm) st->subm->collectHeaderFill(st->ws.p, f);
            else st->sparse->collectHeaderFill(st->ws.p, f);
        }
        SESSD_TRY(launch_fill(f, stream));
        SESSD_TRY(clearTables(stream));
        tables_ready = true;
        return SESSD_OK;
    }
    static hipStreamCaptureStatus captureStatus(hipStream_t s) {
        hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &c) == hipSuccess) return c;
        (void)hipGetLastError();
        return hipStreamCaptureStatusNone;
    }
    int joinAux(hipStream_t stream) {
        if (!aux) return SESSD_OK;
        SESSD_HIP_TRY(hipEventRecord(ev_head, aux));
        SESSD_HIP_TRY(hipStreamWaitEvent(stream, ev_head, 0));
        return SESSD_OK;
    }
    // Behind a call that failed with `rc`, which is returned.  Its launches may have left cells in the tables, and a graph
    // that the caller captured from an earlier frame does not clear them: the clear goes to `stream` right here, behind
    // what the call has launched on either stream.  Where `stream` is being captured nothing has run; only `aux` has to
    // come back to it, so that the capture can be ended.
    int recover(hipStream_t stream, int rc) {
        char why[1024];
        snprintf(why, sizeof(why), "%s", sessd_last_error());
        (void)hipGetLastError();  // (reported already; the launches below ask for theirs)
        if (captureStatus(stream) != hipStreamCaptureStatusNone) {
            if (aux && captureStatus(aux) == hipStreamCaptureStatusActive) (void)joinAux(stream);
        } else {
            tables_ready = false;
            if (joinAux(stream) == SESSD_OK) (void)resetState(stream);
        }
        (void)hipGetLastError();
        return fail(rc, "%s", why);
    }

    // The rows of stage 0 are the voxels, those of stage i the output rows of the i-th strided layer.
    struct Stage {
        int layer = -1;            // the strided layer that makes the rows (-1: the voxelizer)
        std::vector<int> lookups;  // layers whose rulebook is looked up once the rows are numbered
        std::vector<int> builds;   // SubM layers on a grid of their own: the plugin's own build
    };
    std::vector<Stage> coordStages() const {
        std::vector<Stage> v(1);
        int gx = vg->grid_x_size_, gy = vg->grid_y_size_, gz = vg->grid_z_size_;
        for (size_t l = 0; l < stages.size(); ++l) {
            const ConvStage& st = *stages[l];
            if (st.sparse) {
                v.emplace_back();
                v.back().layer = (int)l;
                v.back().lookups.push_back((int)l);
                gx = st.sparse->out_shape_x_;
                gy = st.sparse->out_shape_y_;
                gz = st.sparse->out_shape_z_;
            } else if (st.rulebook_from < 0) {
                // The pass that numbers a stage's rows leaves a cell -> row table behind.  Keys are (z*Y + y)*X + x: the
                // same number in both grids when X and Y agree; cells of the layer's grid beyond the table's z extent
                // are simply absent.
                const bool same = st.subm->out_shape_x_ == gx && st.subm->out_shape_y_ == gy && st.subm->out_shape_z_ >= gz;
                (same ? v.back().lookups : v.back().builds).push_back((int)l);
            }
        }
        return v;
    }

    // One frame.  The rulebooks depend only on coordinates, the GEMMs on rulebooks + features.  The coordinate chain
    // (coord.h) is  vg_insert | vg_flags | vg_finalize + insert 1 | then per stage i: flags i+1 + lookups on stage i |
    // number i+1 + insert i+2 + tile cuts of those rulebooks.  With `aux`, everything behind the lookups on the voxels, or behind the
    // passes that share launches with the first layers, runs there, and the GEMM chain waits for the passes its layers' rulebooks come from (one by one at first, further on for
    // some at once: wait_for), so that the passes of later layers overlap the GEMMs of earlier ones; under stream capture
    // that becomes two branches of the graph.
    int enqueueFrame(const void* points, const void* points_size, void* dense, hipStream_t stream) {
        const std::vector<Stage> cs = coordStages();
        const int m = (int)cs.size() - 1;  // strided layers
        const int V = max_voxels;
        // rows and table of every stage
        struct Rows {
            const int32_t *coors, *num;
            CellTable table;
            const int32_t* table_num;  // the row count the table was opened with
            int table_max;
        };
        std::vector<Rows> rows(cs.size());
        rows[0] = {static_cast<const int32_t*>(vg_coors.p), static_cast<const int32_t*>(vg_num.p), voxelTable(),
                   static_cast<const int32_t*>(points_size), desc.max_points};
        std::vector<SpPart> part(cs.size());
        // cleared beside vg_insert: the cells of the last frame's rows, the dense tensor; beside vg_flags: coordinate
        // rows beyond the active ones where the flags ask for them (the cells are found by them)
        FillArgs clears, pads;
        std::vector<FillArgs> overflow;  // (of a backbone with dozens of strided layers)
        std::vector<CleanPart> cleans;
        for (int i = 1; i <= m; ++i) {
            ConvStage& st = *stages[(size_t)cs[(size_t)i].layer];
            rows[(size_t)i] = {static_cast<const int32_t*>(st.coors.p), static_cast<const int32_t*>(st.num.p), cellTable(st),
                               rows[(size_t)i - 1].num, V};
            part[(size_t)i] = st.sparse->part(rows[(size_t)i - 1].coors, rows[(size_t)i - 1].num, static_cast<int32_t*>(st.coors.p),
                                              static_cast<int32_t*>(st.num.p), st.ws.p, false);
            part[(size_t)i].t = rows[(size_t)i].table;
            part[(size_t)i].taken = st.cells.taken();
            for (FillArgs* f : {&clears, &pads})
                if (f->n + 6 > FillArgs::kMaxRegions) {
                    overflow.push_back(*f);
                    *f = FillArgs();
                }
            if (st.cells.cells && cleans.size() < (size_t)kMaxCleans) {
                cleans.push_back(st.cells.clean(rows[(size_t)i].table, V));
            } else if (st.cells.cells) {
                st.cells.collectFill(clears);
            } else {
                st.sparse->collectTableFill(st.ws.p, clears);
            }
            st.sparse->collectPadFill(static_cast<int32_t*>(st.coors.p), pads);
        }
        vg->collectPadFill(static_cast<float*>(vg_voxels.p), static_cast<int32_t*>(vg_coors.p), clears);
        if (denseByEpilogue()) s2d->collectFill(dense, s2d_ws.p, clears);

        VgPart v = vg->part(static_cast<const float*>(points), static_cast<const int32_t*>(points_size), desc.max_points,
                                  desc.point_features, static_cast<float*>(vg_voxels.p), static_cast<int32_t*>(vg_coors.p),
                                  static_cast<int32_t*>(vg_num.p), vg_ws.p);
        v.t = rows[0].table;
        v.taken = vg_cells.taken();
        SESSD_TRY(launch_vg_insert(v, cleans.data(), (int)cleans.size(), clears, stream));
        for (const FillArgs& f : overflow) SESSD_TRY(launch_fill(f, stream));
        SESSD_TRY(launch_vg_flags(v, pads, stream));
        SESSD_TRY(launch_vg_finalize(v, m ? &part[1] : nullptr, stream));

        // Coordinate passes are counted 2i (flags + lookups of stage i) and 2i + 1 (numbering, cuts, builds).  ready[l] = the
        // pass layer l's rulebook is complete after; pass 0 runs on the caller's stream.  works[p]: it does something on the other.
        std::vector<int> ready(stages.size(), 0);
        std::vector<char> works((size_t)(2 * m + 2), 0);
        for (int i = 0; i <= m; ++i) {
            const Stage& sg = cs[(size_t)i];
            works[(size_t)(2 * i)] = i > 0;
            works[(size_t)(2 * i + 1)] = i < m || i == 1 || m == 0 || !sg.builds.empty();
            for (int l : sg.lookups) {
                const ConvStage& st = *stages[(size_t)l];
                const bool cuts = st.subm ? st.subm->wantTileCuts() : st.sparse->wantTileCuts();
                ready[(size_t)l] = 2 * i + (cuts ? 1 : 0);
                if (cuts) works[(size_t)(2 * i + 1)] = 1;
            }
            for (int l : sg.builds) ready[(size_t)l] = 2 * i + 1;
        }
        // The first layers and the passes up to the first strided layer's rulebook take about as long as each other, and between two
        // branches a graph loses 7 us where the second begins and 8 to 10 where one waits for what the other has just done.  So
        // they share launches on the caller's stream: pass 1 with layer 0's products, where its kernel leaves the pass room, pass 2 with layer 1's
        // (or, where the first strided layer is next, alone).  The other branch begins behind pass 1, with the flags for pass 3.  The figures
        // are at the kernels (coord.hip).  (Flags beside the lookups as well, the branch behind pass 2: 2 000 points 1.04x, the passes end too late.)
        // Where pass 2 cannot follow on the caller's stream the branches begin behind pass 0 and nothing is shared.  Layer 0 alone beside pass 1, the
        // branches behind it / so, us: voxels' table not kept, FP32 2 000 points 183.7 / 183.0, 14 000 256.3 / 250.4, 80 000 430.2 / 427.4, FP16 8 000
        // 178.2 / 174.6, 60 000 225.9 / 221.0; FP32 doubled widths 2 000 248.2 / 246.7, 20 000 564.4 / 558.5, 40 000 717.2 / 714.8, 80 000 973.9 / 978.9.  On one stream
        // sharing costs no branch anything: FP32 doubled widths 2 000 points 325.2 -> 320.5, 20 000 626.8 -> 623.7.
        int last_main = 0, clean_at = m < 1 ? 0 : 1;  // (stage 1's own rulebook is the last reader of the voxels' table)
        int beside[3] = {-1, -1, -1};
        auto rulebookPass = [&](size_t l) { return ready[(size_t)(stages[l]->rulebook_from >= 0 ? stages[l]->rulebook_from : (int)l)]; };
        auto productsOf = [&](size_t l) {
            return stages[l]->subm->sharedGemmArgs(l ? stages[l - 1]->feat.p : vg_voxels.p, stages[l]->feat.p, static_cast<const int32_t*>(vg_num.p),
                                                   stages[(size_t)(stages[l]->rulebook_from >= 0 ? stages[l]->rulebook_from : (int)l)]->ws.p);
        };
        const bool fork = aux != nullptr && stages.size() > 0;
        if (m >= 1 && stages.size() > 2 && cs[0].builds.empty() && cs[0].lookups.size() <= (size_t)kMaxCuts && stages[0]->subm && rulebookPass(0) == 0 &&
            number_takes_products(productsOf(0))) {
            beside[1] = 0;
            last_main = 1;
            bool lookups_alone = cs[1].builds.empty() && cs[1].lookups.size() <= (size_t)kMaxLookups;  // (no cuts, no builds: nothing of pass 3 reads them)
            for (int l : cs[1].lookups) lookups_alone = lookups_alone && ready[(size_t)l] == 2;
            if (lookups_alone && rulebookPass(1) == 2) {
                last_main = 2;
            } else if (lookups_alone && stages[1]->subm && rulebookPass(1) == 0 && rows[0].table.dense && rows[1].table.dense &&
                       lookups_take_products(productsOf(1), nullptr, 0)) {
                beside[2] = 1;
                last_main = 2;
            }
            if (fork && last_main == 1) {
                beside[1] = -1;
                last_main = 0;
            }
        }
        const bool apart = fork && last_main == 2;  // pass 2 runs beside the passes behind it but for the one that empties the table
        if (apart && m >= 2) {
            clean_at = 2;
            works[5] = 1;
        }
        int last_side = 2 * m + 1;
        while (last_side > 0 && !works[(size_t)last_side]) --last_side;
        // wait_for[l]: the pass that layer l has the chain wait for (0: none); an event stands for each of them and for the join, for no
        // other pass.  A wait for the other branch costs the chain 4-5 us in a graph, however long the pass has been done.  Behind the
        // second strided layer the branch is ahead of the chain: a layer that waits there waits for the next stage's passes as well, and
        // for all that are left where these are two stages', but for no rulebook that a later layer builds on a grid of its own.
        // Each pass by itself / for the branch's end / so, us: the reference's backbone, FP32 2 000 points 183, 178, 178, 20 000 252, 247, 247,
        // FP16 60 000 222, 219, 219 (so is its end); four strided layers more, each with two SubM layers, FP32 2 000 points 343, 371, 330,
        // 20 000 487, 517, 474, FP16 20 000 319, 328, 311; twelve more, FP32 2 000 675, 770, 645.
        // Passes that are waited for one by one: to the lookups on the second strided layer's rows, with few points where pass 2 is on the caller's
        // stream to their tile cuts.  Four / five so, FP32, us: 2 000 points 179.3 / 165.5 (the branch's end is 15 us away then), 4 000 195.6 / 185.5, 8 000
        // 204.4 / 201.2, 10 000 213.9 / 212.2, 12 000 220.6 / 222.8, 14 000 221.5 / 223.4, 16 000 229.9 / 224.2, 18 000 233.8 / 231.2, 20 000 253.8 / 255.1, 30 000
        // to 80 000 five 1.003-1.008x; one SubM layer in front 2 000 179.0 / 164.0, 20 000 251.3 / 245.5; three 2 000 179.8 / 171.1, 8 000 204.7 / 206.5.
        // Elsewhere: doubled widths 2 000 248.2 / 250.6, 5 000 326.7 / 329.5, 10 000 431.8 / 434.6; without a kept table of the voxels 2 000 183.7 / 187.2, 8 000
        // 224.9 / 227.9.  FP16 layers need no cuts: the same frames.
        const int kOwnWaits = apart && desc.max_points <= 10000 ? 5 : 4;
        constexpr int kAhead = 2, kRest = 4;
        hipStream_t side = fork ? aux : stream;
        std::vector<int> wait_for(stages.size(), 0);
        std::vector<char> awaited((size_t)(2 * m + 2), 0);
        bool join = false;  // at the end, for what no layer has waited for
        int longer = -3;    // passes less layers in front of the last layer until the second strided layer's rulebook that needs a pass anew
        if (fork) {
            int seen = 0;
            for (size_t l = 0; l < stages.size(); ++l) {
                const int pass = rulebookPass(l);
                if (pass <= seen) continue;
                seen = pass;
                if (pass <= 5) longer = pass - (int)l;
            }
            int waited = last_main;
            for (size_t l = 0; l < stages.size(); ++l) {
                const int pass = rulebookPass(l);
                if (pass <= waited) continue;
                waited = pass;
                const int end = pass <= kOwnWaits ? pass : (last_side - pass <= kRest ? last_side : pass + kAhead);
                for (int p = pass + 1; p <= end; ++p) {
                    if (p % 2 && !cs[(size_t)(p / 2)].builds.empty()) break;
                    if (works[(size_t)p]) waited = p;
                }
                wait_for[l] = waited;
                awaited[(size_t)waited] = 1;
            }
            join = last_side > waited;
            if (join) awaited[(size_t)last_side] = 1;
        }
        // The feature chain, as far as the passes up to `last_pass` allow.
        const void* feat = vg_voxels.p;
        const int32_t* coors = static_cast<const int32_t*>(vg_coors.p);
        const int32_t* num = static_cast<const int32_t*>(vg_num.p);
        size_t next_layer = 0;
        bool scattered = false;
        auto layers = [&](int last_pass) -> int {
            for (; next_layer < stages.size(); ++next_layer) {
                ConvStage& st = *stages[next_layer];
                const int owner = st.rulebook_from >= 0 ? st.rulebook_from : (int)next_layer;
                if (ready[(size_t)owner] > last_pass) return SESSD_OK;
                if (wait_for[next_layer]) SESSD_HIP_TRY(hipStreamWaitEvent(stream, ev_pass[(size_t)wait_for[next_layer]], 0));
                DenseTarget dt;
                const bool fuse = next_layer + 1 == stages.size() && denseByEpilogue();
                if (fuse) {
                    const int32_t* oc = st.subm ? coors : static_cast<const int32_t*>(st.coors.p);
                    dt = s2d->denseTarget(dense, oc, s2d_ws.p);
                    scattered = true;
                }
                if (st.subm) {
                    SESSD_TRY(st.subm->enqueueGemm(feat, st.feat.p, num, stages[(size_t)owner]->ws.p, stream, fuse ? &dt : nullptr));
                } else {
                    SESSD_TRY(st.sparse->enqueueGemm(feat, st.feat.p, static_cast<const int32_t*>(st.num.p), st.ws.p, stream,
                                                     fuse ? &dt : nullptr));
                    coors = static_cast<const int32_t*>(st.coors.p);
                    num = static_cast<const int32_t*>(st.num.p);
                }
                feat = st.feat.p;
            }
            return SESSD_OK;
        };
        // Of the two branches the one that is launched first follows at once in a graph, the other 6 us later.  Behind shared launches
        // that is the chain (flags and pass 3 captured in front of pass 2: 2 000 points FP32 165.9 -> 175.6 us, FP16 144.8 -> 152.4, 20 000 252.8 -> 258.2 and 169.6 ->
        // 178.2).  Elsewhere a layer takes a little less than a pass with few points, and layers grow with the points and passes hardly,
        // in FP16 a third as fast: it is the passes with up to two SubM layers in front of the first strided one until 50 000 points (FP16 150 000), with
        // three until 10 000 (30 000), and always the chain with more.  Passes first / chain first, us, FP32 and FP16, the reference's backbone
        // 2 000 points 172.6 / 176.5, 149.6 / 154.6, 20 000 259.2 / 260.0, 174.1 / 179.6, 40 000 311.0 / 311.6, 60 000 350.0 / 344.3, 191.6 / 196.2, 80 000 387.2 / 384.9, on
        // hashes 2 000 195.9 / 199.1, 171.3 / 174.9, 20 000 286.0 / 291.5, 205.6 / 210.0, 60 000 FP16 247.1 / 251.4, 80 000 446.8 / 440.8; one SubM layer 5 000 198.6 /
        // 202.2, 20 000 253.4 / 257.1; three 8 000 215.2 / 215.7, 159.4 / 161.9, 20 000 269.9 / 267.7, 177.8 / 178.8, 40 000 329.9 / 322.3, 60 000 FP16 202.9 / 198.7; four 2 000
        // 179.5 / 177.2, 156.8 / 155.1, 20 000 276.2 / 272.5, 182.7 / 178.4, 40 000 340.4 / 329.3, 60 000 FP16 209.6 / 197.1; doubled widths 5 000 322.5 / 325.3, 20 000 544.0 /
        // 550.5, 80 000 978.9 / 969.2, FP16 8 000 220.4 / 223.5, 60 000 303.6 / 302.6, 150 000 425.7 / 429.9.  The points are those that the tensor holds, which is what the host
        // knows.
        const bool half = desc.feature_dtype == SESSD_HALF;
        const int ahead = longer + (half ? 1 : 0);  // (FP16 layers need no tile cuts: one pass less)
        const bool chain_first = apart || ahead < -1 || desc.max_points > (half ? 3 : 1) * (ahead < 0 ? 10000 : 50000);
        auto behindPass = [&](int pass) -> int {
            if (!fork) return SESSD_OK;
            if (pass == (apart ? 1 : 0)) {
                SESSD_HIP_TRY(hipEventRecord(ev_head, stream));
                SESSD_HIP_TRY(hipStreamWaitEvent(side, ev_head, 0));
            }
            if (apart && pass == 2) SESSD_HIP_TRY(hipEventRecord(ev_pass[2], stream));
            if (pass == last_main && chain_first) return layers(last_main);
            if (awaited[(size_t)pass]) SESSD_HIP_TRY(hipEventRecord(ev_pass[(size_t)pass], side));
            return SESSD_OK;
        };
        auto launched = [&](int l) {  // (beside a pass)
            feat = stages[(size_t)l]->feat.p;
            next_layer = (size_t)l + 1;
        };
        for (int i = 0; i <= m; ++i) {
            const Stage& sg = cs[(size_t)i];
            hipStream_t s = 2 * i <= last_main ? stream : side, s_number = 2 * i + 1 <= last_main ? stream : side;
            const int with_lookups = 2 * i <= last_main ? beside[(size_t)(2 * i)] : -1, with_number = 2 * i + 1 <= last_main ? beside[(size_t)(2 * i + 1)] : -1;
            // flags of the next strided layer and the lookups on this stage's rows
            std::vector<LookupPart> looks;
            std::vector<CutPart> cuts;
            for (int l : sg.lookups) {
                ConvStage& st = *stages[(size_t)l];
                if (st.sparse) {
                    const Rows& in = rows[(size_t)i - 1];
                    looks.push_back(st.sparse->lookupPart(st.ws.p, rows[(size_t)i].coors, rows[(size_t)i].num, in.table, in.table_num, in.table_max));
                    if (st.sparse->wantTileCuts()) cuts.push_back(st.sparse->cutPart(st.ws.p, rows[(size_t)i].num));
                } else {
                    const Rows& r = rows[(size_t)i];
                    looks.push_back(st.subm->lookupPart(st.ws.p, r.coors, r.num, r.table, r.table_num, r.table_max));
                    if (st.subm->wantTileCuts()) cuts.push_back(st.subm->cutPart(st.ws.p, r.num));
                }
            }
            const SpPart* next = i < m ? &part[(size_t)i + 1] : nullptr;
            const SpPart* flags = apart && i == 1 ? nullptr : next;
            size_t at = 0;
            if (with_lookups >= 0) {
                SESSD_TRY(launch_flags_lookups_products(flags, looks.data(), (int)looks.size(), productsOf((size_t)with_lookups), s));
                launched(with_lookups);
                at = looks.size();
            } else do {
                const size_t n = looks.size() - at < (size_t)kMaxLookups ? looks.size() - at : (size_t)kMaxLookups;
                SESSD_TRY(launch_flags_lookups(at == 0 ? flags : nullptr, looks.data() + at, (int)n, s));
                at += n;
            } while (at < looks.size());
            SESSD_TRY(behindPass(2 * i));
            if (next && !flags) SESSD_TRY(launch_sp_flags(*next, side));
            if (apart && i == clean_at) SESSD_HIP_TRY(hipStreamWaitEvent(side, ev_pass[2], 0));
            // numbering of the next strided layer's rows (their tickets for the layer behind it), tile cuts
            FillArgs clear;
            CleanPart clean;
            if (i == clean_at && vg_cells.cells) {
                clean = vg_cells.clean(rows[0].table, desc.voxelgen.max_voxels);
            } else if (i == clean_at) {
                vg->collectTableFill(vg_ws.p, desc.max_points, true, clear);
            }
            const SpPart* after = i + 1 < m ? &part[(size_t)i + 2] : nullptr;
            at = 0;
            bool did = false;
            if (with_number >= 0) {
                SESSD_TRY(launch_number_products(next, after, cuts.data(), (int)cuts.size(), clean.taken ? &clean : nullptr, &clear, productsOf((size_t)with_number),
                                                 s_number));
                launched(with_number);
                at = cuts.size();
                did = true;
            }
            while (at < cuts.size() || (!did && (next || i == clean_at))) {
                const size_t n = cuts.size() - at < (size_t)kMaxCuts ? cuts.size() - at : (size_t)kMaxCuts;
                SESSD_TRY(launch_number(did ? nullptr : next, did ? nullptr : after, cuts.data() + at, (int)n, did || !clean.taken ? nullptr : &clean,
                                        did ? nullptr : &clear, s_number));
                at += n;
                did = true;
            }
            for (int l : sg.builds) {
                ConvStage& st = *stages[(size_t)l];
                SESSD_TRY(st.subm->enqueueBuild(rows[(size_t)i].coors, rows[(size_t)i].num, st.ws.p, side));
            }
            SESSD_TRY(behindPass(2 * i + 1));
        }

        SESSD_TRY(layers(2 * m + 1));
        if (join) SESSD_HIP_TRY(hipStreamWaitEvent(stream, ev_pass[(size_t)last_side], 0));
        if (scattered) return SESSD_OK;
        const void* din[3] = {feat, coors, num};
        void* dout[1] = {dense};
        return s2d->enqueue(s2d_in, s2d_out, din, dout, s2d_ws.p, stream);
    }

    // plugin by plugin, each with its own clears and tables (enqueue_timed: what each of them costs alone)
    int enqueueAfterVoxelizer(void* dense, hipStream_t stream) {
        const void* feat = vg_voxels.p;
        const void* coors = vg_coors.p;
        const void* num = vg_num.p;
        for (auto& st : stages) {
            const void* in[3] = {feat, coors, num};
            if (st->subm) {
                void* out[1] = {st->feat.p};
                if (st->rulebook_from >= 0)
                    SESSD_TRY(st->subm->enqueueShared(st->in_desc, st->out_desc, in, out,
                                                      stages[st->rulebook_from]->ws.p, stream));
                else
                    SESSD_TRY(st->subm->enqueue(st->in_desc, st->out_desc, in, out, st->ws.p, stream));
            } else {
                void* out[3] = {st->feat.p, st->coors.p, st->num.p};
                SESSD_TRY(st->sparse->enqueue(st->in_desc, st->out_desc, in, out, st->ws.p, stream));
                coors = st->coors.p;
                num = st->num.p;
            }
            feat = st->feat.p;
        }
        const void* din[3] = {feat, coors, num};
        void* dout[1] = {dense};
        return s2d->enqueue(s2d_in, s2d_out, din, dout, s2d_ws.p, stream);
    }
};

// largest output grid that gets a kept table (a ticket keeps its cell in 26 bits)
constexpr uint64_t kDenseCells = 1ull << 25;
// ... and largest voxel grid
constexpr uint64_t kDenseVoxelCells = 1ull << 27;

static int build_pipeline(const sessd_pipeline_desc& d, Pipeline* P) {
    if (d.n_layers < 0 || (d.n_layers && (!d.layers || !d.weights)))
        return fail(SESSD_E_INVALID, "pipeline: layers/weights missing");
    if (d.feature_dtype != SESSD_FLOAT && d.feature_dtype != SESSD_HALF)
        return fail(SESSD_E_UNSUPPORTED, "pipeline: feature_dtype must be FP32 or FP16");
    if (d.max_points <= 0 || d.point_features < 4) return fail(SESSD_E_INVALID, "pipeline: bad points shape");
    P->desc = d;
    // rows of every conv-layer tensor; the voxelizer's own cap (voxelgen.max_voxels) may be lower: strided
    // layers can produce more sites than they are given
    const int V = d.layer_max_voxels > 0 ? d.layer_max_voxels : d.voxelgen.max_voxels;
    if (V < d.voxelgen.max_voxels) return fail(SESSD_E_INVALID, "pipeline: layer_max_voxels below the voxelizer's cap");
    const int VG = d.voxelgen.max_voxels;
    P->max_voxels = V;
    const int ft = d.feature_dtype;
    size_t total = 0;

    VoxelGeneratorPlugin* vg = nullptr;
    SESSD_TRY(VoxelGeneratorPlugin::create(d.voxelgen, &vg));
    P->vg.reset(vg);
    vg->flags_ = d.flags;
    P->vg_in[0] = make_desc({1, d.max_points, d.point_features}, SESSD_FLOAT);
    P->vg_in[1] = make_desc({1}, SESSD_INT32);
    P->vg_out[0] = make_desc({1, VG, 4}, SESSD_FLOAT);
    P->vg_out[1] = make_desc({1, VG, 4}, SESSD_INT32);
    P->vg_out[2] = make_desc({1}, SESSD_INT32);
    SESSD_TRY(vg->configurePlugin(P->vg_in, 2, P->vg_out, 3));
    SESSD_TRY(P->vg_ws.alloc(vg->getWorkspaceSize(P->vg_in, 2, P->vg_out, 3)));
    SESSD_TRY(P->vg_voxels.alloc((size_t)V * 4 * sizeof(float)));
    SESSD_TRY(P->vg_coors.alloc((size_t)V * 4 * sizeof(int32_t)));
    SESSD_TRY(P->vg_num.alloc(256));
    total += P->vg_ws.bytes + P->vg_voxels.bytes + P->vg_coors.bytes + 256;

    int in_type = SESSD_FLOAT;  // the voxelizer's means are FP32
    int in_ch = 4;
    int last_subm_with_rulebook = -1;
    for (int l = 0; l < d.n_layers; ++l) {
        const sessd_layer_spec& s = d.layers[l];
        if (s.in_channel != in_ch)
            return fail(SESSD_E_INVALID, "pipeline: layer %d expects %d input channels, previous layer has %d", l,
                        s.in_channel, in_ch);
        auto st = std::make_unique<ConvStage>();
        st->spec = s;
        st->in_desc[0] = make_desc({1, V, s.in_channel}, in_type);
        st->in_desc[1] = make_desc({1, V, 4}, SESSD_INT32);
        st->in_desc[2] = make_desc({1}, SESSD_INT32);
        st->out_desc[0] = make_desc({1, V, s.out_channel}, ft);
        st->out_desc[1] = make_desc({1, V, 4}, SESSD_INT32);
        st->out_desc[2] = make_desc({1}, SESSD_INT32);
        ConvPluginBase* base = nullptr;
        if (s.type == SESSD_LAYER_SUBM) {
            sessd_submconv3d_desc cd;
            std::memset(&cd, 0, sizeof(cd));
            cd.in_channel = s.in_channel;
            cd.out_channel = s.out_channel;
            cd.max_voxels = V;
            cd.feature_num = s.in_channel;  // se-ssd-ai-trt.cpp:739
            for (int a = 0; a < 3; ++a) cd.out_shape[a] = cd.spatial_shape[a] = s.out_shape[a];
            cd.ksize = s.ksize[0];
            cd.stride = s.stride[0];
            cd.padding = s.padding[0];
            cd.dilation = 1;
            SubmConv3dLayerPlugin* p = nullptr;
            SESSD_TRY(SubmConv3dLayerPlugin::create(cd, d.weights[l], &p));
            st->subm.reset(p);
            base = p;
            SESSD_TRY(p->configurePlugin(st->in_desc, 3, st->out_desc, 1));
            if (d.share_rulebooks && last_subm_with_rulebook >= 0) {
                const sessd_layer_spec& o = d.layers[last_subm_with_rulebook];
                bool same = o.ksize[0] == s.ksize[0] && o.padding[0] == s.padding[0];
                for (int a = 0; a < 3; ++a) same = same && o.out_shape[a] == s.out_shape[a];
                if (same) st->rulebook_from = last_subm_with_rulebook;
            }
            if (st->rulebook_from < 0) {
                SESSD_TRY(st->ws.alloc(p->getWorkspaceSize(st->in_desc, 3, st->out_desc, 1)));
                last_subm_with_rulebook = l;
            }
        } else if (s.type == SESSD_LAYER_SPARSE) {
            sessd_sparseconv3d_desc cd;
            std::memset(&cd, 0, sizeof(cd));
            cd.in_channel = s.in_channel;
            cd.out_channel = s.out_channel;
            cd.max_voxels = V;
            cd.feature_num = s.in_channel;
            for (int a = 0; a < 3; ++a) {
                cd.out_shape[a] = s.out_shape[a];
                cd.ksize[a] = s.ksize[a];
                cd.stride[a] = s.stride[a];
                cd.padding[a] = s.padding[a];
            }
            cd.dilation = 1;
            SparseConv3dLayerPlugin* p = nullptr;
            SESSD_TRY(SparseConv3dLayerPlugin::create(cd, d.weights[l], &p));
            st->sparse.reset(p);
            base = p;
            SESSD_TRY(p->configurePlugin(st->in_desc, 3, st->out_desc, 3));
            SESSD_TRY(st->ws.alloc(p->getWorkspaceSize(st->in_desc, 3, st->out_desc, 3)));
            SESSD_TRY(st->coors.alloc((size_t)V * 4 * sizeof(int32_t)));
            SESSD_TRY(st->num.alloc(256));
            last_subm_with_rulebook = -1;  // new coordinates: earlier rulebooks no longer apply
        } else {
            return fail(SESSD_E_INVALID, "pipeline: layer %d has unknown type %d", l, s.type);
        }
        base->flags_ = d.flags;
        SESSD_TRY(base->setEpilogue(d.scale ? d.scale[l] : nullptr, d.shift ? d.shift[l] : nullptr, d.relu));
        SESSD_TRY(st->feat.alloc((size_t)V * s.out_channel * dtype_size(ft)));
        total += st->ws.bytes + st->feat.bytes + st->coors.bytes + st->num.bytes;
        in_type = ft;
        in_ch = s.out_channel;
        P->stages.push_back(std::move(st));
    }

    if (d.dense.feature_map_channel != in_ch)
        return fail(SESSD_E_INVALID, "pipeline: sparse2dense expects %d channels, backbone ends with %d",
                    d.dense.feature_map_channel, in_ch);
    Sparse2DensePlugin* s2d = nullptr;
    SESSD_TRY(Sparse2DensePlugin::create(d.dense, &s2d));
    P->s2d.reset(s2d);
    SESSD_TRY(s2d->setPadding(d.dense_padding[0], d.dense_padding[1], d.dense_padding[2], d.dense_padding[3]));
    P->s2d_in[0] = make_desc({1, V, in_ch}, in_type);
    P->s2d_in[1] = make_desc({1, V, 4}, SESSD_INT32);
    P->s2d_in[2] = make_desc({1}, SESSD_INT32);
    P->s2d_out[0] = make_desc({1, d.dense.feature_map_channel * d.dense.feature_map_size[2], s2d->outHeight(),
                               s2d->outWidth()}, ft);
    SESSD_TRY(s2d->configurePlugin(P->s2d_in, 3, P->s2d_out, 1));
    SESSD_TRY(P->s2d_ws.alloc(s2d->getWorkspaceSize(P->s2d_in, 3, P->s2d_out, 1)));
    total += P->s2d_ws.bytes;
    P->device_bytes = total;
    if (d.overlap_streams) {
        SESSD_HIP_TRY(hipStreamCreateWithFlags(&P->aux, hipStreamNonBlocking));
        SESSD_HIP_TRY(hipEventCreateWithFlags(&P->ev_head, hipEventDisableTiming));
        P->ev_pass.assign(2 * P->coordStages().size(), nullptr);
        for (auto& e : P->ev_pass) SESSD_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    // the layer array of the caller need not outlive create()
    P->desc.layers = nullptr;
    P->desc.weights = P->desc.scale = P->desc.shift = nullptr;
    return SESSD_OK;
}

// Behind everything that a pipeline (all its replicas) cannot do without: the tables it keeps.  Where memory for one is
// short, the table in the workspace does, which every frame clears.
static int finish_pipeline(Pipeline* P) {
    const VoxelGeneratorPlugin& vg = *P->vg;
    const uint64_t cells = (uint64_t)vg.grid_x_size_ * (uint64_t)vg.grid_y_size_ * (uint64_t)vg.grid_z_size_;
    if (cells <= kDenseVoxelCells) (void)P->vg_cells.alloc(cells, P->desc.voxelgen.max_voxels);
    P->device_bytes += P->vg_cells.mem.bytes;
    for (auto& st : P->stages) {
        if (!st->sparse) continue;
        const uint64_t volume = (uint64_t)st->spec.out_shape[0] * (uint64_t)st->spec.out_shape[1] * (uint64_t)st->spec.out_shape[2];
        if (volume <= kDenseCells) (void)st->cells.alloc(volume, P->max_voxels);
        P->device_bytes += st->cells.mem.bytes;
    }
    // what the passes leave as they need it for the next frame has to be right for the first
    SESSD_TRY(P->resetState(nullptr));
    FillArgs counts;  // queries before the first frame find no rows
    counts.add(P->vg_num.p, 4, 0);
    for (auto& st : P->stages) {
        if (counts.full()) {
            SESSD_TRY(launch_fill(counts, nullptr));
            counts = FillArgs();
        }
        counts.add(st->num.p, 4, 0);
    }
    SESSD_TRY(launch_fill(counts, nullptr));
    SESSD_HIP_TRY(hipStreamSynchronize(nullptr));
    return SESSD_OK;
}

}  // namespace sessd

using namespace sessd;

extern "C" {

int sessd_reference_backbone(sessd_layer_spec* layers, int max_layers, sessd_voxelgen_desc* voxelgen,
                             sessd_sparse2dense_desc* dense) {
    // params.h:39-192: {type, cin, cout, ksize zyx, stride zyx, padding zyx, out_shape xyz}
    static const sessd_layer_spec table[14] = {
        {SESSD_LAYER_SUBM, 4, 16, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {1408, 1600, 41}},
        {SESSD_LAYER_SUBM, 16, 16, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {1408, 1600, 41}},
        {SESSD_LAYER_SPARSE, 16, 32, {3, 3, 3}, {2, 2, 2}, {1, 1, 1}, {704, 800, 21}},
        {SESSD_LAYER_SUBM, 32, 32, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {704, 800, 21}},
        {SESSD_LAYER_SUBM, 32, 32, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {704, 800, 21}},
        {SESSD_LAYER_SPARSE, 32, 64, {3, 3, 3}, {2, 2, 2}, {1, 1, 1}, {352, 400, 11}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {352, 400, 11}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {352, 400, 11}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {352, 400, 11}},
        {SESSD_LAYER_SPARSE, 64, 64, {3, 3, 3}, {2, 2, 2}, {0, 1, 1}, {176, 200, 5}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {176, 200, 5}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {176, 200, 5}},
        {SESSD_LAYER_SUBM, 64, 64, {3, 3, 3}, {1, 1, 1}, {1, 1, 1}, {176, 200, 5}},
        {SESSD_LAYER_SPARSE, 64, 64, {3, 1, 1}, {2, 1, 1}, {0, 0, 0}, {176, 200, 2}},
    };
    int n = 0;
    if (layers)
        for (; n < 14 && n < max_layers; ++n) layers[n] = table[n];
    if (voxelgen) {  // params.h:19-36
        voxelgen->max_num_points_per_voxel = 5;
        voxelgen->max_voxels = 60000;
        const float r[6] = {0.0f, -40.0f, -3.0f, 70.4f, 40.0f, 1.0f};
        for (int i = 0; i < 6; ++i) voxelgen->point_cloud_range[i] = r[i];
        voxelgen->voxel_feature_num = 4;
        voxelgen->voxel_size[0] = 0.05f;
        voxelgen->voxel_size[1] = 0.05f;
        voxelgen->voxel_size[2] = 0.1f;
    }
    if (dense) {  // params.h:194-197
        dense->feature_map_size[0] = 176;
        dense->feature_map_size[1] = 200;
        dense->feature_map_size[2] = 2;
        dense->feature_map_channel = 64;
    }
    return n;
}

static int pipeline_create_unguarded(const sessd_pipeline_desc* desc, sessd_pipeline** out) {
    std::unique_ptr<Pipeline> P(new Pipeline());
    if (desc->frames_in_flight >= 2) {
        // R replicas, each a complete pipeline with a stream of its own; this object only holds them and the turn
        if (desc->frames_in_flight > 8) return fail(SESSD_E_INVALID, "pipeline: at most 8 frames in flight");
        if (!desc->overlap_streams)
            return fail(SESSD_E_INVALID, "pipeline: frames_in_flight needs overlap_streams");
        sessd_pipeline_desc one = *desc;
        one.frames_in_flight = 0;
        for (int r = 0; r < desc->frames_in_flight; ++r) {
            std::unique_ptr<Pipeline> rep(new Pipeline());
            SESSD_TRY(build_pipeline(one, rep.get()));
            for (hipEvent_t* e : {&rep->ev_in, &rep->ev_frame_done})
                SESSD_HIP_TRY(hipEventCreateWithFlags(e, hipEventDisableTiming));
            SESSD_HIP_TRY(hipStreamCreateWithFlags(&rep->frame_stream, hipStreamNonBlocking));
            P->max_voxels = rep->max_voxels;
            P->replicas.push_back(std::move(rep));
        }
        for (auto& rep : P->replicas) {
            SESSD_TRY(finish_pipeline(rep.get()));
            P->device_bytes += rep->device_bytes;
        }
        P->desc = *desc;
        P->desc.layers = nullptr;
        P->desc.weights = P->desc.scale = P->desc.shift = nullptr;
    } else {
        SESSD_TRY(build_pipeline(*desc, P.get()));
        SESSD_TRY(finish_pipeline(P.get()));
    }
    *out = reinterpret_cast<sessd_pipeline*>(P.release());
    return SESSD_OK;
}

int sessd_pipeline_create(const sessd_pipeline_desc* desc, sessd_pipeline** out) {
    if (!desc || !out) return fail(SESSD_E_INVALID, "pipeline_create: null argument");
    return guarded(__func__, [&]() -> int { return pipeline_create_unguarded(desc, out); });
}

// the pipeline whose tensors a query is about: with frames in flight, the replica of the last submitted frame
static Pipeline* current(sessd_pipeline* h) {
    auto* P = reinterpret_cast<Pipeline*>(h);
    return P->replicas.empty() ? P : P->replicas[(size_t)P->last_replica].get();
}

// one frame on `stream`: a replay of the captured graph when the pipeline uses graphs (re-captured when a pointer
// changed), direct launches otherwise
static int run_frame(Pipeline* P, const void* points, const void* points_size, void* dense, hipStream_t stream) {
    auto run = [&]() -> int {  // (building the passes of a frame allocates on the host)
        const int rc = guarded("pipeline", [&]() -> int { return P->enqueueFrame(points, points_size, dense, stream); });
        return rc == SESSD_OK ? rc : P->recover(stream, rc);
    };
    if (!P->tables_ready) {
        const bool captured = P->captureStatus(stream) != hipStreamCaptureStatusNone;
        if (!captured) SESSD_TRY(P->joinAux(stream));
        SESSD_TRY(P->resetState(stream));
        if (captured) {  // the caller's own graph: nothing is cleared until it is launched
            P->tables_ready = false;
            return run();
        }
    }
    if (!P->desc.use_graph || stream == nullptr) return run();
    CapturedGraph& g = P->captured;
    if (!g.exec || g.points != points || g.size != points_size || g.dense != dense) {
        g.reset();
        SESSD_HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        const int rc = run();
        hipGraph_t captured = nullptr;
        const hipError_t e = hipStreamEndCapture(stream, &captured);
        if (rc != SESSD_OK) {
            if (captured) (void)hipGraphDestroy(captured);
            return rc;
        }
        if (e != hipSuccess) return fail(SESSD_E_HIP, "pipeline: stream capture failed: %s", hipGetErrorString(e));
        g.graph = captured;
        SESSD_HIP_TRY(hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0));
        size_t nodes = 0;
        if (hipGraphGetNodes(g.graph, nullptr, &nodes) == hipSuccess) g.nodes = (int)nodes;
        g.points = points;
        g.size = points_size;
        g.dense = dense;
    }
    const hipError_t e = hipGraphLaunch(g.exec, stream);
    if (e == hipSuccess) return SESSD_OK;
    return P->recover(stream, fail(SESSD_E_HIP, "pipeline: launching the captured frame failed: %s", hipGetErrorString(e)));
}

int sessd_pipeline_submit(sessd_pipeline* h, const void* points, const void* points_size, void* dense,
                          sessd_stream_t stream_, int64_t* ticket) {
    if (!h || !points || !points_size || !dense) return fail(SESSD_E_INVALID, "pipeline_submit: null argument");
    auto* P = reinterpret_cast<Pipeline*>(h);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int64_t t = P->next_ticket;
    if (P->replicas.empty()) {  // one frame at a time: the frame runs on the caller's stream, join has nothing to add
        if (stream_ == SESSD_STREAM_NONE) return fail(SESSD_E_INVALID, "pipeline_submit: SESSD_STREAM_NONE needs frames_in_flight >= 2");
        SESSD_TRY(run_frame(P, points, points_size, dense, stream));
    } else {
        const int r = (int)(t % (int64_t)P->replicas.size());
        Pipeline* R = P->replicas[(size_t)r].get();
        // the frame starts on the replica's own stream once the caller's inputs are ready (the replica's previous
        // frame precedes it on that stream)
        if (stream_ != SESSD_STREAM_NONE) {
            SESSD_HIP_TRY(hipEventRecord(R->ev_in, stream));
            SESSD_HIP_TRY(hipStreamWaitEvent(R->frame_stream, R->ev_in, 0));
        }
        const int rc = run_frame(R, points, points_size, dense, R->frame_stream);
        if (rc != SESSD_OK) {
            // no join follows: what the call has left on the replica's stream (the clears; while the caller captures, a
            // branch of that capture) is put in front of what comes next on the caller's
            if (stream_ != SESSD_STREAM_NONE && hipEventRecord(R->ev_frame_done, R->frame_stream) == hipSuccess)
                (void)hipStreamWaitEvent(stream, R->ev_frame_done, 0);
            return rc;
        }
        SESSD_HIP_TRY(hipEventRecord(R->ev_frame_done, R->frame_stream));
        P->last_replica = r;
    }
    P->next_ticket = t + 1;
    if (ticket) *ticket = t;
    return SESSD_OK;
}

int sessd_pipeline_join(sessd_pipeline* h, int64_t ticket, sessd_stream_t stream_) {
    if (!h) return fail(SESSD_E_INVALID, "pipeline_join: null handle");
    auto* P = reinterpret_cast<Pipeline*>(h);
    if (ticket < 0 || ticket >= P->next_ticket) return fail(SESSD_E_INVALID, "pipeline_join: no frame with ticket %lld", (long long)ticket);
    if (P->replicas.empty()) return SESSD_OK;  // the frame ran on the stream it was submitted on
    const int64_t R = (int64_t)P->replicas.size();
    // (a ticket older than the last R frames: its replica has been reused since; waiting for the later frame on
    // it is at least as strong)
    Pipeline* rep = P->replicas[(size_t)(ticket % R)].get();
    // no stream to make wait: the calling thread waits (SESSD_STREAM_NONE is not a stream handle)
    if (stream_ == SESSD_STREAM_NONE) SESSD_HIP_TRY(hipEventSynchronize(rep->ev_frame_done));
    else SESSD_HIP_TRY(hipStreamWaitEvent(static_cast<hipStream_t>(stream_), rep->ev_frame_done, 0));
    return SESSD_OK;
}

// Queries (status, layer statistics, layer tensors read back by the caller on `stream`) are about the last submitted
// frame: with frames in flight that frame runs on its replica's own stream, which the caller's stream has to wait
// for first.
static int order_after_last_frame(sessd_pipeline* h, hipStream_t stream) {
    auto* P = reinterpret_cast<Pipeline*>(h);
    if (P->replicas.empty() || P->next_ticket == 0) return SESSD_OK;
    Pipeline* rep = P->replicas[(size_t)P->last_replica].get();
    SESSD_HIP_TRY(hipStreamWaitEvent(stream, rep->ev_frame_done, 0));
    return SESSD_OK;
}

int sessd_pipeline_wait(sessd_pipeline* h, int64_t ticket) {
    if (!h) return fail(SESSD_E_INVALID, "pipeline_wait: null handle");
    auto* P = reinterpret_cast<Pipeline*>(h);
    if (ticket < 0 || ticket >= P->next_ticket) return fail(SESSD_E_INVALID, "pipeline_wait: no frame with ticket %lld", (long long)ticket);
    if (P->replicas.empty()) return fail(SESSD_E_INVALID, "pipeline_wait: this pipeline runs its frames on the caller's stream; synchronise that");
    Pipeline* rep = P->replicas[(size_t)(ticket % (int64_t)P->replicas.size())].get();
    SESSD_HIP_TRY(hipEventSynchronize(rep->ev_frame_done));
    return SESSD_OK;
}

int sessd_pipeline_enqueue(sessd_pipeline* h, const void* points, const void* points_size, void* dense,
                           sessd_stream_t stream) {
    int64_t ticket = 0;
    SESSD_TRY(sessd_pipeline_submit(h, points, points_size, dense, stream, &ticket));
    return sessd_pipeline_join(h, ticket, stream);
}

int sessd_pipeline_layer_io(sessd_pipeline* h, int layer, void** feat, void** coors, void** voxel_num,
                            void** workspace, int32_t* channels) {
    if (!h) return fail(SESSD_E_INVALID, "pipeline_layer_io: null handle");
    Pipeline* P = current(h);
    if (layer < -1 || layer >= (int)P->stages.size()) return fail(SESSD_E_INVALID, "pipeline_layer_io: no layer %d", layer);
    void* f = P->vg_voxels.p;
    void* c = P->vg_coors.p;
    void* n = P->vg_num.p;
    void* w = P->vg_ws.p;
    int ch = 4;
    for (int l = 0; l <= layer; ++l) {
        ConvStage& st = *P->stages[l];
        f = st.feat.p;
        ch = st.spec.out_channel;
        if (st.sparse) {
            c = st.coors.p;
            n = st.num.p;
        }
        w = st.rulebook_from >= 0 ? P->stages[st.rulebook_from]->ws.p : st.ws.p;
    }
    if (feat) *feat = f;
    if (coors) *coors = c;
    if (voxel_num) *voxel_num = n;
    if (workspace) *workspace = w;
    if (channels) *channels = ch;
    return SESSD_OK;
}

int sessd_pipeline_status(sessd_pipeline* h, sessd_stream_t stream_, int32_t* status) {
    if (!h || !status) return fail(SESSD_E_INVALID, "pipeline_status: null argument");
    Pipeline* P = current(h);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    SESSD_TRY(order_after_last_frame(h, stream));
    int32_t acc = 0, s = 0;
    SESSD_TRY(read_status_word(P->vg_ws.p, P->vg->statusOffset(), stream, &s));
    acc |= s;
    for (auto& st : P->stages) {
        if (!st->ws.p) continue;
        const size_t off = st->subm ? st->subm->statusOffset() : st->sparse->statusOffset();
        SESSD_TRY(read_status_word(st->ws.p, off, stream, &s));
        acc |= s;
    }
    SESSD_TRY(read_status_word(P->s2d_ws.p, 0, stream, &s));
    acc |= s;
    *status = acc;
    return SESSD_OK;
}

int sessd_pipeline_enqueue_timed(sessd_pipeline* h, const void* points, const void* points_size, void* dense,
                                 sessd_stream_t stream_, float* segment_ms, int max_segments, int* n_segments) {
    if (!h || !points || !points_size || !dense || !segment_ms || !n_segments)
        return fail(SESSD_E_INVALID, "pipeline_enqueue_timed: null argument");
    if (!reinterpret_cast<Pipeline*>(h)->replicas.empty())
        return fail(SESSD_E_INVALID, "pipeline_enqueue_timed: per-segment timing runs one frame on the caller's stream; "
                                     "create the pipeline without frames_in_flight for it");
    Pipeline* P = current(h);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int L = (int)P->stages.size();
    const int n_seg = 2 * L + 2;  // voxelizer, {rulebook build, gather-GEMM} per layer, sparse2dense
    if (max_segments < n_seg) return fail(SESSD_E_INVALID, "pipeline_enqueue_timed: need room for %d segments", n_seg);
    if (P->events.empty()) {
        SESSD_TRY(guarded(__func__, [&]() -> int {
            P->events.reserve(n_seg + 3);  // + two back-to-back events that bracket nothing (timer overhead)
            return SESSD_OK;
        }));
    }
    while ((int)P->events.size() < n_seg + 3) {
        hipEvent_t e = nullptr;
        SESSD_HIP_TRY(hipEventCreate(&e));
        P->events.push_back(e);
    }
    for (int l = 0; l < L; ++l) {
        ConvPluginBase* b = P->stages[l]->subm ? static_cast<ConvPluginBase*>(P->stages[l]->subm.get())
                                               : static_cast<ConvPluginBase*>(P->stages[l]->sparse.get());
        b->ev_gemm_begin_ = P->events[2 + 2 * l];
        b->ev_gemm_end_ = P->events[3 + 2 * l];
    }
    // boundaries: e0 | voxelizer | e1 | build_0 | gb_0 | gemm_0 | ge_0 | build_1 | ... | ge_{L-1} | s2d | e_last
    // the voxelizer/first-build boundary e1 is recorded by enqueueing the voxelizer separately
    SESSD_HIP_TRY(hipEventRecord(P->events[n_seg + 1], stream));
    SESSD_HIP_TRY(hipEventRecord(P->events[n_seg + 2], stream));
    SESSD_HIP_TRY(hipEventRecord(P->events[0], stream));
    int rc;
    {
        const void* vin[2] = {points, points_size};
        void* vout[3] = {P->vg_voxels.p, P->vg_coors.p, P->vg_num.p};
        rc = P->vg->enqueue(P->vg_in, P->vg_out, vin, vout, P->vg_ws.p, stream);
    }
    if (rc == SESSD_OK) rc = hipEventRecord(P->events[1], stream) == hipSuccess ? SESSD_OK : SESSD_E_HIP;
    if (rc == SESSD_OK) rc = P->enqueueAfterVoxelizer(dense, stream);
    if (rc == SESSD_OK) rc = hipEventRecord(P->events[n_seg], stream) == hipSuccess ? SESSD_OK : SESSD_E_HIP;
    for (int l = 0; l < L; ++l) {
        ConvPluginBase* b = P->stages[l]->subm ? static_cast<ConvPluginBase*>(P->stages[l]->subm.get())
                                               : static_cast<ConvPluginBase*>(P->stages[l]->sparse.get());
        b->ev_gemm_begin_ = b->ev_gemm_end_ = nullptr;
    }
    if (rc == SESSD_OK) rc = P->clearTables(stream);  // (the plugins leave theirs filled)
    if (rc != SESSD_OK) return P->recover(stream, rc);
    SESSD_HIP_TRY(hipStreamSynchronize(stream));
    for (int i = 0; i < n_seg; ++i)
        SESSD_HIP_TRY(hipEventElapsedTime(&segment_ms[i], P->events[i], P->events[i + 1]));
    if (max_segments > n_seg)  // optional extra slot: what an empty segment measures on this stream
        SESSD_HIP_TRY(hipEventElapsedTime(&segment_ms[n_seg], P->events[n_seg + 1], P->events[n_seg + 2]));
    *n_segments = n_seg;
    return SESSD_OK;
}

int sessd_pipeline_layer_stats(sessd_pipeline* h, int layer, sessd_stream_t stream_, int64_t* n_out,
                               int64_t* pairs) {
    if (!h || !n_out || !pairs) return fail(SESSD_E_INVALID, "pipeline_layer_stats: null argument");
    Pipeline* P = current(h);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (layer < -1 || layer >= (int)P->stages.size()) return fail(SESSD_E_INVALID, "pipeline_layer_stats: no layer %d", layer);
    SESSD_TRY(order_after_last_frame(h, stream));
    void* num = nullptr;
    void* ws = nullptr;
    SESSD_TRY(sessd_pipeline_layer_io(h, layer, nullptr, nullptr, &num, &ws, nullptr));  // (of the same replica)
    int32_t n = 0;
    SESSD_HIP_TRY(hipMemcpyAsync(&n, num, sizeof(n), hipMemcpyDeviceToHost, stream));
    SESSD_HIP_TRY(hipStreamSynchronize(stream));
    *n_out = n;
    *pairs = 0;
    if (layer < 0) return SESSD_OK;
    if (!P->stats.p) SESSD_TRY(P->stats.alloc(32 * sizeof(uint32_t)));
    ConvStage& st = *P->stages[layer];
    uint32_t* dev_num = static_cast<uint32_t*>(P->stats.p);
    const int K = st.spec.ksize[0] * st.spec.ksize[1] * st.spec.ksize[2];
    if (st.subm) SESSD_TRY(st.subm->countPairs(ws, dev_num, stream));
    else SESSD_TRY(st.sparse->countPairs(ws, dev_num, stream));
    uint32_t host[32] = {0};
    SESSD_HIP_TRY(hipMemcpyAsync(host, dev_num, K * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    SESSD_HIP_TRY(hipStreamSynchronize(stream));
    for (int k = 0; k < K; ++k) *pairs += host[k];
    return SESSD_OK;
}

size_t sessd_pipeline_device_bytes(const sessd_pipeline* h) {
    return h ? reinterpret_cast<const Pipeline*>(h)->device_bytes : 0;
}

int sessd_pipeline_num_launches(const sessd_pipeline* h) {
    if (!h) return -1;
    const Pipeline* P = reinterpret_cast<const Pipeline*>(h);
    if (!P->replicas.empty()) P = P->replicas[(size_t)P->last_replica].get();
    return P->captured.nodes;
}

void sessd_pipeline_destroy(sessd_pipeline* h) { delete reinterpret_cast<Pipeline*>(h); }

}  // extern "C"
