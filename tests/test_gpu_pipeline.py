"""GPU parity of the whole frame pipeline (voxelGenerator -> 14 conv layers with folded BN + ReLU ->
sparse2Dense) against oracle_frame, plus size-independent properties at the full benchmark size."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_util import (RTOL_FP16, RTOL_FP32, assert_end_to_end_close, assert_features_close, canonical, dev, layer_abs_sum,
                      points_input, to_np)
from sessd3d import api, backbone as B, ctypes_defs as D, frames as F

pytestmark = pytest.mark.gpu


def run_pipeline(pts, layers, W, max_points, max_voxels, **kw):
    pipe = api.Pipeline(layers, W, max_points, max_voxels, **kw)
    p, n = points_input(pts, max_points)
    dense = pipe.new_dense()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        pipe.enqueue(p, n, dense, stream)
    stream.synchronize()
    return pipe, dense, (p, n, stream)


def compare_with_oracle(pipe, dense, pts, layers, W, max_voxels, rtol_layer):
    ref = O.frame(pts, B.voxelgen_desc(max_voxels=max_voxels), layers, W, B.dense_desc())
    feat, coors, n = pipe.read_layer(-1)
    assert n == ref["counts"][0]
    for l, layer in enumerate(layers):
        fbuf = np.zeros((max_voxels, layer.cin), np.float32)
        fbuf[:n] = feat
        cbuf = np.zeros((max_voxels, 4), np.int32)
        cbuf[:n] = coors
        o_out, o_coors, o_n, _, _ = O.conv_layer(fbuf, cbuf, n, layer, W.w[l], W.scale[l], W.shift[l], max_voxels)
        terms = layer_abs_sum(fbuf, cbuf, n, layer, W.w[l], W.scale[l], W.shift[l], max_voxels)
        feat, g_coors, g_n = pipe.read_layer(l)
        assert g_n == o_n == ref["counts"][l + 1], layer.name
        assert np.array_equal(g_coors, o_coors[:o_n]), layer.name          # same numbering, row by row
        assert_features_close(feat, o_out[:o_n], rtol_layer, layer.name, abs_sum=terms[:o_n])
        coors, n = g_coors, g_n
    assert np.array_equal(coors, ref["coors"])
    a, b = canonical(coors, n, feat), canonical(ref["coors"], n, ref["feat"])
    assert np.array_equal(a[0], b[0])
    assert_end_to_end_close(a[1], b[1], False, "last layer features (end to end)")
    assert_end_to_end_close(to_np(dense).astype(np.float32), ref["dense"], False, "dense BEV tensor (end to end)")
    # the dense tensor is an exact scatter of the last layer's rows
    assert np.array_equal(to_np(dense).astype(np.float32), O.sparse2dense(feat, coors, n, B.DENSE_SIZE_XYZ))
    assert pipe.status() == ref["status"]
    return ref


@pytest.mark.parametrize("share,skip_pad", [(True, True), (False, False)])
def test_full_backbone_small_frame(share, skip_pad):
    pts = F.lidar_frame(5000, 11)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=5, w_std=0.05)
    pipe, dense, _ = run_pipeline(pts, layers, W, 8192, 16384, share_rulebooks=share, skip_pad_rows=skip_pad)
    compare_with_oracle(pipe, dense, pts, layers, W, 16384, RTOL_FP32)


@pytest.mark.parametrize("overlap", [False, True])
def test_pipeline_writes_the_zero_padded_dense_tensor(overlap):
    """dense_padding = the reference's ZeroPad2dPlugin (params.h:200-203: 1,1,1,1) folded into the last scatter:
    the padded tensor must equal the oracle's sparse2dense -> zero_pad2d of the same rows, and its interior
    the unpadded pipeline's output, bit for bit."""
    pts = F.lidar_frame(4000, 21)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=6, w_std=0.05)
    kw = dict(share_rulebooks=True, skip_pad_rows=True, overlap_streams=overlap, use_graph=overlap)
    plain, dense, _ = run_pipeline(pts, layers, W, 4096, 16384, **kw)
    pad = (1, 1, 1, 1)
    pipe, padded, (p, n, stream) = run_pipeline(pts, layers, W, 4096, 16384, dense_padding=pad, **kw)
    assert tuple(padded.shape) == (128, 202, 178)
    feat, coors, m = pipe.read_layer(len(layers) - 1)
    want = O.zero_pad2d(O.sparse2dense(feat, coors, m, B.DENSE_SIZE_XYZ), *pad)
    assert np.array_equal(to_np(padded), want)
    assert np.array_equal(to_np(padded)[:, 1:-1, 1:-1], to_np(dense))
    # a second enqueue into a dirty buffer restores the zero border
    padded.fill_(7.0)
    with torch.cuda.stream(stream):
        pipe.enqueue(p, n, padded, stream)
    stream.synchronize()
    assert np.array_equal(to_np(padded), want)


def test_capacity_binds_in_the_voxelizer_and_in_a_strided_layer():
    """One capacity for every tensor (as in the reference), small enough that the voxelizer drops cells and the
    first strided layer drops output sites.  The overlapped schedule -- where SubM layers probe the cell table
    the voxelizer / strided layer left behind, dropped cells included -- must agree with the single-stream run
    bit for bit, and both with the oracle."""
    pts = F.lidar_frame(6000, 13)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=9, w_std=0.05)
    cap = 3000
    ref = O.frame(pts, B.voxelgen_desc(max_voxels=cap), layers, W, B.dense_desc())
    assert ref["status"] & D.SESSD_STATUS_VOXEL_OVERFLOW and ref["counts"][0] == cap and ref["counts"][3] == cap
    plain, dense, _ = run_pipeline(pts, layers, W, 6000, cap, share_rulebooks=True, skip_pad_rows=True)
    fast, fdense, (p, n, stream) = run_pipeline(pts, layers, W, 6000, cap, share_rulebooks=True, skip_pad_rows=True,
                                                overlap_streams=True, use_graph=True)
    with torch.cuda.stream(stream):
        fast.enqueue(p, n, fdense, stream)                      # a replay of the captured graph
    stream.synchronize()
    assert np.array_equal(to_np(fdense), to_np(dense))
    for pipe in (plain, fast):
        assert pipe.status() == ref["status"]
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"])
        feat, coors, cnt = pipe.read_layer(len(layers) - 1)
        assert np.array_equal(coors, ref["coors"])
        assert_end_to_end_close(feat, ref["feat"], False, "last layer features with binding capacities")
    assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense tensor with binding capacities")


def test_overlapped_graph_schedule_with_reference_pad_rows():
    """Reference behaviour for rows past the active count (every output tensor is zero-filled, then BN + ReLU
    runs over all rows: rows >= n hold relu(shift)) under the overlapped schedule and its captured graph: dense
    tensor, active rows and pad rows must equal the single-stream run bit for bit, frame after frame."""
    pts = F.lidar_frame(3000, 17)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=12, w_std=0.05)
    mv = 8192
    plain, dense, _ = run_pipeline(pts, layers, W, 4096, mv, share_rulebooks=True, skip_pad_rows=False)
    fast, fdense, (p, n, stream) = run_pipeline(pts, layers, W, 4096, mv, share_rulebooks=True, skip_pad_rows=False,
                                                overlap_streams=True, use_graph=True)
    for _ in range(2):                                               # graph replays
        with torch.cuda.stream(stream):
            fast.enqueue(p, n, fdense, stream)
        stream.synchronize()
        assert np.array_equal(to_np(fdense), to_np(dense))
    assert fast.status() == plain.status() == 0
    for l in (0, 5, len(layers) - 1):
        rows = []
        for pipe in (plain, fast):
            f, _, _, _, ch = pipe.layer_io(l)
            full = np.zeros((mv, ch), np.float32)
            api._hip_d2h(full, f)
            rows.append((full, 0))
        assert np.array_equal(rows[0][0], rows[1][0]), layers[l].name
        cnt = plain.layer_count(l)
        want_pad = np.maximum(W.shift[l], 0.0).astype(np.float32)    # relu(0 * scale + shift)
        assert np.array_equal(rows[0][0][cnt:], np.broadcast_to(want_pad, (mv - cnt, len(want_pad)))), layers[l].name


@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
def test_tiny_frames_through_the_pipeline(dtype):
    """Frames of 0, 1, 7, 40 and 150 points through one pipeline (overlapped schedule, captured graph): the wide
    layers then see far fewer rows than they have tiles.  Site counts exact, dense tensor against the oracle."""
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=3, w_std=0.05)
    half = dtype == "fp16"
    if half:
        W = half_weights(W)
    mp, mv = 1024, 4096
    pipe = api.Pipeline(layers, W, mp, mv, feature_dtype=dtype, share_rulebooks=True, skip_pad_rows=True,
                        use_graph=True, overlap_streams=True)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    for npts in (150, 0, 1, 40, 7):
        pts = F.lidar_frame(npts, 100 + npts) if npts else np.zeros((0, 4), np.float32)
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc(), round_half=half)
        assert pipe.status() == ref["status"] == 0
        for l in range(-1, len(layers)):
            assert pipe.layer_count(l) == ref["counts"][l + 1], (npts, l)
        assert_end_to_end_close(to_np(dense).astype(np.float32), ref["dense"], half, "dense, %d points" % npts)


def test_full_backbone_config3_frame_and_graph_replay():
    """Benchmark configuration 3: the 20 000-point frame (~17 k voxels) through the reference's 14 conv layers.
    The eager enqueue and repeated replays of the captured graph must give identical bits."""
    pts = F.lidar_frame(20000, 0)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=1, w_std=0.05)
    pipe, dense, _ = run_pipeline(pts, layers, W, 20000, 60000, share_rulebooks=True, skip_pad_rows=True)
    ref = compare_with_oracle(pipe, dense, pts, layers, W, 60000, RTOL_FP32)
    assert 15000 < ref["counts"][0] < 19000
    eager = to_np(dense).copy()

    # two-stream schedule, eager: same bits as the single-stream run
    opipe, odense, _ = run_pipeline(pts, layers, W, 20000, 60000, share_rulebooks=True, skip_pad_rows=True,
                                    overlap_streams=True)
    assert np.array_equal(to_np(odense), eager), "two-stream schedule differs from the single-stream result"
    assert opipe.status() == 0

    gpipe = api.Pipeline(layers, W, 20000, 60000, share_rulebooks=True, skip_pad_rows=True, use_graph=True,
                         overlap_streams=True)
    p, n = points_input(pts, 20000)
    gd = gpipe.new_dense()
    stream = torch.cuda.Stream()
    for rep in range(3):
        gd.fill_(float(rep + 1))                        # eager work between replays
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            gpipe.enqueue(p, n, gd, stream)
        stream.synchronize()
        assert np.array_equal(to_np(gd), eager), "graph replay %d differs from the eager result" % rep
    assert gpipe.num_launches() > 0
    # a different frame in the same buffers: the replayed graph reads the new data
    pts2 = F.lidar_frame(18000, 1)
    p2, n2 = points_input(pts2, 20000)
    p.copy_(p2)
    n.copy_(n2)
    with torch.cuda.stream(stream):
        gpipe.enqueue(p, n, gd, stream)
    stream.synchronize()
    ref2 = O.frame(pts2, B.voxelgen_desc(max_voxels=60000), layers, W, B.dense_desc())
    assert_end_to_end_close(to_np(gd), ref2["dense"], False, "graph replay on a new frame")


def half_weights(W):
    """The FP16 configurations store weights in half: round once, hand the same values to both sides."""
    return B.Weights([O.round_to_half(w) for w in W.w], W.scale, W.shift)


def test_fp16_backbone_against_half_rounding_oracle():
    """FP16 features/weights with FP32 accumulate through all 14 layers.  The oracle keeps FP32 arithmetic
    but rounds every layer's output to half, as the FP16 pipeline stores it.  Sites are bit-exact; features
    within 1e-2 relative per layer (oracle fed the GPU's rows) and end to end."""
    pts = F.lidar_frame(12000, 21)
    layers = B.reference_layers()
    W = half_weights(B.random_weights(layers, seed=9, w_std=0.05))
    mv = 40000
    pipe, dense, _ = run_pipeline(pts, layers, W, 12000, mv, feature_dtype="fp16", share_rulebooks=True,
                                  skip_pad_rows=True, overlap_streams=True)
    assert dense.dtype == torch.float16
    ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc(), round_half=True)
    feat, coors, n = pipe.read_layer(-1)
    for l, layer in enumerate(layers):
        fbuf = np.zeros((mv, layer.cin), np.float32)
        fbuf[:n] = feat
        cbuf = np.zeros((mv, 4), np.int32)
        cbuf[:n] = coors
        o_out, o_coors, o_n, _, _ = O.conv_layer(fbuf, cbuf, n, layer, W.w[l], W.scale[l], W.shift[l], mv)
        terms = layer_abs_sum(fbuf, cbuf, n, layer, W.w[l], W.scale[l], W.shift[l], mv)
        feat, g_coors, g_n = pipe.read_layer(l)
        assert g_n == o_n == ref["counts"][l + 1] and np.array_equal(g_coors, o_coors[:o_n]), layer.name
        assert_features_close(feat, O.round_to_half(o_out[:o_n]), RTOL_FP16, "fp16 " + layer.name, abs_sum=terms[:o_n], half=True)
        coors, n = g_coors, g_n
    assert np.array_equal(coors, ref["coors"])
    # end to end a half-rounding that falls the other way in an early layer is carried on by the layers after
    # it (gpu_util.END_TO_END_RMS / END_TO_END_MAX say how far, measured); in the L2 norm the error must stay within 1e-2
    assert_end_to_end_close(feat, ref["feat"], True, "fp16 last layer (end to end)")
    d = to_np(dense.float())
    assert_end_to_end_close(d, ref["dense"], True, "fp16 dense (end to end)")
    assert np.linalg.norm(d - ref["dense"]) <= RTOL_FP16 * np.linalg.norm(ref["dense"])
    assert pipe.status() == ref["status"]


def test_properties_at_full_size():
    """Size-independent checks on a frame too large to push through the CPU oracle quickly:
    determinism, active-site bookkeeping and dense/sparse consistency."""
    pts = F.lidar_frame(60000, 7)
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=2, w_std=0.05)
    pipe, dense, (p, n, stream) = run_pipeline(pts, layers, W, 60000, 60000, skip_pad_rows=True)
    first = to_np(dense).copy()
    with torch.cuda.stream(stream):
        pipe.enqueue(p, n, dense, stream)
    stream.synchronize()
    assert np.array_equal(to_np(dense), first)                     # run-to-run bit identical
    feat, coors, cnt = pipe.read_layer(len(layers) - 1)
    assert len(np.unique(coors[:, 1:] @ np.array([200 * 176, 176, 1]))) == cnt     # unique sites
    assert coors[:, 1].max() < 2 and coors[:, 2].max() < 200 and coors[:, 3].max() < 176 and coors.min() >= 0
    back = first.reshape(64, 2, 200, 176)[:, coors[:, 1], coors[:, 2], coors[:, 3]].T
    assert np.array_equal(back, feat)                               # dense holds exactly the sparse rows
    assert np.count_nonzero(first) == np.count_nonzero(feat)
    # voxelizer output is independent of everything downstream: compare with the oracle's voxelizer
    vfeat, vcoors, vn = pipe.read_layer(-1)
    o = O.voxelize(pts, B.POINT_CLOUD_RANGE, B.VOXEL_SIZE, 5, 60000)
    assert vn == o[2] and np.array_equal(vcoors, o[1][:vn]) and np.array_equal(vfeat.view(np.uint32), o[0][:vn].view(np.uint32))


def test_stress_configuration_properties():
    """Benchmark configuration 5: 150 000 points over 360 degrees (cropped to range), voxel cap 60 000, doubled
    channel widths, FP16 features.  Too heavy for the scalar oracle's conv layers, so: the voxelizer part
    is compared with the oracle exactly (the cap binds -> overflow flag), the rest through properties."""
    pts = F.lidar_frame(150000, 5, full_circle=True)
    layers = B.reference_layers(width_mult=2)
    W = half_weights(B.random_weights(layers, seed=4, w_std=0.03))
    pipe, dense, (p, n, stream) = run_pipeline(pts, layers, W, 150000, 200000, feature_dtype="fp16",
                                               skip_pad_rows=True, overlap_streams=True, use_graph=True,
                                               voxel_cap=60000)
    assert tuple(dense.shape) == (256, 200, 176)
    first = to_np(dense).copy()
    for _ in range(2):                                               # graph replays are bit identical
        with torch.cuda.stream(stream):
            pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        assert np.array_equal(to_np(dense), first)
    vfeat, vcoors, vn = pipe.read_layer(-1)
    o = O.voxelize(pts, B.POINT_CLOUD_RANGE, B.VOXEL_SIZE, 5, 60000)
    assert vn == o[2] == 60000 and o[4] & D.SESSD_STATUS_VOXEL_OVERFLOW
    assert np.array_equal(vcoors, o[1][:vn]) and np.array_equal(vfeat.view(np.uint32), o[0][:vn].view(np.uint32))
    assert pipe.status() & D.SESSD_STATUS_VOXEL_OVERFLOW
    counts = [pipe.layer_stats(l)[0] for l in range(len(layers))]
    assert counts[0] == counts[1] == 60000 and max(counts) <= 200000
    assert counts[2] > 60000                                         # the first strided layer grows the set
    feat, coors, cnt = pipe.read_layer(len(layers) - 1)
    assert cnt == counts[-1] and len(np.unique(coors[:, 1:] @ np.array([200 * 176, 176, 1]))) == cnt
    back = first.reshape(128, 2, 200, 176)[:, coors[:, 1], coors[:, 2], coors[:, 3]].T
    assert np.array_equal(back.astype(np.float32), feat)
    assert np.isfinite(first.astype(np.float32)).all()


def test_frames_in_flight_give_the_bits_of_one_frame_at_a_time():
    """frames_in_flight = 3: three replicas of the pipeline, successive frames on successive replicas (submit / join).
    A sequence of DIFFERENT frames, submitted ahead of their joins, must give exactly the dense tensors, statuses and
    layer counts of the one-frame-at-a-time pipeline; enqueue() on the same object is submit + join."""
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=8, w_std=0.05)
    mp, mv, R = 8192, 16384, 3
    kw = dict(share_rulebooks=True, skip_pad_rows=True, use_graph=True, overlap_streams=True)
    one = api.Pipeline(layers, W, mp, mv, **kw)
    many = api.Pipeline(layers, W, mp, mv, frames_in_flight=R, **kw)
    frames = [F.lidar_frame(npts, 40 + i) for i, npts in enumerate((6000, 2500, 8000, 50, 7000, 3000, 6500))]
    stream = torch.cuda.Stream()
    want, counts = [], []
    p, n = points_input(frames[0], mp)
    dense = one.new_dense()
    for pts in frames:
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            one.enqueue(p, n, dense, stream)
        stream.synchronize()
        want.append(to_np(dense).copy())
        counts.append([one.layer_count(l) for l in range(-1, len(layers))])
    # every frame in flight has its own input and output buffers (they must stay untouched until its join)
    ins = [points_input(pts, mp) for pts in frames]
    outs = [many.new_dense() for _ in frames]
    tickets = []
    with torch.cuda.stream(stream):
        for i in range(len(frames)):
            tickets.append(many.submit(ins[i][0], ins[i][1], outs[i], stream))
            if i >= R - 1:
                many.join(tickets[i - (R - 1)], stream)
        for t in tickets[-(R - 1):]:
            many.join(t, stream)
    stream.synchronize()
    assert tickets == list(range(len(frames)))
    for i in range(len(frames)):
        assert np.array_equal(to_np(outs[i]), want[i]), "frame %d differs with frames in flight" % i
    assert [many.layer_count(l) for l in range(-1, len(layers))] == counts[-1]        # queries: the frame submitted last
    assert many.status() == one.status() == 0 and many.num_launches() == one.num_launches()
    # enqueue = submit + join, again and again into the same buffers
    for rep in range(4):
        outs[0].fill_(3.0)
        with torch.cuda.stream(stream):
            many.enqueue(ins[2][0], ins[2][1], outs[0], stream)
        stream.synchronize()
        assert np.array_equal(to_np(outs[0]), want[2]), rep
    # host-driven loop: the inputs are resident (synchronised above), nothing is ordered after a stream, the host
    # blocks on the oldest frame in flight
    for o in outs:
        o.fill_(5.0)
    torch.cuda.synchronize()
    tickets = []
    for i in range(len(frames)):
        tickets.append(many.submit(ins[i][0], ins[i][1], outs[i], api.STREAM_NONE))
        if i >= R - 1:
            many.wait(tickets[i - (R - 1)])
            j = i - (R - 1)
            assert np.array_equal(to_np(outs[j]), want[j]), "frame %d differs after a host-side wait" % j
    for t in tickets[-(R - 1):]:
        many.wait(t)
    for i in range(len(frames)):
        assert np.array_equal(to_np(outs[i]), want[i]), i
    with pytest.raises(api.SessdError, match="no frame with ticket"):
        many.join(10 ** 6, stream)
    with pytest.raises(api.SessdError, match="no frame with ticket"):
        many.wait(10 ** 6)
    with pytest.raises(api.SessdError, match="STREAM_NONE needs frames_in_flight"):
        one.submit(p, n, dense, api.STREAM_NONE)
    with pytest.raises(api.SessdError, match="runs its frames on the caller's stream"):
        one.wait(one.submit(p, n, dense, stream))
    stream.synchronize()


def test_fp16_stack_ending_in_a_3x3x3_layer_scatters_from_its_own_kernel():
    """A stack whose LAST layer is a 3x3x3 FP16 layer of 32 channels: that layer's kernel (conv_tall.hip) also writes
    the dense tensor, in both schedules.  Dense tensor, sites and status against the oracle, and each schedule's tensor
    equal to a scatter of its last layer's rows and to the plugin's cell-major pass over them bit for bit."""
    S, P = D.SESSD_LAYER_SUBM, D.SESSD_LAYER_SPARSE
    layers = [B.Layer("subm0", S, 4, 32, (1408, 1600, 41), (3, 3, 3), (1, 1, 1), (1, 1, 1)),
              B.Layer("sparse1", P, 32, 64, (704, 800, 21), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("sparse2", P, 64, 64, (352, 400, 11), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("sparse3", P, 64, 32, (176, 200, 5), (3, 3, 3), (2, 2, 2), (0, 1, 1)),
              B.Layer("subm4", S, 32, 32, (176, 200, 5), (3, 3, 3), (1, 1, 1), (1, 1, 1))]
    W = half_weights(B.random_weights(layers, seed=12, w_std=0.08))
    pts = F.lidar_frame(9000, 33)
    mv = 16384
    dsize = (176, 200, 5)
    kw = dict(feature_dtype="fp16", share_rulebooks=True, skip_pad_rows=True, dense_size_xyz=dsize, dense_padding=(1, 1, 1, 1))
    fused, d_fused, _ = run_pipeline(pts, layers, W, 9000, mv, use_graph=True, overlap_streams=True, **kw)
    plain, d_plain, _ = run_pipeline(pts, layers, W, 9000, mv, use_graph=False, overlap_streams=False, **kw)
    ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc(dsize, 32), round_half=True)
    want = np.pad(ref["dense"], ((0, 0), (1, 1), (1, 1)))
    assert fused.status() == plain.status() == ref["status"] == 0
    assert [fused.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"])
    assert np.array_equal(fused.read_layer(len(layers) - 1)[1], ref["coors"])
    assert_end_to_end_close(to_np(d_fused).astype(np.float32), want, True, "dense from conv_tall")
    assert torch.equal(d_fused, d_plain)
    for pipe, d in ((fused, d_fused), (plain, d_plain)):
        feat, coors, m = pipe.read_layer(len(layers) - 1)
        assert np.array_equal(to_np(d).astype(np.float32), O.zero_pad2d(O.sparse2dense(feat, coors, m, dsize), 1, 1, 1, 1))
    rows, cbuf = np.zeros((mv, 32), np.float32), np.zeros((mv, 4), np.int32)
    rows[:m], cbuf[:m] = feat, coors
    s2d = api.Sparse2Dense(dsize, 32, padding=(1, 1, 1, 1))
    as_plugin = s2d(dev(rows, torch.float16), dev(cbuf), dev(np.array([m], np.int32)))
    torch.cuda.synchronize()
    assert torch.equal(as_plugin.view(torch.int16).reshape(d_plain.shape), d_plain.view(torch.int16))


@pytest.mark.parametrize("overlap", [True, False])
@pytest.mark.parametrize("full_resolution", [False, True])
def test_cell_tables_kept_between_frames_carry_nothing_over(full_resolution, overlap):
    """The pipeline keeps its dense cell tables from frame to frame and empties them row by row.  Frames of different
    sizes through one pipeline, an empty one and a plugin-by-plugin run (enqueue_timed, which overwrites the rows the
    tables are emptied by) between them, each against the oracle.  full_resolution: a strided layer of stride 1 whose
    output grid is too large for a dense table, so that its hash is cleared instead."""
    layers = B.reference_layers()
    if full_resolution:
        at = next(i for i, l in enumerate(layers) if l.name == "sparse6")
        wide = B.Layer("sparse5", D.SESSD_LAYER_SPARSE, 16, 16, layers[0].out_shape, (3, 3, 3), (1, 1, 1), (1, 1, 1))
        layers = layers[:at] + [wide] + layers[at:]
    W = B.random_weights(layers, seed=11, w_std=0.05)
    mp, mv = 1024, 40000
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, skip_pad_rows=overlap, use_graph=True, overlap_streams=overlap)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    for step, npts in enumerate((400, 1000, 0, 250, 250)):
        pts = F.lidar_frame(npts, 60 + step) if npts else np.zeros((0, 4), np.float32)
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            if step == 3:
                pipe.enqueue_timed(p, n, dense, stream)
            else:
                pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc())
        assert pipe.status() == ref["status"] == 0
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), npts
        assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), npts
        assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)


@pytest.mark.parametrize("max_pts", [1, 2, 5, 6, 9])
def test_voxelizer_keeps_the_first_points_of_crowded_cells(max_pts):
    """More points per cell than are averaged, at point counts around a block: the later points of a cell go through a
    chain of places behind its first one, of which four are read ahead."""
    rng = np.random.default_rng(max_pts)
    for npts in (1, 255, 257, 3000):
        pts = np.zeros((npts, 4), np.float32)
        pts[:, :3] = np.array([1.0, -2.0, -1.0]) + rng.uniform(0, 0.25, (npts, 3))
        pts[:, 3] = rng.uniform(0, 1, npts)
        vg = api.VoxelGenerator(max_voxels=4096, max_num_points_per_voxel=max_pts)
        voxels, coors, num = vg(*points_input(pts, npts + 5))
        torch.cuda.synchronize()
        ref = O.voxelize(pts, B.POINT_CLOUD_RANGE, B.VOXEL_SIZE, max_pts, 4096)
        assert int(num[0]) == ref[2]
        assert np.array_equal(to_np(coors)[:ref[2]], ref[1][:ref[2]])
        assert np.array_equal(to_np(voxels)[:ref[2]].view(np.uint32), ref[0][:ref[2]].view(np.uint32))


@pytest.mark.parametrize("overlap", [True, False])
def test_a_frame_in_the_callers_own_graph_finds_its_tables_empty(overlap):
    """The first frame of a pipeline is captured by the caller and launched only after a frame of another size has run
    directly; later replays follow direct frames and a plugin-by-plugin run.  No frame may depend on clears that another
    one was meant to make."""
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=12, w_std=0.05)
    mp, mv = 1024, 20000
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, skip_pad_rows=True, overlap_streams=overlap)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        pipe.enqueue(p, n, dense, stream)
    for step, how in enumerate(("direct", "graph", "timed", "graph", "direct", "graph", "graph")):
        npts = (700, 300, 1000, 500, 0, 900, 200)[step]
        pts = F.lidar_frame(npts, 80 + step) if npts else np.zeros((0, 4), np.float32)
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            if how == "graph":
                graph.replay()
            elif how == "timed":
                pipe.enqueue_timed(p, n, dense, stream)
            else:
                pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc())
        assert pipe.status() == ref["status"] == 0
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), (step, how)
        assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), (step, how)
        assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)


@pytest.mark.parametrize("schedule", [{}, dict(overlap_streams=True), dict(overlap_streams=True, use_graph=True)], ids=["one", "two", "graph"])
def test_dozens_of_strided_layers(schedule):
    """More strided layers than the clears of one launch can hold, on one stream and with the coordinate branch on another; two frames,
    the second smaller."""
    layers = B.reference_layers()
    grid = layers[-2].out_shape
    layers[-1:-1] = [B.Layer("s%d" % i, D.SESSD_LAYER_SPARSE, 64, 64, grid, (3, 1, 1), (1, 1, 1), (1, 0, 0)) for i in range(46)]
    W = B.random_weights(layers, seed=13, w_std=0.05)
    mp, mv = 512, 8000
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, **schedule)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    for step, npts in enumerate((400, 250)):
        pts = F.lidar_frame(npts, 90 + step)
        p, n = points_input(pts, mp)
        torch.cuda.synchronize()
        pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc())
        assert pipe.status() == ref["status"] == 0
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"])
        assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"])


class _Words:
    """`n` 32-bit words of device memory that the library owns, for torch.as_tensor."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), version=2)


@pytest.mark.parametrize("coordinate,count", [(0, None), (3, 0), (1 << 30, 1 << 30), (-1, -1)])
def test_writing_to_a_layers_tensors_after_a_frame_leaves_the_next_one_alone(coordinate, count):
    """sessd_pipeline_layer_io hands out the tensors of a finished frame.  What a caller does to them must not reach the
    next frame: the cells that the kept tables are emptied by are listed in memory of the pipeline's own."""
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=14, w_std=0.05)
    mp, mv = 1024, 20000
    overlap = coordinate >= 0
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, skip_pad_rows=True, use_graph=overlap, overlap_streams=overlap)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    for step, npts in enumerate((900, 1000, 300)):
        pts = F.lidar_frame(npts, 110 + step)
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc())
        assert pipe.status() == ref["status"] == 0
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), step
        assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), step
        assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)
        for l in range(-1, len(layers)):
            _, coors, num, _, _ = pipe.layer_io(l)
            torch.as_tensor(_Words(coors, mv * 4), device="cuda:0").fill_(coordinate)
            if count is not None:
                torch.as_tensor(_Words(num, 1), device="cuda:0").fill_(count)
        torch.cuda.synchronize()


def _leave_an_error_pending():
    """What a failed HIP call of the application's own leaves behind: the library's next launch check meets it, after the
    launch itself has gone through."""
    with open("/proc/self/maps") as f:
        path = next(l.split()[-1] for l in f if "libamdhip64" in l)
    assert ctypes.CDLL(path).hipSetDevice(12345) != 0


@pytest.mark.parametrize("overlap", [True, False])
def test_a_frame_in_the_callers_own_graph_survives_a_call_that_failed(overlap):
    """An enqueue that fails after its first launch leaves the voxelizer's table filled.  The graph that the caller
    captured before holds no clear; the failed call has to leave the tables as it found them."""
    layers = B.reference_layers()
    W = B.random_weights(layers, seed=15, w_std=0.05)
    mp, mv = 1024, 20000
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, skip_pad_rows=True, overlap_streams=overlap)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        pipe.enqueue(p, n, dense, stream)
    for step, how in enumerate(("graph", "failed", "graph", "graph", "timed, failed", "graph", "direct", "graph")):
        pts = F.lidar_frame((700, 900, 400, 1000, 800, 300, 600, 500)[step], 130 + step)
        hp, hn = points_input(pts, mp)
        with torch.cuda.stream(stream):
            p.copy_(hp)
            n.copy_(hn)
            if "failed" in how:
                stream.synchronize()
                _leave_an_error_pending()
                with pytest.raises(api.SessdError):
                    (pipe.enqueue_timed if "timed" in how else pipe.enqueue)(p, n, dense, stream)
            elif how == "graph":
                graph.replay()
            else:
                pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        if "failed" in how:
            continue
        ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc())
        assert pipe.status() == ref["status"] == 0
        assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), (step, how)
        assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), (step, how)
        assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)


def test_a_voxel_grid_too_large_for_a_kept_table(monkeypatch):
    """Voxels of half the size: neither the voxelizer's table nor the first strided layer's has room for a word per cell,
    so every frame clears their hashes -- as it does where the memory for kept tables is short.  The frames shrink and
    grow, so that what one leaves behind would reach the next."""
    size = (0.025, 0.025, 0.1)
    desc = lambda cap, pts=5: B.voxelgen_desc(cap, pts, B.POINT_CLOUD_RANGE, size)  # noqa: E731
    S, P = D.SESSD_LAYER_SUBM, D.SESSD_LAYER_SPARSE
    layers = [B.Layer("subm0", S, 4, 16, (2816, 3200, 41), (3, 3, 3), (1, 1, 1), (1, 1, 1)),
              B.Layer("sparse1", P, 16, 32, (1408, 1600, 21), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("subm2", S, 32, 32, (1408, 1600, 21), (3, 3, 3), (1, 1, 1), (1, 1, 1)),
              B.Layer("sparse3", P, 32, 64, (704, 800, 11), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("sparse4", P, 64, 64, (352, 400, 5), (3, 3, 3), (2, 2, 2), (0, 1, 1))]
    W = B.random_weights(layers, seed=16, w_std=0.05)
    mp, mv, dsize = 4096, 20000, (352, 400, 5)
    with monkeypatch.context() as m:
        original = B.voxelgen_desc
        m.setattr(api.B, "voxelgen_desc", lambda cap, pts=5: original(cap, pts, B.POINT_CLOUD_RANGE, size))
        pipes = [api.Pipeline(layers, W, mp, mv, dense_size_xyz=dsize, share_rulebooks=True, skip_pad_rows=True, use_graph=o,
                              overlap_streams=o) for o in (True, False)]
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    stream = torch.cuda.Stream()
    for step, npts in enumerate((3000, 600, 0, 4000, 1200)):
        pts = F.lidar_frame(npts, 150 + step) if npts else np.zeros((0, 4), np.float32)
        hp, hn = points_input(pts, mp)
        p.copy_(hp)
        n.copy_(hn)
        torch.cuda.synchronize()
        ref = O.frame(pts, desc(mv), layers, W, B.dense_desc(dsize, 64))
        for pipe in pipes:
            dense = pipe.new_dense()
            torch.cuda.synchronize()
            pipe.enqueue(p, n, dense, stream)
            stream.synchronize()
            assert pipe.status() == ref["status"] == 0
            assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), step
            assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), step
            assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)


@pytest.mark.parametrize("overlap", [True, False])
def test_more_points_than_the_numbering_reads_one_by_one(overlap):
    """A points tensor of more than 1 048 576 rows: the pass that numbers voxels goes by sums over 64 blocks' counts.  Three
    frames, the second small."""
    S, P = D.SESSD_LAYER_SUBM, D.SESSD_LAYER_SPARSE
    layers = [B.Layer("subm0", S, 4, 16, (1408, 1600, 41), (3, 3, 3), (1, 1, 1), (1, 1, 1)),
              B.Layer("sparse1", P, 16, 16, (704, 800, 21), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("sparse2", P, 16, 16, (352, 400, 11), (3, 3, 3), (2, 2, 2), (1, 1, 1)),
              B.Layer("sparse3", P, 16, 16, (176, 200, 5), (3, 3, 3), (2, 2, 2), (0, 1, 1)),
              B.Layer("sparse4", P, 16, 16, (176, 200, 2), (3, 1, 1), (2, 1, 1), (0, 0, 0))]
    W = B.random_weights(layers, seed=17, w_std=0.1)
    mp, mv = 1500000, 280000
    pipe = api.Pipeline(layers, W, mp, mv, share_rulebooks=True, skip_pad_rows=True, use_graph=overlap, overlap_streams=overlap)
    p, n = points_input(np.zeros((0, 4), np.float32), mp)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    O.set_threads(16)
    try:
        for step, npts in enumerate((mp, 5000, 1048577)):
            pts = np.concatenate([F.lidar_frame(-(-npts // 4), 170 + 4 * step + i, full_circle=i > 1) for i in range(4)])[:npts]
            hp, hn = points_input(pts, mp)
            with torch.cuda.stream(stream):
                p.copy_(hp)
                n.copy_(hn)
                pipe.enqueue(p, n, dense, stream)
            stream.synchronize()
            ref = O.frame(pts, B.voxelgen_desc(max_voxels=mv), layers, W, B.dense_desc(B.DENSE_SIZE_XYZ, 16))
            assert pipe.status() == ref["status"]
            assert [pipe.layer_count(l) for l in range(-1, len(layers))] == list(ref["counts"]), step
            vox = O.voxelize(pts, B.POINT_CLOUD_RANGE, B.VOXEL_SIZE, 5, mv)
            feat, coors, cnt = pipe.read_layer(-1)
            assert np.array_equal(coors, vox[1][:cnt]) and np.array_equal(feat.view(np.uint32), vox[0][:cnt].view(np.uint32))
            assert np.array_equal(pipe.read_layer(len(layers) - 1)[1], ref["coors"]), step
            assert_end_to_end_close(to_np(dense), ref["dense"], False, "dense, step %d" % step)
    finally:
        O.set_threads(1)


@pytest.mark.parametrize("width", [1, 2])
@pytest.mark.parametrize("schedule", [{}, dict(overlap_streams=True, use_graph=True, skip_pad_rows=True)], ids=["direct", "graph"])
def test_frame_of_very_small_features_through_the_split_products(width, schedule):
    """The first layer scales its features to 2^-108 and below, the last one back: rows whose elements do not fit their BF16 parts
    in every layer from 32 channels up, the last one with its scatter into the dense tensor among them.  Against the VALU kernels,
    within the whole-frame bound."""
    pts = F.lidar_frame(3000, 5)
    layers = B.reference_layers(width_mult=width)
    W = B.random_weights(layers, seed=9, w_std=0.05, bn=False)
    W.scale[0] *= np.float32(2.0 ** -108)
    W.scale[-1] *= np.float32(2.0 ** 108)
    kw = dict(share_rulebooks=True, **schedule)
    fast, a, _ = run_pipeline(pts, layers, W, 3000, 20000, **kw)
    slow, b, _ = run_pipeline(pts, layers, W, 3000, 20000, force_valu=True, **kw)
    inside = fast.read_layer(len(layers) - 3)[0]
    assert 0 < np.abs(inside).max() < 2.0 ** -90 and (np.abs(inside[inside != 0]) < 2.0 ** -110).mean() > 0.05
    a, b = to_np(a), to_np(b)
    assert np.isfinite(a).all() and a.any()
    assert_end_to_end_close(a, b, False, "very small features, MFMA vs VALU")
