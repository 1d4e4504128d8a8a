"""GPU parity: every plugin of libsessd3d, called through the C-ABI, against the CPU oracle on the same
seeded inputs.  Integer results (voxel coordinates, active sites, rulebooks, counts) must be
bit-exact, after canonical sort where the numbering is free; FP32 features within 1e-4 relative."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_util import (DEV, RTOL_FP16, RTOL_FP32, abs_sum_of, assert_features_close, canonical, dev, points_input, to_np)
from sessd3d import api, backbone as B, ctypes_defs as D, frames as F

pytestmark = pytest.mark.gpu

RANGE, VSIZE = B.POINT_CLOUD_RANGE, B.VOXEL_SIZE


def run_voxelgen(pts, max_points, max_voxels, max_pts=5):
    vg = api.VoxelGenerator(max_voxels=max_voxels, max_num_points_per_voxel=max_pts)
    p, n = points_input(pts, max_points)
    vox, coors, num = vg(p, n)
    torch.cuda.synchronize()
    return to_np(vox), to_np(coors), int(to_np(num)[0]), vg.status()


def check_voxelgen(pts, max_points, max_voxels, max_pts=5):
    vox, coors, n, st = run_voxelgen(pts, max_points, max_voxels, max_pts)
    o_vox, o_coors, o_n, _, o_st = O.voxelize(pts[:max_points], RANGE, VSIZE, max_pts, max_voxels)
    assert n == o_n
    assert st == o_st
    # same numbering (first appearance) -> comparable row by row, and again after canonical sort
    assert np.array_equal(coors, o_coors)
    assert np.array_equal(vox.view(np.uint32), o_vox.view(np.uint32))      # bit-exact means
    a = canonical(coors, n, vox)
    b = canonical(o_coors, o_n, o_vox)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    return n


@pytest.mark.parametrize("seed", [0, 1])
def test_voxelgen_config2(seed):
    """Benchmark configuration 2: 20 000 points, voxel 0.05x0.05x0.1, <= 5 points/voxel, cap 20 000."""
    pts = F.lidar_frame(20000, seed)
    n = check_voxelgen(pts, 20000, 20000)
    assert 14000 < n <= 20000


def test_voxelgen_reference_shapes_and_padding():
    """MAX_POINTS 80000 / MAX_VOXELS 60000 as in params.h; rows past points_size are ignored even if
    they hold in-range garbage."""
    pts = F.lidar_frame(20000, 2)
    vg = api.VoxelGenerator(max_voxels=60000)
    buf = np.tile(pts[:100], (800, 1)).astype(np.float32)      # 80000 rows of valid-looking points
    buf[:20000] = pts
    vox, coors, num = vg(dev(buf), dev(np.array([20000], np.int32)))
    torch.cuda.synchronize()
    o = O.voxelize(pts, RANGE, VSIZE, 5, 60000)
    assert int(to_np(num)[0]) == o[2]
    assert np.array_equal(to_np(coors), o[1]) and np.array_equal(to_np(vox).view(np.uint32), o[0].view(np.uint32))
    assert vg.status() == 0


@pytest.mark.parametrize("npts", [1048476, 1048477, 1048576 + 16384, 1300001])
def test_voxelgen_with_more_points_than_its_last_pass_reads_one_by_one(npts):
    """Beyond 1 048 576 rows of points the pass that numbers voxels goes by sums over 64 blocks of 256 points.  A second call
    on the same workspace with a third of the points, one that ends with a sum, and an empty one."""
    pts = np.concatenate([F.lidar_frame(-(-npts // 3), s, full_circle=True) for s in (41, 42, 43)])[:npts]
    vg = api.VoxelGenerator(max_voxels=npts)
    p, size = points_input(pts, npts + 100)
    for n in (npts, npts // 3, 4 * 16384, 4 * 16384 + 1, 0):
        size.fill_(n)
        voxels, coors, num = vg(p, size)
        torch.cuda.synchronize()
        ref = O.voxelize(pts[:n], RANGE, VSIZE, 5, npts)
        assert int(num[0]) == ref[2] and vg.status() == ref[4]
        assert np.array_equal(to_np(coors)[:ref[2]], ref[1][:ref[2]])
        assert np.array_equal(to_np(voxels)[:ref[2]].view(np.uint32), ref[0][:ref[2]].view(np.uint32))


def test_voxelgen_crowded_voxels_and_shuffled_order():
    rng = np.random.default_rng(3)
    pts = F.lidar_frame(12000, 3)
    extra = pts[rng.integers(0, len(pts), 6000)] + rng.normal(0, 0.004, (6000, 4)).astype(np.float32)
    pts = np.concatenate([pts, extra.astype(np.float32)])[rng.permutation(18000)]
    check_voxelgen(pts, 18000, 20000)
    check_voxelgen(pts, 18000, 20000, max_pts=3)
    check_voxelgen(pts, 18000, 20000, max_pts=8)


def test_voxelgen_cap_overflow_and_edges():
    pts = F.lidar_frame(20000, 4)
    check_voxelgen(pts, 20000, 5000)                 # cap binds: first 5000 cells kept, flag raised
    vox, coors, n, st = run_voxelgen(pts, 20000, 5000)
    assert n == 5000 and st & D.SESSD_STATUS_VOXEL_OVERFLOW
    check_voxelgen(pts[:0], 1024, 1000)              # empty cloud
    check_voxelgen(pts[:1], 1024, 1000)
    # points_size larger than the tensor: clamped to max_points
    vox, coors, n, st = run_voxelgen(pts, 4096, 20000)
    assert n == O.voxelize(pts[:4096], RANGE, VSIZE, 5, 20000)[2]
    f = np.float32
    below = lambda v: np.nextafter(f(v), f(-np.inf))   # noqa: E731
    edge = np.array([[0.0, -40.0, -3.0, 0.1], [70.4, 0.0, 0.0, 0.2], [10.0, 40.0, 0.0, 0.3], [10.0, 0.0, 1.0, 0.4],
                     [10.0, 0.0, below(1.0), 0.5], [10.0, below(40.0), 0.0, 0.6], [below(70.4), 0.0, 0.0, 0.7],
                     [-0.0, 0.0, 0.0, 0.8], [np.nan, 0.0, 0.0, 0.9], [np.inf, 0.0, 0.0, 1.0]], np.float32)
    assert check_voxelgen(edge, 64, 100) == 3


def test_voxelgen_five_point_features():
    pts = F.lidar_frame(8000, 5)
    pts5 = np.concatenate([pts, np.full((8000, 1), 7.0, np.float32)], axis=1)
    check_voxelgen(pts5, 8192, 20000)


def run_subm(coors_np, n, feat_np, w, grid_zyx, max_voxels, scale=None, shift=None, relu=False):
    conv = api.SubmConv3d(w.shape[1], w.shape[2], grid_zyx[::-1], w, max_voxels)
    if scale is not None or relu:
        conv.set_epilogue(scale, shift, relu)
    cbuf = np.zeros((max_voxels, 4), np.int32)
    cbuf[:n] = coors_np[:n]
    fbuf = np.zeros((max_voxels, w.shape[1]), np.float32)
    fbuf[:n] = feat_np[:n]
    out = conv(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    pairs, num = conv.export_rulebook()
    torch.cuda.synchronize()
    return conv, to_np(out), to_np(pairs), to_np(num).astype(np.uint32), cbuf


def test_subm_config1_rulebook_and_features():
    """Benchmark configuration 1: one SubMConv3d 4->16 on 2000 uniform voxels in 41x160x140."""
    grid = (41, 160, 140)
    n, mv = 2000, 2000
    rng = np.random.default_rng(0)
    coors = F.random_active_voxels(n, grid, 0)
    feat = rng.uniform(0, 1, (n, 4)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, 4, 16)).astype(np.float32)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv)
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    assert np.array_equal(num, o_num)
    assert np.array_equal(O.canonical_rulebook(pairs, num, cbuf, cbuf), O.canonical_rulebook(o_pairs, o_num, coors, coors))
    o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
    assert_features_close(out, o_out, RTOL_FP32, "subm config 1")
    assert conv.status() == 0


@pytest.mark.parametrize("n,mv,ksize,cin,cout", [(0, 1, 3, 4, 16), (1, 1, 3, 4, 16), (64, 64, 3, 4, 16), (65, 70, 3, 64, 64), (1024, 1025, 3, 4, 16),
                                                 (2047, 2048, 3, 64, 64), (2049, 2049, 1, 5, 7), (5000, 8191, 3, 64, 64), (8192, 8192, 3, 4, 16)])
def test_subm_rulebook_of_a_small_layer_equals_the_general_one(n, mv, ksize, cin, cout):
    """A layer of at most 8 192 rows builds its rulebook in one launch; with one row more it takes the passes over a table in memory.
    Same pairs, status and outputs, also where two rows name one cell and where rows lie outside the grid."""
    rng = np.random.default_rng(n + mv)
    grid, most = (41, 300, 200), 8193
    coors = np.zeros((most, 4), np.int32)
    coors[:n] = F.clustered_active_voxels(n, grid, 7, n_blobs=12)[:n] if n else 0
    if n >= 64:
        coors[n - 5:n] = coors[3:8]  # (the first row of a cell has it)
        coors[10, 1], coors[20, 2], coors[30, 3] = -1, grid[1], grid[2] + 7
    feat = np.zeros((most, cin), np.float32)
    feat[:n] = rng.uniform(-1, 1, (n, cin))
    w = rng.normal(0, 0.1, (ksize ** 3, cin, cout)).astype(np.float32)
    got = []
    for rows in (mv, most):
        conv = api.SubmConv3d(cin, cout, grid[::-1], w, rows, ksize=ksize, padding=ksize // 2)
        out = conv(dev(feat[:rows]), dev(coors[:rows]), dev(np.array([n], np.int32)))
        pairs, num = conv.export_rulebook()
        got.append((to_np(pairs)[:, :, :n], to_np(num), to_np(out)[:n], conv.status()))
        conv.close()
    assert got[0][3] == got[1][3] == (D.SESSD_STATUS_BAD_COORD if n >= 64 else 0)
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][0], got[1][0])
    # (the general path's workgroups may hold other tiles: sums in another order, 2^-24 a term and fewer than 27 Cin terms of 0.5 |x w|)
    assert np.allclose(got[0][2], got[1][2], rtol=0, atol=ksize ** 3 * cin * 2.0 ** -24)


@pytest.mark.parametrize("side", [1, 2, 3, 9])
def test_small_layer_whose_rows_name_few_cells(side):
    """8 192 rows on 1, 8, 27 and 729 cells: the pairs of the general path, in a time that does not grow with the rows of a cell (a walk
    through all of them for each took 0.9 ms; 17 us now)."""
    rng = np.random.default_rng(side)
    n, grid = 8192, (41, 300, 200)
    coors = np.zeros((n + 1, 4), np.int32)
    coors[:n, 1:] = [20, 100, 100] + rng.integers(0, side, (n, 3))
    feat, w = rng.uniform(-1, 1, (n + 1, 4)).astype(np.float32), rng.normal(0, 0.1, (27, 4, 16)).astype(np.float32)
    got = []
    for rows in (n, n + 1):
        conv = api.SubmConv3d(4, 16, grid[::-1], w, rows)
        args = dev(feat[:rows]), dev(coors[:rows]), dev(np.array([n], np.int32))
        out = conv(*args)
        pairs, num = conv.export_rulebook()
        got.append((to_np(pairs)[:, :, :n], to_np(num), to_np(out)[:n]))
        if rows == n:
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                conv(*args)
            end.record()
            end.synchronize()
            assert begin.elapsed_time(end) / 20 < 0.3
        conv.close()
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][0], got[1][0])
    assert np.allclose(got[0][2], got[1][2], rtol=0, atol=27 * 4 * 2.0 ** -24)


@pytest.mark.parametrize("cin,cout,half", [(4, 16, False), (16, 32, False), (32, 32, False), (64, 64, False), (64, 128, False), (4, 32, True),
                                           (16, 16, True), (32, 64, True), (64, 64, True), (64, 128, True), (128, 128, True)])
def test_rows_beyond_the_active_ones_beside_the_products_and_behind_them(cin, cout, half):
    """Rows beyond the active ones are written beside the products or behind them: on both sides of the lines between the two (as many of
    them as of the others in conv_wide.hip; a quarter of the workgroups with a tile in conv_tile.hip: 4 096 rows with 64 columns, 2 048 with
    128, on 256 compute units), without active rows, with more tiles than workgroups.  The active rows are the bits of a launch that
    leaves the others alone, and nothing behind the tensor is touched."""
    rng = np.random.default_rng(cin + cout)
    grid = (21, 400, 352)
    base = F.clustered_active_voxels(30000, grid, 9, n_blobs=300)
    sc, sh = rng.uniform(0.5, 1.5, cout).astype(np.float32), rng.uniform(-0.5, 0.5, cout).astype(np.float32)
    w = O.round_to_half(rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32))
    t_in, t_out = torch.float16 if half and cin != 4 else torch.float32, torch.float16 if half else torch.float32
    for n, mv in ((0, 1), (0, 9000), (1, 2), (2000, 4001), (2000, 4000), (2000, 3999), (2047, 9000), (2048, 9000), (4095, 9000), (4096, 9000),
                  (4096, 4097), (9000, 9000), (30000, 30001), (30000, 59999), (30000, 60000), (30000, 80000)):
        coors = np.zeros((mv, 4), np.int32)
        coors[:n] = base[:n]
        args = [dev(rng.uniform(-1, 1, (mv, cin)).astype(np.float32), t_in), dev(coors), dev(np.array([n], np.int32))]
        conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
        for relu in (False, True):
            conv.set_epilogue(sc if relu else None, sh, relu=relu)
            got = []
            for flags in (D.SESSD_FLAG_SKIP_PAD_ROWS, 0):
                conv.set_flags(flags)
                out = torch.full((mv + 64, cout), 7.0, dtype=t_out, device="cuda:0")
                conv.configure(args, [out[:mv]])
                conv.enqueue(args, [out[:mv]])
                got.append(to_np(out.float()))
            assert np.array_equal(got[0][:n], got[1][:n]) and (got[0][n:] == 7).all() and (got[1][mv:] == 7).all(), (n, mv)
            want = np.maximum(sh, 0) if relu else sh
            assert np.array_equal(got[1][n:mv], np.broadcast_to(O.round_to_half(want) if half else want, (mv - n, cout))), (n, mv)
        conv.close()


def _replays(calls, times=15):
    """The least time of `times` replays of each call, captured 16 times over, the calls in turn: ms."""
    graphs, keep, stream = [], [], torch.cuda.Stream()
    for call in calls:
        with torch.cuda.stream(stream):
            keep.append(call())
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=stream):
                keep += [call() for _ in range(16)]
        graphs.append(g)
    least = [float("inf")] * len(graphs)
    with torch.cuda.stream(stream):
        for _ in range(times):
            for i, g in enumerate(graphs):
                begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                begin.record()
                g.replay()
                end.record()
                end.synchronize()
                least[i] = min(least[i], begin.elapsed_time(end))
    return least


@pytest.mark.parametrize("channels", [64, 128])
def test_a_full_tensor_pays_nothing_for_rows_beyond_the_active_ones(channels):
    """A launch that may write rows beyond the active ones and has none to write, next to one that leaves such rows alone: the least of 15
    replays of 16 launches each (0.99 to 1.00 of it; 1.07 when every stage of the products asked whether there was something to write)."""
    grid, n = (21, 400, 352), 16000
    rng = np.random.default_rng(channels)
    args = [dev(rng.uniform(-1, 1, (n, channels)).astype(np.float32), torch.float16), dev(F.clustered_active_voxels(n, grid, 3, n_blobs=160)),
            dev(np.array([n], np.int32))]
    w = rng.normal(0, 0.1, (27, channels, channels)).astype(np.float32)
    owner = api.SubmConv3d(channels, channels, grid[::-1], w, n)
    owner(*args)
    torch.cuda.synchronize()
    convs = []
    for flags in (D.SESSD_FLAG_SKIP_PAD_ROWS, 0):
        convs.append(api.SubmConv3d(channels, channels, grid[::-1], w, n))
        convs[-1].set_flags(flags)
    for _ in range(3):  # (a neighbour's work may disturb a measurement)
        least = _replays([lambda c=c: c(*args, rulebook_from=owner) for c in convs])
        if least[1] < 1.03 * least[0]:
            break
    assert least[1] < 1.03 * least[0], least


@pytest.mark.parametrize("cin,cout", [(4, 16), (4, 32), (16, 16)])
def test_small_layer_without_rows_is_no_longer_than_two_launches(cin, cout):
    """A captured call of a layer of at most 8 192 rows with none active, rulebook and products in one launch, next to the same with
    products of its own launch on the vector units (half of it; 1.0 to 1.3 when it built the rulebook of no rows and multiplied)."""
    grid, mv = (41, 300, 200), 2000
    w = np.random.default_rng(cin).normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    args = dev(np.ones((mv, cin), np.float32)), dev(np.zeros((mv, 4), np.int32)), dev(np.zeros(1, np.int32))
    convs = [api.SubmConv3d(cin, cout, grid[::-1], w, mv) for _ in range(2)]
    convs[1].set_flags(D.SESSD_FLAG_FORCE_VALU)
    for _ in range(3):  # (a neighbour's work may disturb a measurement)
        least = _replays([lambda c=c: c(*args) for c in convs])
        if least[0] < least[1]:
            break
    print("one launch %.2f us, two %.2f" % tuple(1e3 / 16 * t for t in least))
    assert least[0] < least[1], least
    for c in convs:
        pairs, num = (to_np(t) for t in c.export_rulebook())
        assert c.status() == 0 and (num == 0).all() and (pairs == -1).all()


@pytest.mark.parametrize("ksize", [1, 3])
@pytest.mark.parametrize("cin,cout", [(4, 16), (4, 32), (16, 16)])
def test_small_layer_with_its_products_in_the_same_launch(cin, cout, ksize):
    """FP32 layers of at most 8 192 rows and few channels multiply in the launch that builds their rulebook: the outputs of the
    two launches (the layer on its own rulebook as a sharer), and all rows beyond the active ones.  An infinite weight reaches the
    rows that have the neighbour, and no other."""
    rng = np.random.default_rng(cin + cout + ksize)
    grid, K = (41, 300, 200), ksize ** 3
    sc, sh = rng.uniform(0.5, 1.5, cout).astype(np.float32), rng.uniform(-0.5, 0.5, cout).astype(np.float32)
    for n, mv, infinite in ((0, 1, False), (1, 1, False), (0, 130, False), (63, 64, False), (64, 65, False), (65, 400, True), (2000, 2000, False),
                            (4097, 5000, True), (8192, 8192, False)):
        coors = np.zeros((mv, 4), np.int32)
        coors[:n] = F.clustered_active_voxels(n, grid, 7, n_blobs=12)[:n] if n else 0
        if n >= 64:
            coors[n - 5:n] = coors[3:8]
            coors[10, 1], coors[20, 2], coors[30, 3] = -1, grid[1], grid[2] + 7
        feat = rng.uniform(-1, 1, (mv, cin)).astype(np.float32)
        w = rng.normal(0, 0.1, (K, cin, cout)).astype(np.float32)
        if infinite:
            w[K // 3, 1, 2] = np.inf
        conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv, ksize=ksize, padding=ksize // 2)
        args = dev(feat), dev(coors), dev(np.array([n], np.int32))
        for epilogue in (False, True):
            if epilogue:
                conv.set_epilogue(sc, sh, relu=True)
            one = to_np(conv(*args))
            two = to_np(conv(*args, rulebook_from=conv))
            assert np.array_equal(np.isnan(one), np.isnan(two)) and np.array_equal(np.isinf(one), np.isinf(two)), (n, mv)
            assert np.array_equal(one[n:], np.broadcast_to(np.maximum(sh, 0) if epilogue else np.float32(0), (mv - n, cout))), (n, mv)
            # (sums in another order: 2^-24 a term of at most 0.5, times a scale of 1.5)
            some = np.isfinite(two)
            assert np.allclose(one[some], two[some], rtol=0, atol=1.5 * K * cin * 2.0 ** -24), (n, mv)
        conv.set_flags(D.SESSD_FLAG_SKIP_PAD_ROWS)
        out = torch.full((mv, cout), 7.0, device="cuda:0")
        conv.enqueue(list(args), [out])
        assert np.array_equal(to_np(out)[:n], one[:n], equal_nan=True) and (to_np(out)[n:] == 7).all(), (n, mv)
        conv.close()


@pytest.mark.parametrize("cin,cout", [(4, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
                                      (5, 7), (8, 32)])
def test_subm_clustered_with_epilogue_and_pad_rows(cin, cout):
    grid = (21, 200, 176)
    n, mv = 6000, 8192
    rng = np.random.default_rng(cin)
    coors = F.clustered_active_voxels(n, grid, 1, n_blobs=60)
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    sc = rng.uniform(0.5, 1.5, cout).astype(np.float32)
    sh = rng.uniform(-0.2, 0.2, cout).astype(np.float32)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv, sc, sh, True)
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    assert int(o_num.sum()) > 4 * n
    assert np.array_equal(num, o_num)
    assert np.array_equal(O.canonical_rulebook(pairs, num, cbuf, cbuf), O.canonical_rulebook(o_pairs, o_num, coors, coors))
    # within an offset the exported pairs are in ascending output-row order, unused entries are -1
    for k in (0, 13, 26):
        assert np.all(np.diff(pairs[k, 1, :num[k]]) > 0) and np.all(pairs[k, :, num[k]:] == -1)
    o_out = O.scale_shift_relu(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), mv, sc, sh, True)
    assert_features_close(out, o_out, RTOL_FP32, "subm %d->%d" % (cin, cout),   # incl. pad rows = relu(shift)
                          abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv, sc, sh))


@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
def test_equal_work_tiles_with_dense_and_isolated_regions(dtype):
    """A fully dense block (27 pairs per row) followed by isolated voxels (1 pair per row): the equal-work tile
    cuts give the isolated stretch runs far longer than the kernel's tile capacity, which it walks in pieces.
    Shuffled row order as a second case (every tile mixes both kinds)."""
    grid = (21, 800, 704)
    rng = np.random.default_rng(31)
    z, y, x = np.meshgrid(np.arange(2, 14), np.arange(100, 114), np.arange(200, 214), indexing="ij")
    dense = np.stack([np.zeros(z.size, np.int64), z.ravel(), y.ravel(), x.ravel()], 1)
    iso = np.stack([np.zeros(4000, np.int64), rng.integers(0, 21, 4000) // 3 * 3, 300 + 3 * (np.arange(4000) // 60),
                    3 * (np.arange(4000) % 60)], 1)
    iso = np.unique(iso, axis=0)
    for order in ("blocked", "shuffled"):
        coors = np.concatenate([dense, iso]).astype(np.int32)
        if order == "shuffled":
            coors = coors[rng.permutation(len(coors))]
        n, mv = len(coors), 8192
        feat = rng.uniform(-1, 1, (n, 64)).astype(np.float32)
        w = rng.normal(0, 0.05, (27, 64, 64)).astype(np.float32)
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        assert o_num[13] == n and int(o_num.sum()) > 20 * len(dense)
        if dtype == "fp32":
            conv, out, pairs, num, _ = run_subm(coors, n, feat, w, grid, mv)
            assert np.array_equal(num, o_num)
            assert_features_close(out[:n], O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)[:n], RTOL_FP32, order,
                                  abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv)[:n])
        else:
            conv = api.SubmConv3d(64, 64, grid[::-1], w, mv)
            cbuf = np.zeros((mv, 4), np.int32)
            cbuf[:n] = coors
            fbuf = np.zeros((mv, 64), np.float16)
            fbuf[:n] = feat
            out = to_np(conv(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32))).float())
            wh = w.astype(np.float16).astype(np.float32)
            want = O.gather_gemm_scatter(fbuf[:n].astype(np.float32), wh, o_pairs, o_num, mv)[:n]
            assert_features_close(out[:n], want, RTOL_FP16, order, half=True,
                                  abs_sum=abs_sum_of(fbuf[:n].astype(np.float32), wh, o_pairs, o_num, mv)[:n])
        assert conv.status() == 0


def test_mfma_and_valu_paths_agree():
    """The matrix-core kernel against the shape-agnostic VALU kernel on the same rulebook (both FP32)."""
    grid = (11, 120, 120)
    n, mv = 9000, 9001                      # a last tile that is only partly active
    rng = np.random.default_rng(7)
    coors = F.clustered_active_voxels(n, grid, 5, n_blobs=30, sigma=(1.5, 5.0, 5.0))
    feat = rng.uniform(-1, 1, (n, 64)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, 64, 64)).astype(np.float32)
    outs = []
    for flags in (0, D.SESSD_FLAG_FORCE_VALU):
        conv = api.SubmConv3d(64, 64, grid[::-1], w, mv)
        conv.set_flags(flags)
        cbuf = np.zeros((mv, 4), np.int32)
        cbuf[:n] = coors
        fbuf = np.zeros((mv, 64), np.float32)
        fbuf[:n] = feat
        outs.append(to_np(conv(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))))
    o_pairs, o_num, _ = O.subm_rulebook(cbuf, n, grid[::-1], mv)
    assert_features_close(outs[0], outs[1], RTOL_FP32, "mfma vs valu", abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv))


@pytest.mark.parametrize("cin,cout", [(4, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
                                      (8, 32)])
def test_subm_fp16_features(cin, cout):
    """FP16 features and weights, FP32 accumulate (benchmark configurations 4-5).  The oracle runs in FP32 on the
    half-rounded inputs and weights and rounds its output to half: agreement within 1e-2 relative."""
    grid = (21, 200, 176)
    n, mv = 6000, 8192
    rng = np.random.default_rng(100 + cin)
    coors = F.clustered_active_voxels(n, grid, 2, n_blobs=60)
    in_half = cin != 4                               # the first layer reads the voxelizer's FP32 means
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    if in_half:
        feat = O.round_to_half(feat)
    w = O.round_to_half(rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32))
    sc = rng.uniform(0.5, 1.5, cout).astype(np.float32)
    sh = rng.uniform(-0.2, 0.2, cout).astype(np.float32)
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
    conv.set_epilogue(sc, sh, True)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, cin), np.float32)
    fbuf[:n] = feat
    d_feat = dev(fbuf, torch.float16 if in_half else torch.float32)
    out = conv(d_feat, dev(cbuf), dev(np.array([n], np.int32)), out_dtype=torch.float16)
    torch.cuda.synchronize()
    assert out.dtype == torch.float16
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    o_out = O.round_to_half(O.scale_shift_relu(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), mv, sc, sh, True))
    assert_features_close(to_np(out.float()), o_out, RTOL_FP16, "fp16 subm %d->%d" % (cin, cout))
    # the MFMA and VALU FP16 paths agree much more tightly than the 1e-2 bound
    conv.set_flags(D.SESSD_FLAG_FORCE_VALU)
    out2 = conv(d_feat, dev(cbuf), dev(np.array([n], np.int32)), out_dtype=torch.float16)
    torch.cuda.synchronize()
    assert_features_close(to_np(out.float()), to_np(out2.float()), 2e-3, "fp16 mfma vs valu %d->%d" % (cin, cout))


def test_sparse_fp16_features():
    layer = SPARSE_LAYERS[1]        # 32 -> 64, stride 2
    ig = sparse_input_grid(layer)
    n, mv = 5000, 30000
    rng = np.random.default_rng(77)
    coors = F.clustered_active_voxels(n, (ig[0], 300, 300), 3, n_blobs=50)
    feat = O.round_to_half(rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32))
    conv = api.SparseConv3d(layer.cin, layer.cout, layer.out_shape, ig[::-1], layer.ksize, layer.stride,
                            layer.padding, w, mv)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, layer.cin), np.float32)
    fbuf[:n] = feat
    out, oc, on = conv(dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32)))
    torch.cuda.synchronize()
    o_pairs, o_num, o_oc, o_on, _ = O.sparse_rulebook(coors, n, layer.out_shape, layer.ksize, layer.stride,
                                                      layer.padding, mv)
    assert int(to_np(on)[0]) == o_on and np.array_equal(to_np(oc), o_oc)
    o_out = O.round_to_half(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv))
    assert_features_close(to_np(out.float()), o_out, RTOL_FP16, "fp16 sparse15")


def test_sparse2dense_fp16():
    rng = np.random.default_rng(3)
    n, mv, c = 1500, 4096, 64
    coors = F.random_active_voxels(n, (2, 200, 176), 9)
    feat = O.round_to_half(rng.uniform(0.1, 1, (n, c)).astype(np.float32))
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, c), np.float32)
    fbuf[:n] = feat
    s2d = api.Sparse2Dense()
    dense = s2d(dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32)))
    torch.cuda.synchronize()
    assert dense.dtype == torch.float16
    assert np.array_equal(to_np(dense.float()), O.sparse2dense(feat, coors, n, B.DENSE_SIZE_XYZ))


def test_subm_shared_rulebook_skip_pad_and_empty():
    grid = (11, 100, 88)
    n, mv = 3000, 4096
    rng = np.random.default_rng(5)
    coors = F.clustered_active_voxels(n, grid, 2)
    feat = rng.uniform(-1, 1, (n, 16)).astype(np.float32)
    w1 = rng.normal(0, 0.1, (27, 16, 16)).astype(np.float32)
    w2 = rng.normal(0, 0.1, (27, 16, 32)).astype(np.float32)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, 16), np.float32)
    fbuf[:n] = feat
    a = api.SubmConv3d(16, 16, grid[::-1], w1, mv)
    b = api.SubmConv3d(16, 32, grid[::-1], w2, mv)
    b.set_flags(D.SESSD_FLAG_SKIP_PAD_ROWS)
    d_coors, d_num = dev(cbuf), dev(np.array([n], np.int32))
    y1 = a(dev(fbuf), d_coors, d_num)
    y2 = b(y1, d_coors, d_num, rulebook_from=a)           # GEMM only, on a's rulebook
    torch.cuda.synchronize()
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    o1 = O.gather_gemm_scatter(feat, w1, o_pairs, o_num, mv)
    o2 = O.gather_gemm_scatter(o1, w2, o_pairs, o_num, mv)
    assert_features_close(to_np(y1), o1, RTOL_FP32, "shared: layer 1")
    assert_features_close(to_np(y2)[:n], o2[:n], RTOL_FP32, "shared: layer 2")
    # empty input: nothing active, all rows are pad rows
    y0 = a(dev(fbuf), d_coors, dev(np.array([0], np.int32)))
    pairs, num = a.export_rulebook()
    torch.cuda.synchronize()
    assert np.all(to_np(y0) == 0) and np.all(to_np(num) == 0) and np.all(to_np(pairs) == -1)


@pytest.mark.parametrize("owner_cout,sharer_cout", [(64, 32), (32, 64)])
def test_shared_rulebook_between_layers_of_different_tile_capacity(owner_cout, sharer_cout):
    """Two FP16 3x3x3 layers of different widths on one rulebook.  Both run on the kernel of conv_tall.hip, which cuts
    its own tiles (a rulebook built by such a layer carries no equal-work cuts) and whose order of sums follows from the
    row count alone, the same in both calls: the sharer's output on the owner's rulebook must equal its output on its
    own bit for bit."""
    grid = (21, 400, 352)
    n, mv, cin = 15000, 16384, 32
    rng = np.random.default_rng(41)
    coors = F.clustered_active_voxels(n, grid, 2, n_blobs=120)
    feat = O.round_to_half(rng.uniform(-1, 1, (n, cin)).astype(np.float32))
    w1 = O.round_to_half(rng.normal(0, 0.1, (27, cin, owner_cout)).astype(np.float32))
    w2 = O.round_to_half(rng.normal(0, 0.1, (27, cin, sharer_cout)).astype(np.float32))
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, cin), np.float32)
    fbuf[:n] = feat
    a = api.SubmConv3d(cin, owner_cout, grid[::-1], w1, mv)
    b = api.SubmConv3d(cin, sharer_cout, grid[::-1], w2, mv)
    d_feat, d_coors, d_num = dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32))
    y1 = a(d_feat, d_coors, d_num, out_dtype=torch.float16)
    y2 = b(d_feat, d_coors, d_num, out_dtype=torch.float16, rulebook_from=a)
    torch.cuda.synchronize()
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    o1 = O.round_to_half(O.gather_gemm_scatter(feat, w1, o_pairs, o_num, mv))
    o2 = O.round_to_half(O.gather_gemm_scatter(feat, w2, o_pairs, o_num, mv))
    assert_features_close(to_np(y1.float()), o1, RTOL_FP16, "owner %d" % owner_cout)
    assert_features_close(to_np(y2.float()), o2, RTOL_FP16, "sharer %d" % sharer_cout)
    y3 = b(d_feat, d_coors, d_num, out_dtype=torch.float16)      # the sharer on its own rulebook
    torch.cuda.synchronize()
    assert torch.equal(y2, y3)


@pytest.mark.parametrize("n", [1, 17, 300])
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
def test_fewer_rows_than_tiles_in_a_wide_layer(n, dtype):
    """A handful of active rows in a layer wide enough to get equal-work tile cuts: the rows weigh more than
    total / tiles, and every entry of the cut table up to the last tile must still be written."""
    grid = (3, 48, 15)
    mv, cin, cout = n + 225, 64, 64
    half = dtype == "fp16"
    rng = np.random.default_rng(n)
    coors = F.clustered_active_voxels(n, grid, 5, n_blobs=2)
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    if half:
        feat, w = O.round_to_half(feat), O.round_to_half(w)
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, cin), np.float32)
    fbuf[:n] = feat
    tdt = torch.float16 if half else torch.float32
    for _ in range(2):                                       # the second call finds the first one's table
        out = conv(dev(fbuf, tdt), dev(cbuf), dev(np.array([n], np.int32)), out_dtype=tdt)
        torch.cuda.synchronize()
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
        terms = abs_sum_of(feat, w, o_pairs, o_num, mv)
        if half:
            assert_features_close(to_np(out.float()), O.round_to_half(o_out), RTOL_FP16, "few rows fp16", abs_sum=terms, half=True)
        else:
            assert_features_close(to_np(out), o_out, RTOL_FP32, "few rows fp32", abs_sum=terms)
        assert conv.status() == 0


def test_few_output_sites_in_a_wide_strided_layer():
    """36 input cells, kernel (3,3,1), stride (3,1,2): a few dozen output rows in a 32 -> 64 layer."""
    k, s, p, ig = (3, 3, 1), (3, 1, 2), (0, 1, 0), (3, 26, 7)
    og = tuple(B.conv_out_size(ig[a], k[a], s[a], p[a]) for a in range(3))
    layer = B.Layer("t", D.SESSD_LAYER_SPARSE, 32, 64, og[::-1], k, s, p)
    n, mv = 36, 86
    rng = np.random.default_rng(4)
    coors = F.random_active_voxels(n, ig, 11)
    feat = rng.uniform(-1, 1, (n, 32)).astype(np.float32)
    w = rng.normal(0, 0.1, (layer.kvol, 32, 64)).astype(np.float32)
    conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
    o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, og[::-1], k, s, p, mv)
    assert on == o_on and conv.status() == o_st and np.array_equal(oc, o_oc) and np.array_equal(num, o_num)
    assert_features_close(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), RTOL_FP32, "few output sites")


def test_subm_bad_coordinate_is_flagged_not_written():
    grid = (5, 20, 20)
    coors = np.array([[0, 1, 1, 1], [0, 1, 1, 2], [0, 7, 1, 1], [0, 1, 25, 1]], np.int32)   # rows 2,3 outside
    feat = np.ones((4, 4), np.float32)
    w = np.ones((27, 4, 4), np.float32)
    conv, out, pairs, num, _ = run_subm(coors, 4, feat, w, grid, 64)
    assert conv.status() & D.SESSD_STATUS_BAD_COORD
    o_pairs, o_num, o_st = O.subm_rulebook(coors, 4, grid[::-1], 64)
    assert o_st & D.SESSD_STATUS_BAD_COORD and np.array_equal(num, o_num)
    assert np.array_equal(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, 64))


SPARSE_LAYERS = [l for l in B.reference_layers() if l.type == D.SESSD_LAYER_SPARSE]


def sparse_input_grid(layer):
    """Input grid (z,y,x) of a reference sparse layer = out grid of the stage before it."""
    prev = {"sparse6": (41, 1600, 1408), "sparse15": (21, 800, 704), "sparse27": (11, 400, 352), "sparse39": (5, 200, 176)}
    return prev[layer.name]


def run_sparse(layer, coors, n, feat, w, mv, in_grid_zyx, **kw):
    conv = api.SparseConv3d(layer.cin, layer.cout, layer.out_shape, in_grid_zyx[::-1], layer.ksize, layer.stride,
                            layer.padding, w, mv)
    if kw.get("epilogue"):
        conv.set_epilogue(*kw["epilogue"])
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors[:n]
    fbuf = np.zeros((mv, layer.cin), np.float32)
    fbuf[:n] = feat[:n]
    out, oc, on = conv(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    pairs, num = conv.export_rulebook()
    torch.cuda.synchronize()
    return conv, to_np(out), to_np(oc), int(to_np(on)[0]), to_np(pairs), to_np(num).astype(np.uint32)


@pytest.mark.parametrize("layer", SPARSE_LAYERS, ids=[l.name for l in SPARSE_LAYERS])
def test_sparse_layers_of_the_backbone(layer):
    """Each strided layer shape of params.h on a neighbour-rich active set in its own input grid."""
    ig = sparse_input_grid(layer)
    n, mv = 5000, 30000
    rng = np.random.default_rng(len(layer.name))
    sub = (ig[0], min(ig[1], 300), min(ig[2], 300))
    coors = F.clustered_active_voxels(n, sub, 3, n_blobs=50)
    feat = rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32)
    conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
    o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, layer.out_shape, layer.ksize, layer.stride,
                                                         layer.padding, mv)
    assert on == o_on and conv.status() == o_st == 0
    assert np.array_equal(oc, o_oc)                       # first-seen numbering reproduced row by row
    assert np.array_equal(canonical(oc, on)[0], canonical(o_oc, o_on)[0])
    assert np.array_equal(num, o_num)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    assert np.array_equal(O.canonical_rulebook(pairs, num, cbuf, oc), O.canonical_rulebook(o_pairs, o_num, coors, o_oc))
    o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
    terms = abs_sum_of(feat, w, o_pairs, o_num, mv)
    assert_features_close(out, o_out, RTOL_FP32, layer.name, abs_sum=terms)
    a = canonical(oc, on, out)
    b = canonical(o_oc, o_on, o_out)
    assert_features_close(a[1], b[1], RTOL_FP32, layer.name + " (canonical order)", abs_sum=canonical(o_oc, o_on, terms)[1])


@pytest.mark.parametrize("n", [32768, 32769, 66000, 150001])
def test_strided_layer_with_more_chunks_than_blocks(n):
    """A strided layer's passes have at most 1024 blocks of 256 tickets (32 768 rows of a stride-2 layer), the tile cuts 512 of
    256 rows: beyond, a block walks several chunks and carries the count in front of it along."""
    layer = SPARSE_LAYERS[1]                                    # 32 -> 64: the narrowest layer that gets tile cuts
    ig = sparse_input_grid(layer)
    rng = np.random.default_rng(n)
    coors = F.clustered_active_voxels(n, ig, n, n_blobs=n // 50)
    feat = rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32)
    mv = n + 37
    O.set_threads(16)
    try:
        conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
        o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, layer.out_shape, layer.ksize, layer.stride, layer.padding, mv)
        assert on == o_on and conv.status() == o_st
        assert np.array_equal(oc, o_oc) and np.array_equal(num, o_num)
        o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
        assert_features_close(out, o_out, RTOL_FP32, layer.name, abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv))
        # (tile cuts of as many output rows)
        sub = api.SubmConv3d(32, 64, ig[::-1], w, n)
        cbuf = np.zeros((n, 4), np.int32)
        cbuf[:] = coors
        got = to_np(sub(dev(feat), dev(cbuf), dev(np.array([n], np.int32))))
        s_pairs, s_num, _ = O.subm_rulebook(coors, n, ig[::-1], n)
        want = O.gather_gemm_scatter(feat, w, s_pairs, s_num, n)
        assert_features_close(got, want, RTOL_FP32, "subm, %d rows" % n, abs_sum=abs_sum_of(feat, w, s_pairs, s_num, n, n))
    finally:
        O.set_threads(1)


def test_sparse_cap_overflow_and_empty():
    layer = SPARSE_LAYERS[0]
    ig = sparse_input_grid(layer)
    n = 4000
    rng = np.random.default_rng(9)
    coors = F.random_active_voxels(n, (ig[0], 200, 200), 4)    # uncorrelated sites: the set grows ~8x
    feat = rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32)
    mv = 8192
    conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
    o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, layer.out_shape, layer.ksize, layer.stride,
                                                         layer.padding, mv)
    assert o_st & D.SESSD_STATUS_VOXEL_OVERFLOW and conv.status() & D.SESSD_STATUS_VOXEL_OVERFLOW
    assert on == o_on == mv and np.array_equal(oc, o_oc) and np.array_equal(num, o_num)
    assert_features_close(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), RTOL_FP32, "capped sparse layer")
    # an empty frame through the same plugin and workspace, which still hold the full frame's tickets and flags
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, layer.cin), np.float32)
    fbuf[:n] = feat
    out2, oc2, on2 = conv(dev(fbuf), dev(cbuf), dev(np.array([0], np.int32)))
    num2 = conv.export_rulebook()[1]
    torch.cuda.synchronize()
    assert int(to_np(on2)[0]) == 0 and not to_np(out2).any() and not to_np(oc2).any() and not to_np(num2).any()
    assert conv.status() == 0
    conv, out, oc, on, pairs, num = run_sparse(layer, coors, 0, feat, w, mv, ig)
    assert on == 0 and np.all(out == 0) and np.all(oc == 0) and np.all(num == 0)


def test_sparse_layer_refuses_negative_coordinates():
    """Rows with a negative coordinate (for which getValidOutPos' truncating divisions give kernel offsets outside
    the rulebook) contribute nothing and raise BAD_COORD; everything else equals the oracle, which drops them too."""
    layer = SPARSE_LAYERS[0]
    ig = sparse_input_grid(layer)
    n, mv = 3000, 16384
    rng = np.random.default_rng(12)
    coors = F.clustered_active_voxels(n, (ig[0], 200, 200), 8, n_blobs=30)
    bad = rng.choice(n, 40, replace=False)
    coors[bad[:15], 1] = -rng.integers(1, 4, 15)
    coors[bad[15:30], 2] = -rng.integers(1, 40, 15)
    coors[bad[30:], 3] = -2
    feat = rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32)
    conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
    o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, layer.out_shape, layer.ksize, layer.stride,
                                                         layer.padding, mv)
    assert conv.status() == o_st == D.SESSD_STATUS_BAD_COORD
    assert on == o_on and np.array_equal(oc, o_oc) and np.array_equal(num, o_num)
    assert not np.isin(pairs[:, 0, :][pairs[:, 0, :] >= 0], bad).any()       # no pair names a refused row
    assert_features_close(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), RTOL_FP32, "rows with negative coordinates")


def test_sparse_generic_stride1_and_corner_truncation():
    """stride 1 (27 candidates per input) and cells at coordinate 0 with padding 0 (C division
    truncates toward zero in getValidOutPos)."""
    cases = [((3, 3, 3), (1, 1, 1), (1, 1, 1), (6, 9, 8)), ((3, 3, 3), (2, 2, 2), (0, 0, 0), (9, 9, 9)),
             ((2, 2, 2), (2, 2, 2), (0, 0, 0), (8, 8, 8)), ((1, 3, 3), (1, 2, 2), (0, 1, 1), (4, 9, 9))]
    rng = np.random.default_rng(1)
    for k, s, p, ig in cases:
        og = tuple(B.conv_out_size(ig[a], k[a], s[a], p[a]) for a in range(3))
        layer = B.Layer("t", D.SESSD_LAYER_SPARSE, 8, 16, og[::-1], k, s, p)
        n = ig[0] * ig[1] * ig[2] // 2
        coors = F.random_active_voxels(n, ig, 6)
        feat = rng.uniform(-1, 1, (n, 8)).astype(np.float32)
        w = rng.normal(0, 0.1, (layer.kvol, 8, 16)).astype(np.float32)
        mv = 1024
        conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
        o_pairs, o_num, o_oc, o_on, _ = O.sparse_rulebook(coors, n, og[::-1], k, s, p, mv)
        assert on == o_on and np.array_equal(oc, o_oc) and np.array_equal(num, o_num), (k, s, p)
        assert_features_close(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), RTOL_FP32, str((k, s, p)))


@pytest.mark.parametrize("less", [0, 1])
@pytest.mark.parametrize("padding", [(2, 2, 2), (2, 0, 1), (0, 2, 1), (1, 1, 2)])
def test_sparse_kernels_of_3_with_strides_of_2(padding, less):
    """Candidates that are found without a division, for every padding up to 2, grids of even and odd size, and an output grid that the
    last candidates lie outside of."""
    k, s, rng = (3, 3, 3), (2, 2, 2), np.random.default_rng(7)
    for ig in ((6, 9, 8), (7, 12, 11)):
        og = tuple(B.conv_out_size(ig[a], k[a], s[a], padding[a]) - less for a in range(3))
        layer = B.Layer("t", D.SESSD_LAYER_SPARSE, 8, 16, og[::-1], k, s, padding)
        n, mv = ig[0] * ig[1] * ig[2] // 2, 1024
        coors = F.random_active_voxels(n, ig, 6)
        feat = rng.uniform(-1, 1, (n, 8)).astype(np.float32)
        w = rng.normal(0, 0.1, (27, 8, 16)).astype(np.float32)
        conv, out, oc, on, pairs, num = run_sparse(layer, coors, n, feat, w, mv, ig)
        o_pairs, o_num, o_oc, o_on, o_st = O.sparse_rulebook(coors, n, og[::-1], k, s, padding, mv)
        assert conv.status() == o_st
        assert on == o_on and np.array_equal(oc, o_oc) and np.array_equal(num, o_num), ig
        assert_features_close(out, O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), RTOL_FP32, str((ig, padding)))


def test_sparse2dense_with_folded_zero_pad():
    # sparse2Dense followed by ZeroPad2dPlugin (se-ssd-ai-trt.cpp:1253) in one scatter; a copy: bit-exact
    rng = np.random.default_rng(12)
    n, mv, c = 2739, 8192, 64
    coors = F.random_active_voxels(n, (2, 200, 176), 9)
    coors[:4] = [(0, 0, 0, 0), (0, 1, 199, 175), (0, 0, 199, 0), (0, 1, 0, 175)]      # the four corners
    coors = np.unique(coors, axis=0)
    n = len(coors)
    feat = rng.uniform(0.1, 1, (n, c)).astype(np.float32)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, c), np.float32)
    fbuf[:n] = feat
    for pad in [(1, 1, 1, 1), (2, 0, 1, 3)]:
        for dt in (torch.float32, torch.float16):
            s2d = api.Sparse2Dense(padding=pad)
            f = dev(fbuf).to(dt)
            dense = s2d(f, dev(cbuf), dev(np.array([n], np.int32)))
            torch.cuda.synchronize()
            want = O.zero_pad2d(O.sparse2dense(to_np(f[:n].float()), coors, n, B.DENSE_SIZE_XYZ), *pad)
            assert tuple(dense.shape) == want.shape
            assert np.array_equal(to_np(dense.float()), want), (pad, dt)
            assert s2d.status() == 0
    # the output descriptor must carry the padded shape
    s2d = api.Sparse2Dense(padding=(1, 1, 1, 1))
    bad = torch.empty((128, 200, 176), dtype=torch.float32, device="cuda")
    with pytest.raises(api.SessdError):
        s2d.configure([dev(fbuf), dev(cbuf), dev(np.array([n], np.int32))], [bad])


@pytest.mark.parametrize("size_xyz,channel,pad", [((1000, 12, 3), 40, (0, 0, 0, 0)), ((1000, 12, 3), 40, (1, 0, 3, 2)),
                                                  ((449, 9, 1), 5, (0, 1, 0, 0)), ((7, 5, 2), 3, (0, 0, 0, 0))])
def test_sparse2dense_long_lines_and_odd_shapes(size_xyz, channel, pad):
    """Lines longer than one LDS segment, widths no 16-byte run divides, fewer channels than a channel group."""
    rng = np.random.default_rng(5)
    W, H, Dz = size_xyz
    n, mv = min(3000, W * H * Dz // 3), 4000
    coors = F.random_active_voxels(n, (Dz, H, W), 8)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = rng.uniform(0.1, 1, (mv, channel)).astype(np.float32)
    for dt in (torch.float32, torch.float16):
        s2d = api.Sparse2Dense(size_xyz, channel, padding=pad)
        f = dev(fbuf).to(dt)
        dense = s2d(f, dev(cbuf), dev(np.array([n], np.int32)))
        torch.cuda.synchronize()
        want = O.zero_pad2d(O.sparse2dense(to_np(f[:n].float()), coors, n, size_xyz), *pad)
        assert tuple(dense.shape) == want.shape
        assert np.array_equal(to_np(dense.float()), want), dt
        assert s2d.status() == 0


@pytest.mark.parametrize("size_xyz,channel,pad", [((178, 20, 2), 33, (0, 0, 0, 0)), ((176, 20, 1), 64, (1, 1, 1, 1)), ((450, 7, 2), 40, (0, 0, 0, 0)),
                                                  ((2, 5, 1), 3, (0, 0, 0, 0)), ((5, 6, 1), 8, (0, 0, 1, 0))])
@pytest.mark.parametrize("tin", [torch.float32, torch.float16])
@pytest.mark.parametrize("tout", [torch.float32, torch.float16])
def test_sparse2dense_lines_of_an_even_width(size_xyz, channel, pad, tin, tout):
    """Lines that no 16-byte run divides but pairs of elements do, also in two segments and with two cells only: a copy, bit for bit."""
    rng = np.random.default_rng(9)
    W, H, Dz = size_xyz
    n, mv = min(1500, W * H * Dz // 2), 1600
    coors = F.random_active_voxels(n, (Dz, H, W), 8)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    f = dev(rng.uniform(0.1, 1, (mv, channel)).astype(np.float32)).to(tin)
    s2d = api.Sparse2Dense(size_xyz, channel, padding=pad)
    dense = s2d(f, dev(cbuf), dev(np.array([n], np.int32)), out_dtype=tout)
    torch.cuda.synchronize()
    want = O.zero_pad2d(O.sparse2dense(to_np(f[:n].to(tout).float()), coors, n, size_xyz), *pad)
    assert dense.dtype == tout and np.array_equal(to_np(dense.float()), want)
    assert s2d.status() == 0


def test_sparse2dense():
    rng = np.random.default_rng(2)
    n, mv, c = 2739, 60000, 64
    coors = F.random_active_voxels(n, (2, 200, 176), 8)
    feat = rng.uniform(0.1, 1, (n, c)).astype(np.float32)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = rng.uniform(5, 6, (mv, c)).astype(np.float32)      # rows >= n hold garbage that must not leak
    fbuf[:n] = feat
    s2d = api.Sparse2Dense()
    dense = s2d(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    torch.cuda.synchronize()
    want = O.sparse2dense(feat, coors, n, B.DENSE_SIZE_XYZ)
    assert dense.shape == (128, 200, 176)
    assert np.array_equal(to_np(dense), want)
    assert s2d.status() == 0
    # the workspace may hold anything: the cell map is never cleared, a stale or random entry must not leak a row
    ws = s2d.ws.clone()
    for fill in (lambda t: t.fill_(0), lambda t: t.fill_(0x7f), lambda t: t.copy_(torch.randint(0, 256, t.shape, dtype=torch.uint8))):
        fill(ws)
        dense.fill_(3.0)
        s2d.enqueue([dev(fbuf), dev(cbuf), dev(np.array([n], np.int32))], [dense], workspace=ws)
        torch.cuda.synchronize()
        assert np.array_equal(to_np(dense), want)
    ws32 = ws.view(torch.int32)
    ws32.copy_(torch.randint(-3, 2 * n, ws32.shape, dtype=torch.int32))   # plausible row numbers everywhere
    s2d.enqueue([dev(fbuf), dev(cbuf), dev(np.array([n], np.int32))], [dense], workspace=ws)
    torch.cuda.synchronize()
    assert np.array_equal(to_np(dense), want)
    assert int(ws32[0].item()) == 0
    # idempotent on a dirty output buffer, empty input gives all zeros
    dense.fill_(3.0)
    s2d.enqueue([dev(fbuf), dev(cbuf), dev(np.array([0], np.int32))], [dense])
    torch.cuda.synchronize()
    assert float(dense.abs().max()) == 0.0
    cbuf[5] = (0, 2, 0, 0)                                        # z outside D=2
    s2d(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    assert s2d.status() & D.SESSD_STATUS_BAD_COORD


def test_conv_serialization_round_trip():
    rng = np.random.default_rng(4)
    w = rng.normal(0, 0.1, (27, 4, 16)).astype(np.float32)
    a = api.SubmConv3d(4, 16, (140, 160, 41), w, 2000)
    blob = a.serialize()
    assert len(blob) == 16 * 4 + w.size * 4                     # submConv3dlayer.cu:684-687
    head = np.frombuffer(blob[:64], np.int32)
    assert head.tolist() == [4, 16, 2000, 4, 140, 160, 41, 140, 160, 41, 3, 1, 1, 1, 0, w.size]
    assert np.array_equal(np.frombuffer(blob[64:], np.float32), w.ravel())
    a.set_epilogue(np.ones(16), np.zeros(16), True)
    blob2 = a.serialize()
    assert blob2[:len(blob)] == blob and len(blob2) > len(blob)
    b = api.SubmConv3d.deserialize(blob2)
    assert b.serialize() == blob2
    layer = SPARSE_LAYERS[2]
    ws = rng.normal(0, 0.1, (27, 64, 64)).astype(np.float32)
    s = api.SparseConv3d(64, 64, layer.out_shape, (352, 400, 11), layer.ksize, layer.stride, layer.padding, ws, 60000)
    sb = s.serialize()
    assert len(sb) == 22 * 4 + ws.size * 4                      # sparseConv3dlayer.cu:863-866
    assert np.frombuffer(sb[:88], np.int32).tolist() == [64, 64, 60000, 64, 176, 200, 5, 352, 400, 11, 3, 3, 3,
                                                          2, 2, 2, 0, 1, 1, 1, 0, ws.size]
    assert api.SparseConv3d.deserialize(sb).serialize() == sb


def test_conv_plugins_by_name_and_their_clones():
    """createPlugin(name, fields) and clone() of the reference's plugin surface for the two conv plugins: the plugin
    built from named fields, and its clone (own device weights, epilogue and flags carried over), give the bits of the
    plugin built from the descriptor."""
    grid = (21, 200, 176)
    n, mv = 3000, 4096
    rng = np.random.default_rng(77)
    coors = F.clustered_active_voxels(n, grid, 2, n_blobs=30)
    feat = rng.uniform(-1, 1, (n, 16)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, 16, 32)).astype(np.float32)
    sc, sh = rng.uniform(0.5, 1.5, 32).astype(np.float32), rng.uniform(-0.2, 0.2, 32).astype(np.float32)
    i32 = lambda *v: np.array(v, np.int32)  # noqa: E731
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, 16), np.float32)
    fbuf[:n] = feat
    ins = (dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    # SubM
    base = api.SubmConv3d(16, 32, grid[::-1], w, mv)
    named = api.create_plugin("SubmConv3dLayerPlugin", dict(
        in_channel=i32(16), out_channel=i32(32), max_voxels=i32(mv), feature_num=i32(16), out_shape=i32(*grid[::-1]),
        spatial_shape=i32(*grid[::-1]), ksize=i32(3), stride=i32(1), padding=i32(1), dilation=i32(1), out_padding=i32(0),
        weights=w))
    assert named.serialize() == base.serialize()
    for p in (base, named):
        p.set_epilogue(sc, sh, True)
        p.set_flags(D.SESSD_FLAG_SKIP_PAD_ROWS)
    twin = named.clone()
    assert twin.serialize() == named.serialize()
    named.close()                                         # the clone owns its own copies
    outs = [to_np(p(*ins))[:n] for p in (base, twin)]
    torch.cuda.synchronize()
    assert np.array_equal(outs[0], outs[1]) and np.abs(outs[0]).max() > 0
    # SparseConv
    layer = SPARSE_LAYERS[1]
    ig = sparse_input_grid(layer)
    coors = F.clustered_active_voxels(n, (ig[0], 200, 176), 4, n_blobs=30)
    cbuf[:n] = coors
    feat = rng.uniform(-1, 1, (n, layer.cin)).astype(np.float32)
    fbuf = np.zeros((mv, layer.cin), np.float32)
    fbuf[:n] = feat
    w = rng.normal(0, 0.1, (layer.kvol, layer.cin, layer.cout)).astype(np.float32)
    ins = (dev(fbuf), dev(cbuf), dev(np.array([n], np.int32)))
    base = api.SparseConv3d(layer.cin, layer.cout, layer.out_shape, ig[::-1], layer.ksize, layer.stride, layer.padding, w, mv)
    named = api.create_plugin("SparseConv3dLayerPlugin", dict(
        in_channel=i32(layer.cin), out_channel=i32(layer.cout), max_voxels=i32(mv), feature_num=i32(layer.cin),
        out_shape=i32(*layer.out_shape), spatial_shape=i32(*ig[::-1]), ksize=i32(*layer.ksize), stride=i32(*layer.stride),
        padding=i32(*layer.padding), dilation=i32(1), out_padding=i32(0), weights=w))
    assert named.serialize() == base.serialize()
    twin = named.clone()
    a, b = base(*ins), twin(*ins)
    torch.cuda.synchronize()
    na = int(to_np(a[2])[0])
    assert na == int(to_np(b[2])[0]) > 0 and np.array_equal(to_np(a[1]), to_np(b[1]))
    assert np.array_equal(to_np(a[0])[:na], to_np(b[0])[:na])


# ---------------------------------------------------------------------------------------------
# the FP16 kernels that cut their own tiles (3x3x3 layers from 16 channels up): with 16 and 32 input channels the one that keeps all
# weights in LDS (conv_tall.hip), from 64 up the ring of LDS buffers (conv_tile.hip); tile edges and tile heights
# ---------------------------------------------------------------------------------------------
def _fp16_subm_against_oracle(cin, cout, n, mv, grid, seed, clustered=True, epilogue=True):
    rng = np.random.default_rng(seed)
    coors = (F.clustered_active_voxels(n, grid, seed, n_blobs=max(4, n // 100)) if clustered
             else F.random_active_voxels(n, grid, seed))
    feat = O.round_to_half(rng.uniform(-1, 1, (n, cin)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32))
    sc = rng.uniform(0.5, 1.5, cout).astype(np.float32) if epilogue else None
    sh = rng.uniform(-0.2, 0.2, cout).astype(np.float32) if epilogue else None
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
    if epilogue:
        conv.set_epilogue(sc, sh, True)
    cbuf = np.zeros((mv, 4), np.int32)
    cbuf[:n] = coors
    fbuf = np.zeros((mv, cin), np.float32)
    fbuf[:n] = feat
    out = conv(dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32)), out_dtype=torch.float16)
    torch.cuda.synchronize()
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
    o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
    if epilogue:
        o_out = O.scale_shift_relu(o_out, mv, sc, sh, True)
    # every row of the tensor: rows >= n are the epilogue of zero (the reference zero-fills, then BN + ReLU)
    assert_features_close(to_np(out.float()), O.round_to_half(o_out), RTOL_FP16, "fp16 %d->%d, %d rows" % (cin, cout, n))
    conv.close()


@pytest.mark.parametrize("cin,cout", [(32, 32), (64, 64), (128, 128)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 300])
def test_fp16_kernels_row_counts_around_their_tiles(cin, cout, n):
    """A wave of the kernel with all weights in LDS has 16 rows (32 -> 32), a tile of the ring kernel 64 or 32 at these row counts:
    row counts on either side of a block and a tile, down to a single row, against the oracle (pad rows
    included)."""
    _fp16_subm_against_oracle(cin, cout, n, 512, (5, 40, 40), 900 + n, epilogue=(n % 2 == 1))


@pytest.mark.parametrize("cin,cout,n", [(32, 32, 66000), (64, 64, 40000), (64, 128, 66000), (128, 128, 40000), (128, 128, 66000)])
def test_fp16_kernels_with_many_rows(cin, cout, n):
    """Launches of many rows, the last tile partly filled, against the oracle on 16 threads: two or three blocks for a wave, one
    after the other with 32 channels, in one tile on the ring kernel."""
    O.set_threads(16)
    try:
        _fp16_subm_against_oracle(cin, cout, n, 66560, (21, 400, 352), 4000 + cin + cout)
    finally:
        O.set_threads(1)


@pytest.mark.parametrize("cout,n", [(32, 81920), (32, 81921), (32, 120000), (32, 163841), (64, 65536), (64, 65537), (64, 100000), (64, 131073)])
def test_fp16_kernel_with_all_weights_in_lds_whose_waves_walk_many_blocks(cout, n):
    """Launches of so many rows that every wave walks two to six blocks of 16, some a block more than others."""
    O.set_threads(16)
    try:
        _fp16_subm_against_oracle(32, cout, n, n + 70, (41, 400, 352), 8000 + cout)
    finally:
        O.set_threads(1)


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 32), (32, 64)])
@pytest.mark.parametrize("n", [1, 17, 4095, 8192, 8193, 16385, 32768, 32769, 33000, 66000])
def test_fp16_kernel_with_all_weights_in_lds(cin, cout, n):
    """On 256 compute units four waves share 16 rows up to 8 192 rows, two up to 16 384; from 32 769 on waves take a second block."""
    O.set_threads(16)
    try:
        _fp16_subm_against_oracle(cin, cout, n, n + 70 if n % 2 else n, (41, 400, 352), n + cout)
    finally:
        O.set_threads(1)


def _check_infinite_weight(conv, out, n_out, feat, w):
    """Column 2 of the rows with a neighbour at the weight's offset is infinite; everything else is what the oracle makes of the other
    weights and the layer's own rulebook."""
    pairs, num = (to_np(t) for t in conv.export_rulebook())
    (k,), mv = np.unique(np.nonzero(~np.isfinite(O.round_to_half(w)))[0]), len(feat)
    has = np.zeros(n_out, bool)
    has[pairs[k, 1, :num[k]]] = True
    assert has.any() and not has.all()
    assert not np.isnan(out).any() and np.array_equal(np.isinf(out[:n_out, 2]), has)
    finite = np.where(np.isfinite(O.round_to_half(w)), w, np.float32(0))
    O.set_threads(16)
    try:
        want = O.gather_gemm_scatter(feat, finite, pairs, num, mv)
        terms = O.gather_gemm_scatter(np.abs(feat), np.abs(finite), pairs, num, mv)
    finally:
        O.set_threads(1)
    got = out.copy()
    for v in (got, want, terms):
        v[:n_out][has, 2] = 0
    return got, want, terms


@pytest.mark.parametrize("cin,cout,half", [(16, 16, True), (16, 32, True), (32, 32, True), (32, 64, True), (64, 64, True), (64, 128, True),
                                           (128, 128, True), (4, 16, False), (16, 16, False)])
def test_an_infinite_weight_reaches_the_rows_that_have_the_neighbour(cin, cout, half):
    """... and makes no NaN of the others, whose absent neighbours are multiplied as rows of zeros where all weights are finite; the other
    columns are what they are without it."""
    rng = np.random.default_rng(cin + cout)
    grid, n, mv = (11, 200, 176), 9000, 9100
    coors = np.zeros((mv, 4), np.int32)
    coors[:n] = F.clustered_active_voxels(n, grid, 3, n_blobs=60)
    feat = O.round_to_half(rng.uniform(0.5, 1, (mv, cin)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32))
    w[5, 1, 2] = 1e6 if half else np.inf  # (infinite as a half)
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
    out = to_np(conv(dev(feat, torch.float16 if half else None), dev(coors), dev(np.array([n], np.int32))).float())
    got, want, terms = _check_infinite_weight(conv, out, n, feat, w)
    assert_features_close(got, O.round_to_half(want) if half else want, RTOL_FP16 if half else RTOL_FP32, "%d->%d beside an infinite weight" % (cin, cout),
                          abs_sum=terms, half=half)
    conv.close()


@pytest.mark.parametrize("channels", [64, 128])
def test_an_infinite_weight_of_the_last_layer_reaches_the_rows_that_have_the_neighbour(channels):
    """The same for the 3x1x1 layer that ends an FP16 backbone."""
    layer = SPARSE_LAYERS[3]
    ig = sparse_input_grid(layer)
    rng = np.random.default_rng(channels)
    n, mv = 9000, 18000
    coors = np.zeros((mv, 4), np.int32)
    coors[:n] = F.clustered_active_voxels(n, ig, 5, n_blobs=60)
    feat = O.round_to_half(rng.uniform(0.5, 1, (mv, channels)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (3, channels, channels)).astype(np.float32))
    w[1, 1, 2] = 1e6  # (infinite as a half)
    op = api.SparseConv3d(channels, channels, layer.out_shape, ig[::-1], layer.ksize, layer.stride, layer.padding, w, mv)
    out, _, num_out = op(dev(feat, torch.float16), dev(coors), dev(np.array([n], np.int32)))
    got, want, terms = _check_infinite_weight(op, to_np(out.float()), int(to_np(num_out)[0]), feat, w)
    assert_features_close(got, O.round_to_half(want), RTOL_FP16, "3x1x1 beside an infinite weight", abs_sum=terms, half=True)
    op.close()


@pytest.mark.parametrize("cin,cout,n", [(64, 64, 16384), (64, 64, 16385), (64, 64, 65537), (64, 64, 81920), (64, 64, 81921),
                                        (64, 128, 8193), (128, 128, 8192), (128, 128, 8193), (128, 128, 32769), (128, 128, 49152),
                                        (128, 128, 49153)])
def test_fp16_ring_kernel_around_the_row_counts_of_its_tile_heights(cin, cout, n):
    """On 256 compute units a tile of the LDS-ring kernel is 64 m rows high with 64 columns (m = 1 .. 5) and 32 m with 128
    (m = 1 .. 6), the smallest that makes the launch one round of tiles; beyond the tallest there are two rounds."""
    O.set_threads(16)
    try:
        _fp16_subm_against_oracle(cin, cout, n, n + 70, (21, 400, 352), 6000 + cin + cout)
    finally:
        O.set_threads(1)


@pytest.mark.parametrize("cin,cout,n", [(64, 64, 3060), (64, 64, 26247), (64, 64, 90000), (64, 128, 8193), (64, 128, 30000), (128, 128, 2833),
                                        (128, 128, 19825), (128, 128, 40422), (128, 128, 60000)])
def test_fp16_ring_kernel_gives_the_same_bits_launch_after_launch(cin, cout, n):
    """The ring's waits are counted by hand over requests that go straight to LDS: a wait that covered one request too few
    would show in a few tiles out of many launches.  1200 launches per shape, half of them while copies on another
    stream load the memory; every output word against the first launch's."""
    grid = (21, 400, 352)
    coors = F.clustered_active_voxels(n, grid, 7100 + n, n_blobs=max(4, n // 100))
    rng = np.random.default_rng(n)
    cbuf = np.zeros((n, 4), np.int32)
    cbuf[:, :] = coors
    feat = dev(rng.uniform(-1, 1, (n, cin)).astype(np.float32), torch.float16)
    args = (feat, dev(cbuf), dev(np.array([n], np.int32)))
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, n)
    first = conv(*args).view(torch.int16)
    op = api.SubmConv3d(cin, cout, grid[::-1], w, n)
    bad = torch.zeros((), dtype=torch.int64, device="cuda:0")
    other, (a, b) = torch.cuda.Stream(), torch.zeros((2, 32 << 20), dtype=torch.uint8, device="cuda:0")
    torch.cuda.synchronize()
    for i in range(1200):
        if i >= 600 and i % 3 == 0:
            with torch.cuda.stream(other):
                b.copy_(a)
        bad += (op(*args, rulebook_from=conv).view(torch.int16) != first).sum()
    torch.cuda.synchronize()
    assert int(bad) == 0


@pytest.mark.parametrize("channels,n", [(64, 5000), (64, 40000), (128, 20000)])
def test_fp16_ring_kernel_of_the_last_layer_gives_the_same_bits_launch_after_launch(channels, n):
    """The same for the 3x1x1 layer that ends the backbone, whose whole walk is three offsets: 400 calls, each with its
    rulebook built anew."""
    layer = SPARSE_LAYERS[3]
    ig = sparse_input_grid(layer)
    coors = F.clustered_active_voxels(n, ig, 7300 + n, n_blobs=n // 100)
    rng = np.random.default_rng(n)
    cbuf = np.zeros((n, 4), np.int32)
    cbuf[:, :] = coors
    args = (dev(rng.uniform(-1, 1, (n, channels)).astype(np.float32), torch.float16), dev(cbuf), dev(np.array([n], np.int32)))
    w = rng.normal(0, 0.1, (3, channels, channels)).astype(np.float32)
    op = api.SparseConv3d(channels, channels, layer.out_shape, ig[::-1], layer.ksize, layer.stride, layer.padding, w, n)
    first, fc, fn = op(*args)
    bad = torch.zeros((), dtype=torch.int64, device="cuda:0")
    for _ in range(400):
        out, oc, on = op(*args)
        bad += (out.view(torch.int16) != first.view(torch.int16)).sum() + (oc != fc).sum() + (on != fn).sum()
    torch.cuda.synchronize()
    assert int(bad) == 0 and int(fn[0]) > 0


# ---------------------------------------------------------------------------------------------
# the FP32 kernel (conv_wide.hip)
# ---------------------------------------------------------------------------------------------
def _fp32_subm_wide_against_oracle(n, mv, grid, seed, clustered=True, epilogue=True, threads=1, cin=64):
    rng = np.random.default_rng(seed)
    coors = (F.clustered_active_voxels(n, grid, seed, n_blobs=max(4, n // 100)) if clustered
             else F.random_active_voxels(n, grid, seed))
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, 64)).astype(np.float32)
    sc = rng.uniform(0.5, 1.5, 64).astype(np.float32) if epilogue else None
    sh = rng.uniform(-0.2, 0.2, 64).astype(np.float32) if epilogue else None
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv, sc, sh, epilogue)
    O.set_threads(threads)
    try:
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
    finally:
        O.set_threads(1)
    assert np.array_equal(num, o_num)
    if epilogue:
        o_out = O.scale_shift_relu(o_out, mv, sc, sh, True)
    # every row of the tensor: rows >= n are the epilogue of zero (the reference zero-fills, then BN + ReLU)
    assert_features_close(out, o_out, RTOL_FP32, "wide fp32 %d->64, %d rows" % (cin, n),
                          abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv, sc, sh))
    assert conv.status() == 0
    conv.close()


@pytest.mark.parametrize("cin", [64, 32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 95, 96, 97, 255, 256, 257, 1000])
def test_wide_fp32_kernel_row_counts_around_its_tiles(n, cin):
    """Few rows: tiles of one row to eight on 256 compute units, fewer rows than tiles, as many, and one more; two workgroups share
    the columns of each.  (Tiles whose lists fill their two halves of 64 rows are in the tests below.)  Against the oracle (pad rows
    included)."""
    _fp32_subm_wide_against_oracle(n, n + 200, (5, 40, 40), 700 + n, epilogue=(n % 2 == 1), cin=cin)


@pytest.mark.parametrize("n,clustered,cin", [(20000, True, 64), (20000, True, 32), (24577, False, 64), (50000, True, 64)])
def test_wide_fp32_kernel_tall_tiles_and_two_tiles_per_workgroup(n, clustered, cin):
    """~78-row tiles (20 000 rows: both staging halves in use), the first row count past one 96-row tile per
    compute unit (24 577 rows of scattered voxels: every workgroup walks two tiles), and 50 000 clustered rows
    (tiles of uneven length from the equal-work cuts, two or three per workgroup), against the oracle on 16
    threads."""
    _fp32_subm_wide_against_oracle(n, 51200, (21, 400, 352), 5000 + n, clustered=clustered, threads=16, cin=cin)


@pytest.mark.parametrize("cin", [64, 32])
@pytest.mark.parametrize("n", [3071, 3072, 3073, 7679, 7680, 7681, 9599, 9600, 9601, 10239, 10240, 10241])
def test_wide_fp32_kernel_around_the_row_counts_of_its_column_splits(n, cin):
    """On 256 compute units the columns of a tile are dealt to two workgroups up to 9 600 rows."""
    _fp32_subm_wide_against_oracle(n, n + 7, (11, 200, 176), 900 + n, threads=8, cin=cin)


@pytest.mark.parametrize("cin,cout", [(64, 64), (128, 128)])
@pytest.mark.parametrize("per_unit", [37, 38, 72, 73, 82, 83, 96, 97])
def test_wide_fp32_kernel_around_its_numbers_of_waves(per_unit, cin, cout):
    """64 columns: eight waves multiply a tile of up to 72 rows, seven one of up to 82, six one of up to 96; up to 75 rows for two units
    (37 a unit) these share a tile.  A solid block of voxels (equal tiles) of that many rows for each of 256 units, and half of it
    solid with the rest scattered, whose tiles are several times as long as the others and walked in pieces, against the oracle (pad
    rows included)."""
    n = 256 * per_unit * 64 // cout
    rng = np.random.default_rng(n + cout)
    grid, mv = (21, 400, 352), n + 5
    side = int(np.ceil((n / 16) ** 0.5))
    z, y, x = (a.ravel() for a in np.meshgrid(np.arange(16), np.arange(side), np.arange(side), indexing="ij"))
    solid = np.stack([np.zeros_like(z), z, y, x], 1)[:n].astype(np.int32)
    z, y, x = (a.ravel() for a in np.meshgrid(np.arange(1, 21, 2), np.arange(200, 400, 2), np.arange(1, 352, 2), indexing="ij"))
    far = np.stack([np.zeros_like(z), z, y, x], 1).astype(np.int32)
    mixed = np.concatenate([solid[:n // 2], far[rng.permutation(len(far))[:n - n // 2]]])
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    sc, sh = rng.uniform(0.5, 1.5, cout).astype(np.float32), rng.uniform(-0.2, 0.2, cout).astype(np.float32)
    for coors in (solid, mixed):
        conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv, sc, sh, True)
        O.set_threads(16)
        try:
            o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
            o_out = O.scale_shift_relu(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), mv, sc, sh, True)
        finally:
            O.set_threads(1)
        assert np.array_equal(num, o_num)
        assert_features_close(out, o_out, RTOL_FP32, "wide fp32 %d->%d, %d rows" % (cin, cout, n),
                              abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv, sc, sh))
        assert conv.status() == 0
        conv.close()


@pytest.mark.parametrize("cin,cout,half", [(16, 32, False), (64, 64, False), (32, 64, False), (128, 128, False), (16, 16, True),
                                           (32, 64, True), (64, 64, True), (128, 128, True)])
def test_every_row_is_a_pad_row(cin, cout, half):
    """No active row: all workgroups of a gather-GEMM only write relu(shift), in each kernel, at row counts that do not
    divide by anything the kernels count in."""
    rng = np.random.default_rng(cin + cout)
    sh = rng.uniform(-0.5, 0.5, cout).astype(np.float32)
    for mv in (1, 257, 40003):
        conv = api.SubmConv3d(cin, cout, (40, 40, 5), rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32), mv)
        conv.set_epilogue(np.ones(cout, np.float32), sh, relu=True)
        feat = dev(np.ones((mv, cin), np.float16 if half else np.float32))
        y = conv(feat, dev(np.zeros((mv, 4), np.int32)), dev(np.array([0], np.int32)))
        torch.cuda.synchronize()
        want = np.maximum(sh, 0).astype(np.float16 if half else np.float32)
        assert np.array_equal(to_np(y), np.broadcast_to(want, (mv, cout))), mv
        conv.close()


@pytest.mark.parametrize("cin,cout,half", [(4, 16, False), (16, 32, False), (32, 32, False), (64, 64, False), (128, 128, False), (16, 16, True),
                                           (32, 32, True), (32, 64, True), (64, 64, True), (128, 128, True)])
def test_pad_rows_beside_the_products(cin, cout, half):
    """Rows beyond the active ones are written while a launch multiplies: one of them, fewer than the launch has waves, more than it has
    steps for, and none left for the workgroups without a tile.  The active rows come out as in a tensor with none or few, bit for bit."""
    rng = np.random.default_rng(cin + cout)
    grid = (11, 200, 176)
    coors = F.clustered_active_voxels(12000, grid, 1, n_blobs=60)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    sc, sh = rng.uniform(0.5, 1.5, cout).astype(np.float32), rng.uniform(-0.5, 0.5, cout).astype(np.float32)
    dtype = np.float16 if half else np.float32
    feat = rng.uniform(0, 1, (12000, cin)).astype(dtype)

    def rows(n, mv):
        conv = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
        conv.set_epilogue(sc, sh, relu=True)
        f, c = np.zeros((mv, cin), dtype), np.zeros((mv, 4), np.int32)
        f[:n], c[:n] = feat[:n], coors[:n]
        y = to_np(conv(dev(f), dev(c), dev(np.array([n], np.int32))))
        conv.close()
        return y

    for n, more in ((1, 1), (639, 1), (640, 3), (640, 131), (12000, 1), (12000, 9000), (300, 150000)):
        y = rows(n, n + more)
        few = n if n + more <= 8192 else max(n, 8193)  # (beyond 8 192 rows a rulebook has cuts, by which sums are ordered)
        assert np.array_equal(y[:n], rows(n, few)[:n]), (n, more)
        assert np.array_equal(y[n:], np.broadcast_to(np.maximum(sh, 0).astype(dtype), (more, cout))), (n, more)


@pytest.mark.parametrize("cin", [64, 128])
@pytest.mark.parametrize("n", [1, 65, 97, 1536, 1537, 3840, 3841, 5120, 5121, 12289, 20000])
def test_wide_fp32_kernel_with_128_columns(n, cin):
    """128 output columns: two workgroups take 64 columns each of every tile (128 tiles a round on 256 compute units, of
    up to 96 rows), up to 4 800 rows four; 128 input channels are walked in two parts.  Against
    the oracle (pad rows included)."""
    rng = np.random.default_rng(n + cin)
    grid, mv = ((5, 40, 40) if n < 1000 else (21, 400, 352)), n + 39
    coors = F.clustered_active_voxels(n, grid, n, n_blobs=max(4, n // 100))
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, 128)).astype(np.float32)
    sc, sh = rng.uniform(0.5, 1.5, 128).astype(np.float32), rng.uniform(-0.2, 0.2, 128).astype(np.float32)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv, sc, sh, True)
    O.set_threads(16)
    try:
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        o_out = O.scale_shift_relu(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), mv, sc, sh, True)
    finally:
        O.set_threads(1)
    assert np.array_equal(num, o_num)
    assert_features_close(out, o_out, RTOL_FP32, "wide fp32 %d->128, %d rows" % (cin, n),
                          abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv, sc, sh))
    conv.close()


def _fp32_subm_with_few_columns_against_oracle(n, cin, cout):
    rng = np.random.default_rng(n + cin)
    grid, mv = ((5, 40, 40) if n < 1000 else (21, 400, 352)), n + 39
    coors = F.clustered_active_voxels(n, grid, n, n_blobs=max(4, n // 100))
    feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    sc, sh = rng.uniform(0.5, 1.5, cout).astype(np.float32), rng.uniform(-0.2, 0.2, cout).astype(np.float32)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, mv, sc, sh, True)
    O.set_threads(16)
    try:
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        o_out = O.scale_shift_relu(O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv), mv, sc, sh, True)
    finally:
        O.set_threads(1)
    assert np.array_equal(num, o_num)
    assert_features_close(out, o_out, RTOL_FP32, "fp32 %d->%d, %d rows" % (cin, cout, n),
                          abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv, sc, sh))
    conv.close()


@pytest.mark.parametrize("cin,cout", [(4, 16), (4, 32), (16, 16), (16, 32), (32, 32)])
@pytest.mark.parametrize("n", [1, 16, 63, 65, 113, 129, 16385, 28672, 28673, 40000])
def test_wide_fp32_kernel_with_few_columns(n, cin, cout):
    """16 and 32 output columns: few rows, row counts around a tile's, and some thousands.  Against the oracle (pad rows included)."""
    _fp32_subm_with_few_columns_against_oracle(n, cin, cout)


@pytest.mark.parametrize("cin,cout,rows,groups", [(4, 16, 128, 2), (16, 16, 128, 2), (4, 32, 64, 4), (16, 32, 64, 2), (32, 32, 80, 3)])
def test_wide_fp32_kernel_around_its_workgroups_per_compute_unit(cin, cout, rows, groups):
    """16 and 32 output columns: one workgroup per compute unit while tiles of `rows` rows hold the layer, up to `groups` beyond, then a
    second round of tiles: the row counts on both sides of each of these lines.  Against the oracle (pad rows included)."""
    units = torch.cuda.get_device_properties(0).multi_processor_count
    for held in range(1, groups + 1):
        for n in (units * rows * held, units * rows * held + 1):
            _fp32_subm_with_few_columns_against_oracle(n, cin, cout)


@pytest.mark.parametrize("cout", [16, 32])
@pytest.mark.parametrize("n", [1, 63, 65, 16383, 16385, 40000, 65537])
def test_fp16_kernel_with_16_channels(n, cout):
    """FP16, 16 input channels: tiles of up to 64 rows, one to four workgroups per compute unit (16 384 rows each on 256 units),
    a second round of tiles beyond 65 536 rows.  Against the oracle (pad rows included), one rounding to half apart."""
    rng = np.random.default_rng(n + cout)
    grid, mv = ((5, 40, 40) if n < 1000 else (21, 400, 352)), n + 39
    coors = F.clustered_active_voxels(n, grid, n, n_blobs=max(4, n // 100))
    feat = O.round_to_half(rng.uniform(-1, 1, (n, 16)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (27, 16, cout)).astype(np.float32))
    cbuf, fbuf = np.zeros((mv, 4), np.int32), np.zeros((mv, 16), np.float32)
    cbuf[:n], fbuf[:n] = coors, feat
    conv = api.SubmConv3d(16, cout, grid[::-1], w, mv)
    out = conv(dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32)), out_dtype=torch.float16)
    torch.cuda.synchronize()
    O.set_threads(16)
    try:
        o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], mv)
        o_out = O.gather_gemm_scatter(feat, w, o_pairs, o_num, mv)
    finally:
        O.set_threads(1)
    assert_features_close(to_np(out.float()), O.round_to_half(o_out), RTOL_FP16, "fp16 16->%d, %d rows" % (cout, n), half=True,
                          abs_sum=abs_sum_of(feat, w, o_pairs, o_num, mv, mv))
    conv.close()


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128)])
@pytest.mark.parametrize("k", [(1, 1, 1), (1, 1, 2), (3, 2, 1), (1, 3, 3), (2, 3, 3)])
@pytest.mark.parametrize("n", [1, 97, 6000, 17000])
def test_fp16_kernel_with_pair_lists_whatever_the_kernel_volume(n, k, cin, cout):
    """FP16 layers whose kernel volume is neither 27 nor 3 run on the kernel with pair lists: fewer offsets than waves, more than it
    splits columns from (18), one row, more than a tile, tiles split and not."""
    rng = np.random.default_rng([n, cin, cout, k[0] * 9 + k[1] * 3 + k[2]])
    ig, st, p = (9, 70, 60), (1, 1, 1), tuple(v // 2 for v in k)
    og = tuple(B.conv_out_size(ig[a], k[a], st[a], p[a]) for a in range(3))
    coors = F.random_active_voxels(n, ig, n)
    mv = min(n * k[0] * k[1] * k[2], og[0] * og[1] * og[2]) + 50
    feat = O.round_to_half(rng.uniform(-1, 1, (n, cin)).astype(np.float32))
    w = O.round_to_half(rng.normal(0, 0.1, (k[0] * k[1] * k[2], cin, cout)).astype(np.float32))
    cbuf, fbuf = np.zeros((mv, 4), np.int32), np.zeros((mv, cin), np.float32)
    cbuf[:n], fbuf[:n] = coors, feat
    conv = api.SparseConv3d(cin, cout, og[::-1], ig[::-1], k, st, p, w, mv)
    out, oc, on = conv(dev(fbuf, torch.float16), dev(cbuf), dev(np.array([n], np.int32)))
    O.set_threads(16)
    try:
        pairs, num, o_oc, o_on, status = O.sparse_rulebook(coors, n, og[::-1], k, st, p, mv)
        want, A = O.gather_gemm_scatter(feat, w, pairs, num, mv), abs_sum_of(feat, w, pairs, num, mv)
    finally:
        O.set_threads(1)
    assert int(to_np(on)[0]) == o_on and np.array_equal(to_np(oc), o_oc) and conv.status() == status
    assert_features_close(to_np(out.float()), O.round_to_half(want), RTOL_FP16, "fp16 %s %d->%d, %d rows" % (k, cin, cout, n), half=True,
                          abs_sum=A)
    conv.close()


@pytest.mark.parametrize("cin,cout,half", [(4, 16, False), (16, 16, False), (16, 32, True)])
def test_kernel_with_few_channels_in_a_tensor_of_more_than_2_to_the_24_rows(cin, cout, half):
    """Every cell of a grid of 16 785 408, in the order of its cells: the last two lines in y, whose rows and neighbours lie beyond
    row 2^24, against the dense convolution in 64 bits."""
    grid = (4, 2049, 2048)
    n = grid[0] * grid[1] * grid[2]
    dt = torch.float16 if half else torch.float32
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(cin + cout)
    feat = (torch.rand((n, cin), generator=gen, device="cuda:0") - 0.5).to(dt)
    cell = torch.arange(n, dtype=torch.int32, device="cuda:0")
    coors = torch.stack([torch.zeros_like(cell), cell // (grid[1] * grid[2]), cell // grid[2] % grid[1], cell % grid[2]], 1).contiguous()
    rng = np.random.default_rng(cout)
    w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
    if half:
        w = O.round_to_half(w)
    conv = api.SubmConv3d(cin, cout, grid[::-1], w, n)
    out = conv(feat, coors, dev(np.array([n], np.int32)), out_dtype=dt)
    assert conv.status() == 0
    got = out.view(*grid, cout)[3, -2:].cpu().double()
    x = feat.view(*grid, cin)[2:, -3:].cpu().double().permute(3, 0, 1, 2)[None]
    k = torch.as_tensor(w).double().view(3, 3, 3, cin, cout).permute(4, 3, 0, 1, 2)
    want, A = (torch.nn.functional.conv3d(f(x), f(k), padding=1)[0, :, 1, 1:].permute(1, 2, 0) for f in (lambda t: t, torch.abs))
    assert torch.all((got - want).abs() <= 2e-6 * A + (2.0 ** -10 * want.abs() + 2.0 ** -24 if half else 0.0))
    conv.close()


def _sums_in_64_bits(feat, w, pairs, num, n):
    with np.errstate(all="ignore"):
        out = np.zeros((n, w.shape[2]))
        for k in range(w.shape[0]):
            i, o = pairs[k, 0, :num[k]], pairs[k, 1, :num[k]]
            out[o] += (feat[i].astype(np.float64)[:, :, None] * w[k].astype(np.float64)[None]).sum(1)
    return out


@pytest.mark.parametrize("cin,cout", [(16, 32), (32, 32), (32, 64), (64, 64), (128, 128)])
@pytest.mark.parametrize("lo,hi", [(-60, 60), (-110, -90), (60, 90)])
def test_wide_fp32_kernel_keeps_32_bits_whatever_the_magnitude(cin, cout, lo, hi):
    """Whole rows and whole columns of W of very different magnitude (channels: the test below): the kernel multiplies 16-bit
    parts of the operands.  Bound: 27 * Cin terms of which each side is off by at most one unit in the last place of its
    operands (2^-23 each) and of its sum: SUM_TOL times the sum of the terms' magnitudes, as everywhere in these tests."""
    rng = np.random.default_rng([cin, lo + 200])
    n, grid = 300, (5, 20, 20)
    coors = F.clustered_active_voxels(n, grid, 3, n_blobs=4)
    feat = (rng.uniform(-1, 1, (n, cin)) * 2.0 ** rng.integers(lo, hi, (n, 1))).astype(np.float32)
    w = (rng.normal(0, 0.1, (27, cin, cout)) * 2.0 ** rng.integers(-20, 20, (1, 1, cout))).astype(np.float32)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, n, None, None, False)
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], n)
    want = _sums_in_64_bits(feat, w, o_pairs, o_num, n)
    A = _sums_in_64_bits(np.abs(feat), np.abs(w), o_pairs, o_num, n)
    assert np.all(np.abs(out[:n] - want) <= 2e-6 * A + 2.0 ** -126)
    conv.close()


def _magnitudes_along_channels(kind, n, cin, cout, rng):
    feat = rng.uniform(0.5, 1, (n, cin)) * rng.choice([-1, 1], (n, cin))
    w = rng.uniform(0.5, 1, (27, cin, cout)) * rng.choice([-1, 1], (27, cin, cout))
    if kind[0] == "opposed":  # products all alike
        s = rng.integers(-kind[1], kind[1] + 1, cin)
        s[:2] = kind[1], -kind[1]
        feat *= 2.0 ** s
        w *= 2.0 ** -s[:, None]
    elif kind[0] == "unused":  # a channel without weights
        feat[:, cin // 2], w[:, cin // 2] = kind[1], 0.0
        feat[::2, 1], w[:, 1] = kind[1], 0.0
    elif kind[0] == "small rows":  # features of 2^-100 down to the smallest subnormal numbers
        feat *= 2.0 ** rng.integers(-148, -100, (n, cin))
        feat[:, 0] *= 2.0 ** 30
        w *= 2.0 ** 60
    else:  # small weights, in columns with larger ones beside them and without
        feat *= 2.0 ** 70
        w *= 2.0 ** rng.integers(-148, -100, (27, cin, cout))
        w[:, 0, ::2] *= 2.0 ** 90
        feat[::3, 0] = 0.0
    return feat.astype(np.float32), w.astype(np.float32)


@pytest.mark.parametrize("cin,cout", [(32, 32), (32, 64), (64, 64), (64, 128), (128, 128)])
@pytest.mark.parametrize("kind", [("opposed", 12), ("opposed", 20), ("opposed", 40), ("unused", 1e8), ("unused", 1e12),
                                  ("unused", float(np.finfo(np.float32).min)), ("small rows", 0), ("small weights", 0)], ids=str)
def test_wide_fp32_kernel_keeps_every_channel_whatever_the_magnitude_of_others(cin, cout, kind):
    """Channels of a row, and elements of a column of W, of very different magnitude: an element keeps its bits beside larger
    ones.  The bound is that of the rows and columns of different magnitude above."""
    rng = np.random.default_rng([cin, cout, len(kind[0])])
    n, grid = 300, (5, 20, 20)
    coors = F.clustered_active_voxels(n, grid, 3, n_blobs=4)
    feat, w = _magnitudes_along_channels(kind, n, cin, cout, rng)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, n, None, None, False)
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], n)
    want = _sums_in_64_bits(feat, w, o_pairs, o_num, n)
    A = _sums_in_64_bits(np.abs(feat), np.abs(w), o_pairs, o_num, n)
    worst = float((np.abs(out[:n] - want) / np.maximum(A, 2.0 ** -100)).max())
    assert np.all(np.abs(out[:n] - want) <= 2e-6 * A + 2.0 ** -126), "worst difference %.3g of the sum of |terms|" % worst
    conv.close()


@pytest.mark.parametrize("cin,cout", [(4, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128)])
def test_wide_fp32_kernel_infinities_and_nan(cin, cout):
    """An infinity, a NaN and finite values whose products overflow reach the outputs that plain FP32 sums would make of them,
    and no others."""
    rng = np.random.default_rng(cin * cout)
    n, grid = 400, (5, 30, 30)
    coors = F.clustered_active_voxels(n, grid, 5, n_blobs=8)
    feat = rng.uniform(0.5, 1, (n, cin)).astype(np.float32)
    w = rng.uniform(0.5, 1, (27, cin, cout)).astype(np.float32) * rng.choice([-1, 1], (27, 1, cout)).astype(np.float32)
    feat[10, 1], feat[60, 3], feat[150, 0] = np.inf, -np.inf, np.nan
    feat[250] = np.finfo(np.float32).max  # (times a weight of half and more, Cin times: beyond the range, of one sign per offset)
    conv, out, pairs, num, cbuf = run_subm(coors, n, feat, w, grid, n, None, None, False)
    o_pairs, o_num, _ = O.subm_rulebook(coors, n, grid[::-1], n)
    want = _sums_in_64_bits(feat, w, o_pairs, o_num, n)
    out = out[:n]
    assert np.array_equal(np.isnan(out), np.isnan(want))
    big = ~np.isnan(want) & (np.abs(want) > 3.5e38)  # (infinities and sums beyond the range)
    assert big.sum() > cout and np.array_equal(out[big], np.where(want[big] > 0, np.inf, -np.inf))
    rest = ~np.isnan(want) & (np.abs(want) < 1e30)
    A = _sums_in_64_bits(np.abs(feat), np.abs(w), o_pairs, o_num, n)
    assert rest.sum() > n and np.all(np.abs(out[rest] - want[rest]) <= 2e-6 * A[rest])
    conv.close()
