"""The first layers of a frame, whose products share launches with the passes over coordinates, and the FP32 kernel that they and the
plugins run on: every layer against the oracle at the row counts where the split of the work changes."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from gpu_util import RTOL_FP32, abs_sum_of, assert_features_close, check_frame_against_oracle, dev, points_input, to_np
from sessd3d import api, backbone as B, ctypes_defs as D, frames as F

pytestmark = pytest.mark.gpu

S, P = D.SESSD_LAYER_SUBM, D.SESSD_LAYER_SPARSE
FULL = (1408, 1600, 41)


def strided(cin, *couts):
    """Strided layers down to the dense tensor's grid."""
    shapes = [((704, 800, 21), (2, 2, 2), (1, 1, 1)), ((352, 400, 11), (2, 2, 2), (1, 1, 1)), ((176, 200, 5), (2, 2, 2), (0, 1, 1))]
    layers = []
    for (grid, s, p), cout in zip(shapes, couts):
        layers.append(B.Layer("sparse%d" % len(layers), P, cin, cout, grid, (3, 3, 3), s, p))
        cin = cout
    return layers + [B.Layer("last", P, cin, cin, (176, 200, 2), (3, 1, 1), (2, 1, 1), (0, 0, 0))]


def subm(cin, cout, grid=FULL):
    return B.Layer("subm%dx%d" % (cin, cout), S, cin, cout, grid)


BACKBONES = {
    "one": [subm(4, 16)] + strided(16, 32, 64, 64),                                # pass 2 alone
    "two": [subm(4, 16), subm(16, 16)] + strided(16, 32, 64, 64),                  # passes 1 and 2 with a layer each
    "three": [subm(4, 16), subm(16, 16), subm(16, 16)] + strided(16, 32, 64, 64),  # a layer behind them
    "wide": [subm(4, 32), subm(32, 32)] + strided(32, 64, 64, 64),                 # FP16 as "two"; FP32 on one stream pass 1 with a layer
    "own grid": [subm(4, 16), subm(16, 16, (1409, 1600, 41))] + strided(16, 32, 64, 64),
}


def points_in(cells, seed):
    """A point in the middle of so many distinct cells near each other."""
    rng = np.random.default_rng(seed)
    side = (8, max(4, int((cells / 2.5) ** 0.5)), max(4, int((cells / 2.5) ** 0.5)))
    at = rng.choice(side[0] * side[1] * side[2], cells, replace=False)
    zyx = np.stack(np.unravel_index(at, side), 1) + (4, 300, 200)
    pts = np.zeros((cells, 4), np.float32)
    pts[:, :3] = np.float32(B.POINT_CLOUD_RANGE)[:3] + (zyx[:, ::-1] + 0.5) * np.float32(B.VOXEL_SIZE)
    pts[:, 3] = rng.random(cells)
    return pts


@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("name", ["one", "two", "three", "wide", "own grid"])
def test_layers_that_share_launches_with_passes(name, dtype):
    """Per-layer tolerance of the suite: features 1e-4 (FP16: 1e-2) of each element, cancelling sums by their terms."""
    layers, half, cap = BACKBONES[name], dtype == "fp16", 20480
    W = B.random_weights(layers, seed=4, w_std=0.1)
    if half:
        W = B.Weights([O.round_to_half(w) for w in W.w], W.scale, W.shift)
    # 16 rows a block, a block for four waves up to 256 blocks, for two up to 512
    sizes = [1, 17, 4096, 4097, 8193] if name in ("two", "wide") else [16, 4097]
    for i, cells in enumerate(sizes):
        schedule = dict(use_graph=True, overlap_streams=True) if i % 2 == 0 else dict(overlap_streams=i % 4 == 1)
        pipe = api.Pipeline(layers, W, 10000, cap, feature_dtype=dtype, share_rulebooks=True, skip_pad_rows=False, **schedule)
        pts = points_in(cells, 7 + i)
        p, n = points_input(pts, 10000)
        dense, stream = pipe.new_dense(), torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(3):  # (the tables are left as the next frame needs them)
                pipe.enqueue(p, n, dense, stream)
        stream.synchronize()
        assert pipe.layer_count(0) == cells
        check_frame_against_oracle(pipe, dense, pts, layers, W, cap, cap, half, B.DENSE_SIZE_XYZ)
        for l in (0, 1):  # rows beyond the active ones: relu(0 x scale + shift)
            f, _, _, _, ch = pipe.layer_io(l)
            rows = np.zeros((cap, ch), np.float16 if half else np.float32)
            api._hip_d2h(rows, f)
            shift = np.maximum(W.shift[l], 0).astype(rows.dtype)
            assert (rows[pipe.layer_count(l):] == shift).all(), (cells, l)


@pytest.mark.parametrize("name,dtype", [("two", "fp32"), ("two", "fp16"), ("wide", "fp16")])
@pytest.mark.parametrize("cells", [16385, 40000])
def test_layers_that_share_launches_with_passes_in_several_rounds(name, dtype, cells):
    """A workgroup of these launches has four waves of 16 rows: with more than 16 384 rows on 256 units it goes on to a second round, with 40 000 to
    a third.  Tensors for 50 000 points."""
    layers, half, cap = BACKBONES[name], dtype == "fp16", 45000
    W = B.random_weights(layers, seed=5, w_std=0.1)
    if half:
        W = B.Weights([O.round_to_half(w) for w in W.w], W.scale, W.shift)
    pipe = api.Pipeline(layers, W, 50000, cap, feature_dtype=dtype, share_rulebooks=True, skip_pad_rows=False, use_graph=True, overlap_streams=True)
    pts = points_in(cells, cells)
    p, n = points_input(pts, 50000)
    dense, stream = pipe.new_dense(), torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(3):
            pipe.enqueue(p, n, dense, stream)
    stream.synchronize()
    assert pipe.layer_count(0) == cells
    check_frame_against_oracle(pipe, dense, pts, layers, W, cap, cap, half, B.DENSE_SIZE_XYZ)


@pytest.mark.parametrize("pad", [False, True])
@pytest.mark.parametrize("cin,cout", [(4, 16), (4, 32), (16, 16)])
def test_fp32_layers_with_few_channels(cin, cout, pad):
    """FP32 3x3x3 layers with all weights in LDS: the orders of sums and the last rows of a block.  1e-4 of an element, and in the norm, with
    thousands of rows, no further from 64-bit sums than the oracle's, which adds each offset's products by themselves: here 0.76 to 0.93 of its
    distance, one chain over all products 1.06 to 2.6 from 8 193 rows up, a chain for each channel of a piece 1.18 and 1.34 with 16 channels and
    16 401 and 30 000 rows."""
    rng = np.random.default_rng(cin * cout)
    grid = (12, 60, 70)
    for n in (1, 16, 31, 8192, 8193, 16384, 16401, 30000):
        mv = max(n + 40, 8200) if pad else max(n, 8200)
        coors = F.random_active_voxels(n, grid, n)
        feat = rng.uniform(-1, 1, (n, cin)).astype(np.float32)
        w = rng.normal(0, 0.1, (27, cin, cout)).astype(np.float32)
        op = api.SubmConv3d(cin, cout, grid[::-1], w, mv)
        op.set_flags(0 if pad else D.SESSD_FLAG_SKIP_PAD_ROWS)
        fbuf, cbuf = np.zeros((mv, cin), np.float32), np.zeros((mv, 4), np.int32)
        fbuf[:n], cbuf[:n] = feat, coors
        out = to_np(op(dev(fbuf), dev(cbuf), dev(np.array([n], np.int32))))
        pairs, num, _ = O.subm_rulebook(cbuf, n, grid[::-1], mv)
        want = O.gather_gemm_scatter(fbuf, w, pairs, num, mv)[:n]
        assert_features_close(out[:n], want, RTOL_FP32, "%d rows" % n, abs_sum=abs_sum_of(fbuf, w, pairs, num, mv)[:n])
        exact = sums_in_64_bits(feat, w, pairs, num, n)
        assert np.linalg.norm(out[:n] - exact) <= (1 if n > 1000 else 2) * np.linalg.norm(want - exact) + 1e-30
        if pad:
            assert not out[n:].any()


def sums_in_64_bits(feat, w, pairs, num, n):
    """The same sums in 64 bits."""
    out = np.zeros((n, w.shape[2]))
    for k in range(27):
        i, o = pairs[k][0][:num[k]], pairs[k][1][:num[k]]
        np.add.at(out, o, feat[i].astype(np.float64) @ w[k].astype(np.float64))
    return out
