"""The matrix-core screen of the hypothesis scorers: counts bit-equal to the
CPU restatement of the exact test, at the edges of its tiles, chunks and
workgroups, on data with many tests near the threshold, and on coordinates its
bound does not cover (which take the exact loop). Counts are whole numbers:
no tolerance."""
import numpy as np
import pytest
import torch

from tests.scenes import plane_scene

pytestmark = pytest.mark.gpu


def _dev(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32) if a.dtype == np.uint32 else a).to(dev)


def _idx(n, H, k, seed):
    rng = np.random.default_rng(seed)
    return np.stack([rng.choice(n, k, replace=False) for _ in range(H)]).astype(np.uint32)


def _check(orc, dev, pts, H, mode, t, seed, kind):
    from rapidsfm_amd import ops

    print("[case] screen", kind, pts.shape[0], H, mode, t, flush=True)
    k, fn, ref = (8, ops.ransac_f8, orc.f8_score) if kind == "f8" else (7, ops.ransac_f7, orc.f7_score)
    idx = _idx(pts.shape[0], H, k, seed)
    (o,) = fn([(_dev(pts, dev), _dev(idx, dev))], t, mode=mode)
    c, _ = ref(pts, idx, t, mode, nthreads=8)
    assert np.array_equal(o["counts"].cpu().numpy().view(np.uint32), c)


# one point short of / at / past a 16-point tile and a staged chunk of both
# workgroup shapes, hypothesis counts around a workgroup's
@pytest.mark.parametrize("kind", ["f8", "f7"])
@pytest.mark.parametrize("mode,t", [(0, 2.0), (1, 1.0)])
@pytest.mark.parametrize("n,H", [(8, 1), (15, 63), (16, 64), (17, 65), (127, 128), (128, 129), (129, 200), (257, 16), (513, 300)])
def test_edges(orc, dev, kind, mode, t, n, H):
    pts, _, _, _ = plane_scene(n, n // 3, n // 3 + 1, n - n // 3 - n // 3 - 1, noise=0.5)
    _check(orc, dev, pts, H, mode, t, n + H, kind)


# nearly all inliers with the threshold at the noise: many open tests per chunk
@pytest.mark.parametrize("kind", ["f8", "f7"])
@pytest.mark.parametrize("mode,t", [(0, 0.6), (1, 0.6), (0, 9.6)])
def test_many_open(orc, dev, kind, mode, t):
    pts, _, _, _ = plane_scene(5, 100, 1400, 20, noise=0.5)
    _check(orc, dev, pts, 400, mode, t, 11, kind)


# several pairs at once, enough of them for the 256-hypothesis workgroups
@pytest.mark.parametrize("mode", [0, 1])
def test_wide_workgroups(orc, dev, mode):
    from rapidsfm_amd import ops

    print("[case] screen wide", mode, flush=True)
    pts, _, _, _ = plane_scene(6, 120, 120, 37, noise=0.5)
    idx = [_idx(277, 4090 + 3 * k, 8, 40 + k) for k in range(32)]
    outs = ops.ransac_f8([(_dev(pts, dev), _dev(i, dev)) for i in idx], 1.0, mode=mode)
    for i, o in zip(idx, outs):
        c, _ = orc.f8_score(pts, i, 1.0, mode, nthreads=8)
        assert np.array_equal(o["counts"].cpu().numpy().view(np.uint32), c)


@pytest.mark.parametrize("kind", ["f8", "f7"])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("what", ["nan", "inf", "far", "small", "point", "tiny_t", "huge_t"])
def test_beyond_the_bound(orc, dev, kind, mode, what):
    pts, _, _, _ = plane_scene(9, 60, 80, 40, noise=0.5)
    t = 1.0
    if what == "nan":
        pts[7, 2] = np.nan
    elif what == "inf":
        pts[3, 0] = np.inf
    elif what == "far":
        pts[5] = 3e7
    elif what == "small":
        pts *= np.float32(1e-7)
    elif what == "point":
        pts[:, :2] = pts[0, :2]
    else:
        t = 1e-9 if what == "tiny_t" else 1e12
    _check(orc, dev, pts, 130, mode, t, 3, kind)


# "no limit" as the threshold: its square is infinite in FP32, every point with a
# finite distance is an inlier; point counts that leave padding in the last tile
@pytest.mark.parametrize("kind", ["f8", "f7"])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [15, 181])
@pytest.mark.parametrize("t", [float("inf"), 2e19])
def test_no_limit(orc, dev, kind, mode, n, t):
    pts, _, _, _ = plane_scene(10, n // 3, n // 3, n - 2 * (n // 3), noise=0.5)
    _check(orc, dev, pts, 130, mode, t, 5, kind)


# the same on the 256-hypothesis workgroups
@pytest.mark.parametrize("mode", [0, 1])
def test_no_limit_wide(orc, dev, mode):
    from rapidsfm_amd import ops

    print("[case] screen wide, no limit", mode, flush=True)
    pts, _, _, _ = plane_scene(6, 40, 40, 37, noise=0.5)
    idx = [_idx(117, 1024, 8, 60 + k) for k in range(32)]
    outs = ops.ransac_f8([(_dev(pts, dev), _dev(i, dev)) for i in idx], float("inf"), mode=mode)
    for i, o in zip(idx, outs):
        c, _ = orc.f8_score(pts, i, float("inf"), mode, nthreads=8)
        assert np.array_equal(o["counts"].cpu().numpy().view(np.uint32), c)
