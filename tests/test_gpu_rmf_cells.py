"""The affine filter's matrix-core counts at the edges of their tiles and
chunks, near the threshold, and beyond the screen's bound: votes and affines
bit-equal to the CPU restatement."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(orc, dev, m, cell_cols, n_tests, rel, try_other, seed):
    from rapidsfm_amd import rmf

    r, bounds, order, cols, rows, cw = orc.rmf_bin(4000, 3000, m, cell_cols)
    ref, raff = orc.rmf_filter(r, bounds, cols, rows, n_tests, cw * rel, try_other, seed)
    votes, aff = rmf.filter_votes(torch.from_numpy(r).to(dev), torch.from_numpy(bounds.view(np.int32)).to(dev), cols, rows,
                                  n_tests, cw * rel, try_other, seed)
    assert np.array_equal(votes.cpu().numpy(), ref)
    ga = aff.cpu().numpy()
    assert np.array_equal(np.isnan(ga), np.isnan(raff))
    assert np.array_equal(np.nan_to_num(ga).view(np.uint32), np.nan_to_num(raff).view(np.uint32))


def _matches(seed, n, spread, noise):
    """n matches, two thirds on one affine with noise, the rest uniform, left points in one patch of `spread` px"""
    rng = np.random.default_rng(seed)
    left = np.array([1900.0, 1400.0]) + rng.uniform(0, spread, (n, 2))
    right = left @ np.array([[0.9, 0.2], [-0.15, 1.1]]) + np.array([300.0, -250.0]) + rng.normal(0, noise, (n, 2))
    bad = rng.random(n) < 1 / 3
    right[bad] = rng.uniform([0, 0], [4000, 3000], (int(bad.sum()), 2))
    return np.concatenate([left, right], 1).astype(np.float32)


# one neighbourhood of n matches: below the 9 that a hypothesis needs, around a
# 16-match tile, 8 tiles and the 256-match chunk, and several chunks; tests
# around the 128 of a round
@pytest.mark.parametrize("n,n_tests", [(16, 128), (17, 127), (31, 129), (127, 256), (128, 1), (129, 300), (255, 128),
                                       (256, 128), (257, 128), (300, 256), (700, 256)])
@pytest.mark.parametrize("try_other", [False, True])
def test_neighbourhood_sizes(orc, dev, n, n_tests, try_other):
    print("[case] rmf cells", n, n_tests, try_other, flush=True)
    _check(orc, dev, _matches(n, n, 60.0, 8.0), 16, n_tests, 0.15, try_other, 7 + n)


# noise at the inlier radius: many tests within the screen's bound
@pytest.mark.parametrize("spread,noise,rel", [(200.0, 25.0, 0.15), (900.0, 25.0, 0.15), (3.0, 0.02, 0.0001)])
def test_near_the_threshold(orc, dev, spread, noise, rel):
    print("[case] rmf near", spread, noise, rel, flush=True)
    _check(orc, dev, _matches(3, 1200, spread, noise), 16, 256, rel, True, 5)


@pytest.mark.parametrize("what", ["far", "nan", "inf", "line", "point"])
def test_beyond_the_bound(orc, dev, what):
    print("[case] rmf beyond", what, flush=True)
    m = _matches(4, 200, 300.0, 5.0)
    if what == "far":
        m[5, 2] = 3e7
    elif what == "nan":
        m[5, 2] = np.nan
    elif what == "inf":
        m[5, 3] = np.inf
    elif what == "line":
        m[:, 1] = 0.5 * m[:, 0]
    else:
        m[:, :2] = m[0, :2]
    _check(orc, dev, m, 16, 256, 0.15, True, 9)


# few large cells and the most cells of the batch form
@pytest.mark.parametrize("cell_cols", [1, 2, 3, 32])
def test_cell_counts(orc, dev, cell_cols):
    print("[case] rmf cell columns", cell_cols, flush=True)
    rng = np.random.default_rng(2)
    m = _matches(6, 1500, 900.0, 10.0)
    m[::2, :2] = rng.uniform([0, 0], [4000, 3000], (750, 2))
    _check(orc, dev, m, cell_cols, 128, 0.15, True, 1)


# A steep affine (area kept, one axis stretched T0 times) of one cell, tried on a
# far cell whose matches it hits exactly in FP32: the expression's own rounding
# there, the larger the steeper, is beyond the threshold, and the test accepts
# what the affine in exact arithmetic misses by more than twice the threshold.
@pytest.mark.parametrize("t0,th", [(250.0, 0.005), (400.0, 0.02), (2001.0, 0.1), (30000.0, 1.0)])
@pytest.mark.parametrize("n", [16, 40])
def test_steep_affine_of_another_cell(orc, dev, t0, th, n):
    print("[case] rmf steep", t0, th, n, flush=True)
    rng = np.random.default_rng(1)
    left = np.stack([rng.uniform(2990, 3010, 40), rng.uniform(2400, 2600, 40)], 1).astype(np.float32)
    right = np.stack([(left[:, 0].astype(np.float64) - 3000) * t0 + 2000, (left[:, 1] - 2500.0) / t0 + 1500], 1)
    steep = np.concatenate([left, right], 1).astype(np.float32)
    rel, seed = th / 250, 7
    r, bounds, _, cols, rows, cw = orc.rmf_bin(4000, 3000, steep, 16)
    assert cw == 250
    _, aff = orc.rmf_filter(r, bounds, cols, rows, 256, cw * rel, True, seed)
    T = aff[10 * cols + 12]
    assert abs(T[0] - t0) < 0.01 * t0
    # of the x near 3000 the one where FP32 is furthest from exact arithmetic
    xs = np.unique(rng.uniform(2995, 3005, 4000).astype(np.float32))
    y = np.float32(500.25)
    fl = ((T[0] * xs + T[1] * y) + T[2]).astype(np.float32)
    off = np.abs(T[0].astype(np.float64) * xs + T[1].astype(np.float64) * y + T[2] - fl)
    k = int(np.argmax(off))
    assert off[k] > 2.2 * th
    hit = np.array([xs[k], y, fl[k], (T[3] * xs[k] + T[4] * y) + T[5]], np.float32)
    _check(orc, dev, np.concatenate([steep, np.tile(hit, (n, 1))]), 16, 256, rel, True, seed)


# more matches in one neighbourhood than 25 bits count
def test_largest_neighbourhood(dev):
    from rapidsfm_amd import rmf

    n = (1 << 25) + 3
    print("[case] rmf neighbourhood", n, flush=True)
    g = torch.Generator(device=dev).manual_seed(1)
    m = torch.rand((n, 2), generator=g, device=dev) * 3000.0
    votes, _ = rmf.filter_votes(torch.cat([m, m], 1), torch.tensor([0, n], dtype=torch.int32, device=dev), 1, 1, 128,
                                8.0, False, 3)
    assert int((votes == 1).sum()) == n
