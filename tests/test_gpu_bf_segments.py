"""Matching with short train segments merged in place: best and second best and
the train side against numpy over segment edges, one and several pairs per call,
planted ties across segments. Whole numbers: no tolerance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(q, t):
    d = (q[:, None, :].astype(np.int64) - t[None].astype(np.int64))
    d = (d * d).sum(2)
    k = d * (1 << 32) + np.arange(t.shape[0])[None]
    o = np.sort(k, 1)
    kb = d.T * (1 << 32) + np.arange(q.shape[0])[None]
    none = (1 << 64) - 1
    sec = o[:, 1].astype(np.uint64) if t.shape[0] > 1 else np.full(q.shape[0], none, np.uint64)
    return o[:, 0].astype(np.uint64), sec, kb.min(1).astype(np.uint64)


def _keys(x):
    v = x.cpu().numpy().view(np.uint32).astype(np.uint64)
    return (v[:, 1] << np.uint64(32)) | v[:, 0]


def _desc(rng, n):
    d = rng.integers(0, 60, (n, 128)).astype(np.uint8)
    d[rng.random(n) < 0.2] = 255  # equal rows: ties within and across segments
    return d


# train counts around one, two and several 128-column segments; query counts
# around a row block; pair counts around the small kernel argument
@pytest.mark.parametrize("pairs", [1, 2, 3])
@pytest.mark.parametrize("nA,nB", [(1, 1), (5, 2), (255, 127), (256, 128), (257, 129), (300, 255), (64, 256), (10, 257), (30, 1300)])
def test_segments(dev, pairs, nA, nB):
    import rapidsfm_amd as rs

    print("[case] segments", pairs, nA, nB, flush=True)
    rng = np.random.default_rng(nA * 7 + nB + pairs)
    sizes = [(max(1, nA - 3 * i), max(1, nB - 5 * i)) for i in range(pairs)]
    host = [(_desc(rng, a), _desc(rng, b)) for a, b in sizes]
    for q, t in host:
        if t.shape[0] > 4:
            t[-1] = t[0]  # a tie between the first and the last segment
            q[0] = t[0]
    devp = [(torch.from_numpy(q).to(dev), torch.from_numpy(t).to(dev)) for q, t in host]
    top2 = rs.bf_match_top2(devp)
    top1 = rs.bf_match(devp)
    for (q, t), (a, s, b), (a1, b1) in zip(host, top2, top1):
        ra, rs2, rb = _ref(q, t)
        assert np.array_equal(_keys(a), ra) and np.array_equal(_keys(s), rs2) and np.array_equal(_keys(b), rb)
        assert np.array_equal(_keys(a1), ra) and np.array_equal(_keys(b1), rb)


# a long and a short train set in one call: the short one has fewer segments
def test_uneven_call(dev):
    import rapidsfm_amd as rs

    print("[case] uneven segments", flush=True)
    rng = np.random.default_rng(1)
    host = [(_desc(rng, 70), _desc(rng, 3000)), (_desc(rng, 300), _desc(rng, 40)), (_desc(rng, 9), _desc(rng, 1))]
    devp = [(torch.from_numpy(q).to(dev), torch.from_numpy(t).to(dev)) for q, t in host]
    for (q, t), (a, s, b) in zip(host, rs.bf_match_top2(devp)):
        ra, rs2, rb = _ref(q, t)
        assert np.array_equal(_keys(a), ra) and np.array_equal(_keys(s), rs2) and np.array_equal(_keys(b), rb)
