"""Re-rank selection when one lane of a wave meets most of a query's nearest
records (its short list overflows), against numpy. Whole numbers: no tolerance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _popcount(x):
    return np.unpackbits(x.view(np.uint8), axis=-1).sum(-1)


# `same` of the nearest records sit 64 apart in the bucket, so one lane reads
# them all; around the short list's length and the whole selection
@pytest.mark.parametrize("keep", [8, 16, 32])
@pytest.mark.parametrize("same", [2, 3, 4, 6, 7, 12, 13, 31, 33])
@pytest.mark.parametrize("tables", [1, 3])
def test_one_lane_holds_the_nearest(dev, keep, same, tables):
    from rapidsfm_amd import cashash as ch

    print("[case] rerank lists", keep, same, tables, flush=True)
    rng = np.random.default_rng(keep * 100 + same)
    nT, nQ = 64 * 40 + 17, 5
    def image(n):
        # every descriptor in bucket 3 of every table, buckets in index order
        ends = np.zeros((8, 256), np.int32)
        ends[:, 3:] = n
        return {"desc": rng.integers(0, 128, (n, 128)).astype(np.uint8), "codes": np.full((n, 8), 3, np.uint8),
                "remap": rng.integers(0, 2**32, (n, 4), dtype=np.uint64).astype(np.uint32), "ends": ends,
                "buckets": np.tile(np.arange(n, dtype=np.int32), (8, 1)), "n": n}
    t, q = image(nT), image(nQ)
    lane = 11
    for i in range(same):  # a few bits from query 0
        r = q["remap"][0].copy()
        r[i % 4] ^= np.uint32(1 << (i % 32))
        t["remap"][lane + 64 * i] = r
    d = lambda im: {k: (torch.from_numpy(v.view(np.int32) if v.dtype == np.uint32 else v).to(dev) if k != "n" else v)  # noqa: E731
                    for k, v in im.items()}
    ((bq, bt),) = ch.find_best_match_rerank([d(q)], d(t), tables, keep)
    def ref(a, b):
        out = np.zeros((a["n"], 2), np.uint32)
        for i in range(a["n"]):
            h = _popcount(a["remap"][i][None] ^ b["remap"])
            sel = np.argsort(h * (1 << 24) + np.arange(b["n"]), kind="stable")[:keep]
            l2 = ((a["desc"][i].astype(np.int64)[None] - b["desc"][sel]) ** 2).sum(1)
            k = np.lexsort((sel, l2))[0]
            out[i] = sel[k], l2[k]
        return out
    assert np.array_equal(bq.cpu().numpy().view(np.uint32), ref(q, t))
    assert np.array_equal(bt.cpu().numpy().view(np.uint32)[: 200], ref({**t, "n": 200}, q))
