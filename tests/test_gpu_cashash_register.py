"""One-call registration of an image against the separate entry points: codes,
remap, bucket ends and largest bucket equal, buckets equal as sets. Whole
numbers: no tolerance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _desc(rng, n, skew):
    d = rng.integers(0, 128, (n, 128)).astype(np.uint8)
    if skew and n:
        d[: n // 2] = d[0]  # half of the image in one bucket of every table
    return d


# around a wave's part of the index (64 x 16), a hash block (32), the batch of
# loads (512 per wave) and the largest image of the one-call form
@pytest.mark.parametrize("channels", [64, 192])
@pytest.mark.parametrize("n,skew", [(0, False), (1, False), (31, False), (33, True), (1023, False), (1025, True), (8192, False),
                                    (8193, True), (65536, False), (65537, True)])
def test_register_image(dev, channels, n, skew):
    from rapidsfm_amd import cashash as ch
    from rapidsfm_amd.synth import cashash_weights

    print("[case] register", channels, n, skew, flush=True)
    w, base = cashash_weights(3, 192, dev)
    w, base = w[:channels].contiguous(), base[:channels].contiguous()
    d = torch.from_numpy(_desc(np.random.default_rng(n + channels), n, skew)).to(dev)
    bias = ch.compute_bias(w, base, ch.accumulate(d), max(1, n))
    im = ch.register_image(d, w, bias)
    codes, remap, _ = ch.compute_hash(w, bias, d)
    lo, up, mx = ch.bucket_bounds(ch.build_histogram(codes))
    assert torch.equal(im["codes"], codes) and torch.equal(im["ends"], up) and torch.equal(im["max_bucket"], mx)
    assert (im["remap"] is None) == (channels == 64) and im["n"] == n
    if remap is not None:
        assert torch.equal(im["remap"], remap)
    b = im["buckets"].cpu().numpy().astype(np.int64)
    c = codes.cpu().numpy()
    for s in range(8):
        assert np.array_equal(np.sort(b[s]), np.arange(n))
        assert np.array_equal(c[b[s], s], np.sort(c[:, s]))  # every bucket holds its code's descriptors
