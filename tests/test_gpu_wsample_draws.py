"""The weighted sampler's draws side by side: bit-exact with the oracle where repeats are the
rule (few weights), at counts around powers of two and
the table's 2048 entries, and where the draws run out."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,H,positive", [(8, 65, 8), (9, 64, 9), (16, 63, 9), (17, 257, 17), (2048, 256, 30), (2049, 255, 9),
                                          (4097, 1, 8), (4096, 300, 12),
                                          (300, 70, 7), (300, 70, 1), (65536, 129, 65536), (65537, 64, 65537)])
def test_repeats_and_edges(orc, dev, n, H, positive):
    from rapidsfm_amd import learned

    print("[case] weighted draws", n, H, positive, flush=True)
    rng = np.random.default_rng(n + positive)
    w = np.zeros(n, np.float32)
    # down to the smallest weight that counts, 1 / 65536; the last entry may be one of them or a run of zeros
    w[rng.choice(n, positive, replace=False)] = np.float32(2.0) ** rng.integers(-16, 1, positive)
    # fewer than eight weights: every set is given up after the last draw (all ~0)
    (idx,) = learned.sample_weighted([(torch.from_numpy(w).to(dev), H, n)])
    got = idx.cpu().numpy().view(np.uint32)
    assert np.array_equal(got, orc.sample_weighted(w, H, n))
    assert positive >= 8 or (got == 0xFFFFFFFF).all()
