"""7-point samples whose cubics are bisected away from the lane that owns them: counts and
models bit-exact with the FP32 oracle at the edges of a workgroup's 128 samples, with
samples that have no cubic among the others; and the best hypothesis without a mask."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,H", [(0, 1), (1, 127), (1, 128), (0, 129), (1, 385)])
def test_f7_workgroup_edges(orc, dev, mode, H):
    from rapidsfm_amd import ops
    from rapidsfm_amd._abi import RansacTask, check, lib

    print("[case] f7 roots", mode, H, flush=True)
    pts, _, _ = orc.gen_two_view(31, 500, 120)
    rng = np.random.default_rng(H)
    idx = np.stack([rng.choice(500, 7, replace=False) for _ in range(H)]).astype(np.uint32)
    idx[2::5] = idx[2::5, :1]  # one point seven times: no cubic
    idx[4::7, 6] = 500  # out of range
    idx[1::6, 5] = idx[1::6, 4]  # a point twice: a cubic that is degenerate or nearly so
    ref_c, ref_m = orc.f7_score(pts, idx, 1.5, mode)
    pt, it = torch.from_numpy(pts).to(dev), torch.from_numpy(idx.view(np.int32)).to(dev)
    (o,) = ops.ransac_f7([(pt, it)], 1.5, mode=mode, want_models=True)
    assert np.array_equal(o["counts"].cpu().numpy().view(np.uint32), ref_c)
    assert np.array_equal(o["models"].cpu().numpy().reshape(H, 9).view(np.uint32), ref_m.view(np.uint32))
    counts = torch.empty(H, dtype=torch.int32, device=dev)
    best = torch.full((2,), -7, dtype=torch.int32, device=dev)
    task = (RansacTask * 1)(RansacTask(pt.data_ptr(), 500, None, it.data_ptr(), H, counts.data_ptr(), None,
                                       best.data_ptr(), None))
    check(lib.rsfm_ransac_f7(task, 1, 1.5, mode, 0.0, 0.0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "f7")
    assert torch.equal(best, o["best"]) and torch.equal(counts, o["counts"])
