"""The outputs of a batched call are parts of one allocation: each with its own rows,
aligned, for every count including none and one, on the device of its own problem."""
import pytest
import torch

from rapidsfm_amd import ops


@pytest.mark.parametrize("counts", [[], [5], [0], [0, 0], [1, 0, 255, 256, 257], [4096, 3]])
@pytest.mark.parametrize("cols,dtype", [(None, torch.uint8), (None, torch.int64), (8, torch.int32), (9, torch.float32)])
def test_parts_are_disjoint_and_aligned(counts, cols, dtype):
    likes = [torch.empty(1) for _ in counts]
    parts = ops._rows(likes, counts, cols, dtype)
    assert len(parts) == len(counts)
    for i, (t, n) in enumerate(zip(parts, counts)):
        assert t.shape == ((n,) if cols is None else (n, cols)) and t.dtype == dtype and t.is_contiguous()
        # against the allocation's own start: 256 rows of any row size are a multiple of 256 bytes
        assert n == 0 or len(counts) < 2 or (t.data_ptr() - t.untyped_storage().data_ptr()) % 256 == 0
        t.fill_(i + 1)
    assert all(bool((t == i + 1).all()) for i, t in enumerate(parts))


def test_parts_follow_their_problem_s_device():
    parts = ops._rows([torch.empty(1), torch.empty(1, device="meta")], [3, 4], None, torch.int32)
    assert [t.device.type for t in parts] == ["cpu", "meta"]
