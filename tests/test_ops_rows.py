"""Host helpers. The outputs of a batched call are parts of one allocation: each with its own rows and version,
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


def test_parts_are_tensors_of_their_own():
    """what a caller can do with separate allocations: write in place under autograd, and write
    one part while another is saved for a backward pass"""
    a, b = ops._rows([torch.empty(1)] * 2, [3, 4], 9, torch.float32)
    for t in (a, b):
        assert not t._is_view() and not t.requires_grad
        t.fill_(2.0)
    w = torch.ones(3, 9, requires_grad=True)
    y = (w * a).sum()  # saves a
    b.zero_()
    y.backward()
    assert bool((w.grad == 2.0).all())
    a.mul_(w)
    assert a.requires_grad and not b.requires_grad


def test_models_are_tensors_of_their_own():
    pts = torch.zeros(20, 4)
    idx = torch.zeros((5, 8), dtype=torch.int32)
    _, outs = ops._ransac_tasks([(pts, idx), (pts, idx)], True)
    assert all(o["models"].shape == (5, 3, 3) and not t._is_view() for o in outs for t in o.values())


def test_current_stream_without_the_private_call(monkeypatch):
    class Stream:
        cuda_stream = 42

    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: Stream)
    monkeypatch.setattr(ops, "_current_raw_stream", None, raising=False)
    assert ops._stream(None) == 42 and ops._stream(Stream) == 42


def test_score_takes_any_iterable(monkeypatch):
    from rapidsfm_amd import proposal

    class Lib:
        rsfm_ransac_f8 = staticmethod(lambda tasks, n, *a: 0 if n == 2 and tasks[1].nbPts == 30 else 1)

    monkeypatch.setattr(proposal, "lib", Lib)
    monkeypatch.setattr(proposal, "_stream", lambda s: 0)
    pts = [torch.zeros(20, 4), torch.zeros(30, 4)]
    idx = [torch.zeros((5, 8), dtype=torch.int32)] * 2
    for outs in (proposal.score(list(zip(pts, idx))), proposal.score(zip(pts, idx))):
        assert [len(o["mask"]) for o in outs] == [20, 30]
