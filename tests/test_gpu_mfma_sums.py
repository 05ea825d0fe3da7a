"""The FP32 accumulation error of the f16 matrix instructions that the inlier
screens assume: at most 10 * 2^-24 of the sum of the terms' magnitudes (products
of two f16 values are exact in FP32's 24 bits), against sums in FP64. The unit
aligns an operand below f16's normal range as if it were 2^-14, so it counts as
that; the screens allow 2^-14 times its partner for such an operand, 2^20 times
its part here."""
import ctypes
import os

import pytest
import torch

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(__file__), "hip", "libmfma_sums.so")
BATCHES = 12000  # of 256 dot products: 3e6 a case


def _binades(shape, lo, hi, g, dev):
    """random signs and fractions, exponents uniform in [lo, hi)"""
    e = torch.randint(lo, hi, shape, generator=g, device=dev)
    x = torch.ldexp(1.0 + torch.rand(shape, generator=g, device=dev), e)
    return torch.where(torch.rand(shape, generator=g, device=dev) < 0.5, x, -x).half()


def _operands(kind, k, g, dev):
    shape = (BATCHES, 16, k)
    if kind == "uniform":
        return [(2 * torch.rand(shape, generator=g, device=dev) - 1).half() for _ in range(2)]
    if kind == "binades":
        return [_binades(shape, -6, 6, g, dev) for _ in range(2)]
    if kind == "subnormal":
        a, b = _binades(shape, -24, -12, g, dev), _binades(shape, -24, 10, g, dev)
        a[torch.rand(shape, generator=g, device=dev) < 0.125] = 0
        return [a, b]
    if kind == "cancelling":
        a, b = (_binades(shape, -3, 3, g, dev) for _ in range(2))
        h = k // 2
        a[..., h:] = a[..., :h]
        b[..., h:] = -b[..., :h]
        b[..., -1] *= 1.001
        return [a, b]
    # split: values of 22 bits in two halves, the products hi hi, hi lo, lo hi of each, as the screens lay them out
    out = []
    for order in ("hhl", "hlh"):
        v = (2 * torch.rand((BATCHES, 16, k // 3), generator=g, device=dev) - 1) * 1024
        hi = v.half()
        lo = (v - hi.float()).half()
        t = torch.zeros(shape, dtype=torch.float16, device=dev)
        for j, c in enumerate(order):
            t[..., j: 3 * (k // 3): 3] = hi if c == "h" else lo
        out.append(t)
    return out


@pytest.mark.parametrize("k", [16, 32])
@pytest.mark.parametrize("kind", ["uniform", "binades", "subnormal", "cancelling", "split"])
def test_accumulation_error(dev, k, kind):
    if not os.path.exists(LIB):
        pytest.fail("tests/hip/libmfma_sums.so is not built (run __graft_entry__.build())")
    print("[case] matrix-unit sums", k, kind, flush=True)
    lib = ctypes.CDLL(LIB)
    lib.mfma_sums.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32, ctypes.c_void_p]
    a, b = _operands(kind, k, torch.Generator(device=dev).manual_seed(k), dev)
    assert a.shape == b.shape == (BATCHES, 16, k) and a.is_contiguous() and b.is_contiguous()
    d = torch.empty((BATCHES, 16, 16), dtype=torch.float32, device=dev)
    assert lib.mfma_sums(k, a.data_ptr(), b.data_ptr(), d.data_ptr(), BATCHES, torch.cuda.current_stream().cuda_stream) == 0
    x, y = a.double(), b.double().transpose(1, 2).contiguous()
    err = (d.double() - torch.bmm(x, y)).abs()
    apparent = lambda v: torch.where(v == 0, 0.0, v.abs().clamp_min(2.0**-14))  # noqa: E731
    size = torch.bmm(apparent(x), apparent(y))
    print("largest error / sum of magnitudes: %.2f * 2^-24" % (float((err / size.clamp_min(1e-300)).max()) * 2**24))
    assert bool((err <= 10 * 2.0**-24 * size).all())
