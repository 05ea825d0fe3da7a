"""The proposal network's forward kernel at the edges of its tiles and grid, and
on features that are not numbers."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# one short of / at / past a wave's 32 matches and a workgroup's 128, and past
# one round of the whole grid (512 workgroups x 128); against FP64 with the
# inputs and weights rounded to bf16: the activations' bf16 roundings remain,
# 2^-9 relative per layer on sums of 64 terms
@pytest.mark.parametrize("n", [1, 32, 33, 127, 128, 129, 65535, 65536, 65569, 150001])
def test_forward_edges(dev, n):
    from rapidsfm_amd import learned as L

    print("[case] mlp forward", n, flush=True)
    p = L.init_params(3, device=dev)
    p[L.OFF_B1:L.OFF_W2] = torch.linspace(-0.3, 0.4, 64, device=dev)
    p[L.OFF_B2:L.OFF_W3] = torch.linspace(0.5, -0.2, 64, device=dev)
    p[L.OFF_B3:L.OFF_W4] = torch.linspace(-0.1, 0.3, 64, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    x = torch.randn((n, 8), generator=g, device=dev)
    out = L.forward(p, x)
    r = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    W = lambda a, b, c: r(p[a:b]).view(c, -1)  # noqa: E731
    h = torch.relu(r(x) @ W(L.OFF_W1, L.OFF_B1, 64).T + p[L.OFF_B1:L.OFF_W2].double())
    h = torch.relu(h @ W(L.OFF_W2, L.OFF_B2, 64).T + p[L.OFF_B2:L.OFF_W3].double())
    h = torch.relu(h @ W(L.OFF_W3, L.OFF_B3, 64).T + p[L.OFF_B3:L.OFF_W4].double())
    z = h @ r(p[L.OFF_W4:L.OFF_B4]) + p[L.OFF_B4].double()
    ref = torch.sigmoid(z)
    # three roundings of 2^-9 through layers of gain about 1, sigmoid slope <= 1/4
    assert float((out.double() - ref).abs().max()) <= 3 * 2.0**-9 * float(z.abs().max().clamp_min(1.0))
    assert torch.equal(out, L.forward(p, x))


def test_forward_not_a_number(dev):
    from rapidsfm_amd import learned as L

    print("[case] mlp forward nan", flush=True)
    p = L.init_params(4, device=dev)
    x = torch.randn((200, 8), device=dev)
    clean = L.forward(p, x)
    x[37, 2] = float("nan")
    out = L.forward(p, x)
    # ReLU takes NaN to 0, so the row's probability is a number, and no other row changes
    assert bool(torch.isfinite(out).all())
    keep = torch.arange(200, device=dev) != 37
    assert torch.equal(out[keep], clean[keep])


# partial counts around the reduction's eight groups of eight: 1, 7, 8, 9, 63, 64, 65 workgroups; all 256
# with a step each, one match more, and several ragged steps
@pytest.mark.parametrize("n", [100, 896, 1024, 1152, 8064, 8192, 8320, 32768, 32769, 70000])
def test_gradient_sum_edges(dev, n):
    from rapidsfm_amd import learned as L

    print("[case] mlp grad", n, flush=True)
    p = L.init_params(5, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    x = torch.randn((n, 8), generator=g, device=dev)
    y = (torch.rand(n, generator=g, device=dev) < 0.4).float()
    whole, loss = L.grad(p, x, y)
    # the same samples in one-step pieces (one partial each), weighted by their size
    acc, lacc = torch.zeros(L.N_PARAM, dtype=torch.float64, device=dev), 0.0
    for b in range(0, n, 128):
        gi, li = L.grad(p, x[b:b + 128].contiguous(), y[b:b + 128].contiguous())
        m = min(128, n - b)
        acc += gi.double() * (m / n)
        lacc += float(li) * m / n
    # the pieces round dz = (p - y) / m to bf16 at another scale: 2^-8 per product; the sums are FP32
    assert float((whole.double() - acc).norm() / acc.norm()) < 2.0**-8
    assert abs(float(loss) - lacc) < 1e-5 * max(1.0, abs(lacc))


# a partial a workgroup is all that a gradient writes: the size asked for, up to the 256
# workgroups' and no further, and nothing past it
@pytest.mark.parametrize("n,partials", [(1, 1), (129, 2), (32768, 256), (32769, 256), (65537, 256)])
def test_gradient_workspace(dev, n, partials):
    import ctypes

    from rapidsfm_amd import learned as L
    from rapidsfm_amd._abi import lib

    print("[case] mlp grad workspace", n, flush=True)
    need = ctypes.c_size_t(0)
    assert lib.rsfm_mlp_grad_workspace_size(n, ctypes.byref(need)) == 0
    assert need.value == partials * (L.N_PARAM + 1) * 4
    p = L.init_params(6, device=dev)
    x = torch.randn((n, 8), device=dev)
    y = (torch.rand(n, device=dev) < 0.4).float()
    ws = torch.full((need.value // 4 + 4096,), 7.0, device=dev)
    g, loss = torch.empty(L.N_PARAM, device=dev), torch.empty(1, device=dev)
    call = lambda b: lib.rsfm_mlp_grad(p.data_ptr(), x.data_ptr(), y.data_ptr(), n, g.data_ptr(), loss.data_ptr(),  # noqa: E731
                                       ws.data_ptr(), b, torch.cuda.current_stream().cuda_stream)
    assert call(need.value - 1) != 0  # refused before any launch
    assert call(need.value) == 0
    rg, rl = L.grad(p, x, y)
    assert torch.equal(g, rg) and torch.equal(loss, rl)
    assert bool((ws[need.value // 4:] == 7.0).all())
