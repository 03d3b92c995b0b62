"""Linear's backward over transposed operands: which are transposed, and the
gradients against torch's own and fp64."""

import pytest
import torch
import torch.nn as nn

from deepspeed_amd.ops import linear as L


def test_backward_plan():
    assert L.backward_plan(8192, 14336, 4096) == (True, False, True)
    assert L.backward_plan(8192, 4096, 14336) == (True, True, False)
    assert L.backward_plan(2048, 4096, 4096) == (False, False, True)
    assert L.backward_plan(2047, 4096, 4096) == (False, False, False)
    assert L.backward_plan(32768, 3072, 3072) == (True, False, False)
    assert L.backward_plan(16, 64, 64) == (False, False, False)
    # the weight: where the copy has been measured to pay
    for n, k in ((14336, 4096), (128256, 4096), (4096, 14336), (8192, 3072)):
        for t in (2048, 2560, 3000, 3111, 4000, 8192):
            assert L.backward_plan(t, n, k)[0] == (t > 3100), (t, n, k)
    assert [L.backward_plan(t, 4096, 4096)[0] for t in (3111, 3500)] == \
        [False, True]
    # its gradient: not where the output nearly fills a second round of CUs
    for n, k, much in ((5120, 5120, False), (7168, 4096, False),
                       (6144, 4096, True), (6144, 6144, True)):
        assert L.backward_plan(12288, n, k)[2]
        assert L.backward_plan(16384, n, k)[2] == much


def test_is_torchs_linear_elsewhere():
    """CPU, double backward, vmap and forward-mode tangents."""
    torch.manual_seed(0)
    a = L.Linear(6, 5).double()
    b = nn.Linear(6, 5).double()
    b.load_state_dict(a.state_dict())
    x = torch.randn(3, 6, dtype=torch.float64, requires_grad=True)
    assert torch.equal(a(x), b(x))
    assert torch.autograd.gradgradcheck(a, (x,))
    assert torch.equal(torch.func.vmap(a)(x), torch.func.vmap(b)(x))
    t = torch.ones_like(x)
    _, ja = torch.func.jvp(a, (x,), (t,))
    _, jb = torch.func.jvp(b, (x,), (t,))
    assert torch.equal(ja, jb)


@pytest.mark.parametrize("frozen", ["weight", "input", "bias", None])
def test_saves_what_the_backward_needs(frozen):
    """As torch's layer does: a frozen weight holds no input (adapters over a
    frozen model), an input without gradient no weight."""
    torch.manual_seed(0)
    t = {"input": torch.randn(2, 3, 6), "weight": torch.randn(5, 6),
         "bias": torch.randn(5)}
    grads, kept = [], []
    for f in (L._Linear.apply, nn.functional.linear):
        x, w, b = (t[n].clone().requires_grad_(n != frozen) for n in t)
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(
                lambda s: seen.append(s.numel()) or s, lambda s: s):
            f(x, w, b).sum().backward()
        grads.append([x.grad, w.grad, b.grad])
        kept.append(sorted(seen))
    assert kept[0] == kept[1]
    for a, b in zip(*grads):
        assert a is b is None or torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("r,c", [(1, 1), (8, 64), (127, 63), (128, 64),
                                 (129, 72), (1000, 264), (4000, 3072),
                                 (3, 8200)])
@pytest.mark.parametrize("offset", [0, 3])
def test_transpose_2d_gpu(r, c, offset):
    from deepspeed_amd.ops import _C
    x = torch.randn(r * c + offset, device="cuda").bfloat16()[offset:]
    x = x.view(r, c)
    y = _C.transpose_2d(x)
    assert torch.equal(y, x.t())
    assert y.stride() == (-(-r // 8) * 8, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [((3, 1000), 640, 512), ((4096,), 2048, 2048),
                                   ((2, 2049), 1032, 4096), ((1, 7), 24, 16)])
@pytest.mark.parametrize("plan", [(False, False, False), (True, True, True),
                                  (True, False, True), (False, True, False)])
@pytest.mark.parametrize("bias", [False, True])
def test_linear_backward_gpu(shape, plan, bias, monkeypatch):
    lead, n, k = shape
    monkeypatch.setattr(L, "backward_plan", lambda *a: plan)
    torch.manual_seed(0)
    lin = L.Linear(k, n, bias=bias, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(*lead, k, device="cuda").bfloat16().requires_grad_()
    dy = torch.randn(*lead, n, device="cuda").bfloat16()
    y = lin(x)
    assert torch.equal(y, nn.functional.linear(x, lin.weight, lin.bias))
    y.backward(dy)
    x2, d2, w = (t.detach().double() for t in (x, dy, lin.weight))
    x2, d2 = x2.view(-1, k), d2.view(-1, n)
    for got, want, terms in ((x.grad.view(-1, k), d2 @ w, n),
                             (lin.weight.grad, d2.t() @ x2, len(x2))):
        # one rounding to bf16 of an fp32 sum
        err = (got.double() - want).abs()
        lim = 2.0 ** -8 * want.abs() + 2.0 ** -20 * terms ** 0.5 * \
            want.abs().max()
        assert (err <= lim).all(), (err / lim).max()
    if bias:
        torch.testing.assert_close(lin.bias.grad.double(), d2.sum(0),
                                   rtol=2.0 ** -7, atol=0.05)


@pytest.mark.gpu
def test_linear_double_backward_and_saved_tensor_hooks():
    torch.manual_seed(0)
    lin = L.Linear(512, 512, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(4096, 512, device="cuda").bfloat16().requires_grad_()
    g, = torch.autograd.grad(lin(x).float().square().sum(), x,
                             create_graph=True)
    g.float().sum().backward()
    assert lin.weight.grad is not None and x.grad is not None
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: seen.append(t.shape) or t, lambda t: t):
        lin(x).float().sum().backward()
    assert x.shape in seen and lin.weight.shape in seen
