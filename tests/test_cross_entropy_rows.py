"""Fused cross-entropy over rows of every alignment, against fp64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v", [1, 7, 8, 9, 2047, 8192, 32003, 128256])
@pytest.mark.parametrize("offset", [0, 1, 5])
def test_cross_entropy_rows(v, offset):
    from deepspeed_amd.ops import _C
    g = torch.Generator().manual_seed(v)
    n = 5
    flat = torch.empty(n * v + offset, dtype=torch.bfloat16, device="cuda")
    x = flat[offset:].view(n, v)
    x.copy_(6 * torch.randn(n, v, generator=g))
    x[1, : v // 2] = float("-inf")               # masked
    if v > 9:
        x[2, :9] = torch.finfo(torch.bfloat16).min
    y = torch.randint(0, v, (n,), generator=g)
    y[1], y[3] = v - 1, -100
    y = y.cuda()
    loss, lse = _C.ce_fwd(x, y, -100)
    gs = torch.rand(n, generator=g).cuda()
    d = _C.ce_bwd(x, y, lse, gs, -100)
    xd = x.double()
    want = torch.logsumexp(xd, 1)
    # fp32 sums of v terms by 256 threads and the hardware's exp and log
    torch.testing.assert_close(lse.double(), want, rtol=2e-6, atol=2e-5)
    pick = xd.gather(1, y.clamp(min=0)[:, None])[:, 0]
    live = y != -100
    torch.testing.assert_close(loss.double(), torch.where(
        live, want - pick, torch.zeros_like(want)), rtol=1e-5, atol=4e-5)
    p = torch.softmax(xd, 1)
    p[live.nonzero()[:, 0], y[live]] -= 1
    p = p * (gs * live).double()[:, None]
    # rounded to bf16 once
    assert ((d.double() - p).abs() <= 2.0 ** -8 * p.abs() + 1e-5).all()


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 9001])
@pytest.mark.parametrize("ignored", ["none", "some", "all"])
def test_sum_and_mean(n, ignored):
    from deepspeed_amd.ops import _C
    from deepspeed_amd.ops.cross_entropy import (fused_cross_entropy_mean,
                                                 fused_cross_entropy_sum)
    g = torch.Generator().manual_seed(n)
    x = (3 * torch.randn(n, 24, generator=g)).bfloat16().cuda()
    y = torch.randint(0, 24, (n,), generator=g).cuda()
    if ignored != "none":
        y[:: 1 if ignored == "all" else 3] = -100
    x.requires_grad_()
    rows, lse = _C.ce_fwd(x.detach(), y, -100)
    live = int((y != -100).sum())
    total, count = fused_cross_entropy_sum(x, y)
    mean = fused_cross_entropy_mean(x, y)
    assert count.item() == live
    # fp64 sums, rounded once and once more divided
    want = rows.double().sum()
    torch.testing.assert_close(total.double(), want, rtol=2.0 ** -24, atol=0)
    torch.testing.assert_close(mean.double(), want / max(live, 1),
                               rtol=2.0 ** -23, atol=0)
    mean *= 1.0                                   # its own memory
    (d,) = torch.autograd.grad(mean * 8, x)
    scale = torch.full((n,), 8.0, device="cuda") / max(live, 1)
    assert torch.equal(d, _C.ce_bwd(x.detach(), y, lse, scale, -100))
