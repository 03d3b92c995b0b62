"""Flash attention kernels against fp64 attention, head by head."""

import math

import pytest
import torch

from deepspeed_amd.ops import attention

pytestmark = pytest.mark.gpu


def _reference(q, k, v, do, causal, scale):
    """(value, limit) of o, dq, dk and dv: the gradients in fp64, and for each
    row of a head how far off the norm of its error may be.

    P, dS and the results are rounded to bf16, by 2^-9 of each at most (so a sum
    over them by 2^-9 / sqrt(3) of the root of its squared terms, give or take;
    2^-8 is three and a half times that). sum(do * o), which dS takes off, is
    made from the rounded o: one number a row, whose error nothing averages, and
    of thousands of them the largest is five times that: 2^-7."""
    B, S, H, D = q.shape
    G = H // k.shape[2]
    q, k, v, do = (x.detach().double() for x in (q, k, v, do))
    o, dq = torch.zeros_like(q), torch.zeros_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(k)
    lim = [torch.zeros(x.shape[:3], dtype=x.dtype, device=x.device)
           for x in (o, dq, dk, dv)]
    hidden = torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1)
    eps = 2.0 ** -8

    def sq(x):
        return x.square().sum(-1)

    for b in range(B):
        for h in range(H):
            qq, kk, vv, dd = (t[b, :, j] for t, j in ((q, h), (k, h // G),
                                                      (v, h // G), (do, h)))
            s = qq @ kk.t() * scale
            if causal:
                s = s.masked_fill(hidden, -math.inf)
            p = torch.softmax(s, -1)
            oo = p @ vv
            ds = p * (dd @ vv.t() - (dd * oo).sum(-1, keepdim=True)) * scale
            off = 2 * p * (sq(dd * oo)[:, None].sqrt() * scale)
            at = b, slice(None), h
            kv = b, slice(None), h // G
            o[at], dq[at] = oo, ds @ kk
            dk[kv] += ds.t() @ qq
            dv[kv] += p.t() @ dd
            # squares of the limits: sums of squares of the terms
            lim[0][at] = p.square() @ sq(vv)
            lim[1][at] = ds.square() @ sq(kk) + sq(off @ kk)
            lim[2][kv] += (ds.square() + off.square()).t() @ sq(qq)
            lim[3][kv] += p.square().t() @ sq(dd)
    # and fp32's own rounding where all of a row cancels
    return [(x, eps * (y.sqrt() + sq(x).sqrt()) + 1e-5)
            for x, y in zip((o, dq, dk, dv), lim)]


def _close(got, want, what):
    """Every row of every head within its limit."""
    want, lim = want
    over = (got.double() - want).norm(dim=-1) / lim
    assert got.isfinite().all() and (over <= 1).all(), (what, over.max().item())


SHAPES = [(1, 1, 2, 1), (1, 31, 1, 1), (2, 64, 4, 2), (1, 65, 7, 1),
          (1, 127, 3, 3), (1, 128, 14, 2), (2, 129, 4, 1), (1, 255, 8, 8),
          (1, 257, 16, 2), (1, 777, 28, 4)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_flash_attention(shape, d, causal):
    B, S, H, Hkv = shape
    torch.manual_seed(S + d)
    q = torch.randn(B, S, H, d, device="cuda").bfloat16().requires_grad_()
    k, v = (torch.randn(B, S, Hkv, d, device="cuda").bfloat16()
            .requires_grad_() for _ in range(2))
    do = torch.randn(B, S, H, d, device="cuda").bfloat16()
    o = attention.flash_attn_func(q, k, v, causal=causal)
    o.backward(do)
    want = _reference(q, k, v, do, causal, d ** -0.5)
    for got, w, n in zip((o, q.grad, k.grad, v.grad), want,
                         ("o", "dq", "dk", "dv")):
        _close(got, w, n)
    with torch.no_grad():
        assert torch.equal(attention.flash_attn_fwd(q, k, v, causal), o)


@pytest.mark.parametrize("splits", [1, 2, 3, 4])
def test_splits_agree(splits):
    from deepspeed_amd.ops import _C
    torch.manual_seed(0)
    q, do = (torch.randn(2, 300, 8, 128, device="cuda").bfloat16()
             for _ in range(2))
    k, v = (torch.randn(2, 300, 2, 128, device="cuda").bfloat16()
            for _ in range(2))
    o, lse = _C.flash_attn_fwd(q, k, v, 0.09, True, True)
    got = _C.flash_attn_bwd(q, k, v, o, do, lse, 0.09, True, splits)
    for g, w, n in zip(got, _reference(q, k, v, do, True, 0.09)[1:],
                       ("dq", "dk", "dv")):
        _close(g, w, n)


def test_a_scale_that_is_no_number_shows():
    torch.manual_seed(0)
    q, k, v = (torch.randn(1, 40, 2, 64, device="cuda").bfloat16()
               .requires_grad_() for _ in range(3))
    o = attention.flash_attn_func(q, k, v, True, math.nan)
    o.sum().backward()
    assert o.isnan().all() and q.grad.isnan().all() and k.grad.isnan().all()


@pytest.mark.parametrize("scale", [0.3, -0.2, 0.0])
def test_scales_and_strides(scale):
    """Slices of one buffer, as a joint projection leaves them, BHSD views and
    an odd offset; any sign of the scale."""
    torch.manual_seed(0)
    joint = torch.randn(2, 100, 8, 64, device="cuda").bfloat16()
    q, k, v = joint[:, :, :4], joint[:, :, 4:6], joint[:, :, 6:]
    do = torch.randn(2, 4, 100, 64, device="cuda").bfloat16().transpose(1, 2)
    odd = torch.empty(k.numel() + 1, device="cuda").bfloat16()[1:]
    k2 = odd.view(k.shape).copy_(k)
    for kk in (k, k2):
        a, b, c = (t.detach().requires_grad_() for t in (q, kk, v))
        o = attention.flash_attn_func(a, b, c, True, scale)
        o.backward(do)
        want = _reference(q, kk, v, do, True, scale)
        for got, w, n in zip((o, a.grad, b.grad, c.grad), want,
                             ("o", "dq", "dk", "dv")):
            _close(got, w, n)


def test_backward_repeats():
    torch.manual_seed(0)
    q = torch.randn(1, 500, 8, 128, device="cuda").bfloat16().requires_grad_()
    k, v = (torch.randn(1, 500, 2, 128, device="cuda").bfloat16()
            .requires_grad_() for _ in range(2))
    do = torch.randn_like(q)
    o = attention.flash_attn_func(q, k, v)
    a = torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    b = torch.autograd.grad(o, (q, k, v), do)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("given", [False, True])
def test_rope_flash_is_rope_then_flash(d, given):
    from deepspeed_amd.ops.rope import apply_rope, rope_tables
    torch.manual_seed(d)
    cos, sin = rope_tables(d, 200, 1e4, device="cuda")
    q = torch.randn(2, 75, 6, d, device="cuda").bfloat16()
    k, v = (torch.randn(2, 75, 2, d, device="cuda").bfloat16()
            for _ in range(2))
    pos = torch.randint(0, 200, (2, 75), device="cuda", dtype=torch.int32) \
        if given else None
    do = torch.randn_like(q)
    res = []
    for f in (lambda a, b, c: attention.rope_flash_attention(a, b, c, cos, sin,
                                                             pos),
              lambda a, b, c: attention.flash_attn_func(
                  apply_rope(a, cos, sin, pos), apply_rope(b, cos, sin, pos),
                  c)):
        x = [t.clone().requires_grad_() for t in (q, k, v)]
        o = f(*x)
        o.backward(do)
        res.append([o] + [t.grad for t in x])
    assert all(torch.equal(a, b) for a, b in zip(*res))
    with torch.no_grad():
        assert torch.equal(attention.rope_flash_attention(q, k, v, cos, sin,
                                                          pos), res[0][0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16,
                                   torch.float32])
@pytest.mark.parametrize("d,h", [(2, 3), (34, 1), (64, 5), (96, 2), (128, 8)])
def test_rope_pairs(dtype, d, h):
    from deepspeed_amd.ops import _C
    from deepspeed_amd.ops.rope import _torch_rope, rope_tables
    torch.manual_seed(0)
    cos, sin = rope_tables(d, 50, 1e4, device="cuda")
    x = torch.randn(2, 33, h, d, device="cuda").to(dtype)
    y = torch.randn(2, 33, 2, d, device="cuda").to(dtype)
    for back in (False, True):
        got = _C.rope(x, y, cos, sin, None, back)
        for g, t in zip(got, (x, y)):
            torch.testing.assert_close(
                g, _torch_rope(t, cos, sin, None, back),
                rtol=2 * torch.finfo(dtype).eps, atol=1e-6)
        a = x.clone()
        _C.rope(a, None, cos, sin, None, back, True)
        assert torch.equal(a, got[0])
