"""Linear layers of a few rows: which calls take the kernel (CPU) and the kernel
against fp64 products of the same weights (GPU)."""

import pytest
import torch
import torch.nn as nn

from deepspeed_amd.linear.optimized_linear import (QuantizationConfig,
                                                   WOQLinear)
from deepspeed_amd.ops import linear as L
from deepspeed_amd.ops.linear import (SWIGLU, rows_linear, tile_linear,
                                      unhooked, untransformed)


def test_unhooked():
    lin = nn.Linear(8, 8)
    assert unhooked(lin)
    for register in (lin.register_forward_hook,
                     lin.register_forward_pre_hook,
                     lin.register_full_backward_hook,
                     lin.register_full_backward_pre_hook):
        h = register(lambda *a: None)
        assert not unhooked(lin)
        h.remove()
    h = nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not unhooked(lin)
    h.remove()
    assert unhooked(lin)


def test_cpu_and_grad_calls_are_left_alone():
    lin = nn.Linear(256, 16).bfloat16()
    x = torch.randn(2, 256).bfloat16()
    with torch.no_grad():
        assert rows_linear(x, (lin,)) is None
    assert rows_linear(x, (lin,)) is None


def _under_transforms(f, x, all=True):
    """f(x) as transforms, tangents, a trace and a dispatch mode make the
    call, by name."""
    import torch.autograd.forward_ad as fwad
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode
    out = {"vmap": torch.func.vmap(f)(x)}
    with fwad.dual_level():
        out["dual"] = fwad.unpack_dual(f(fwad.make_dual(x, 2 * x))).tangent
    with FlopCounterMode(display=False) as mode:
        f(x)
    out["flops"] = mode.get_total_flops()
    if not all:
        return out
    out["jvp"] = torch.func.jvp(f, (x,), (2 * x,))[1]
    # traced on one input, run on another
    out["make_fx"] = make_fx(f)(x)(3 * x)
    out["trace"] = torch.jit.trace(f, x, check_trace=False)(3 * x)
    return out


def test_untransformed():
    seen = []

    def f(x):
        seen.append(untransformed())
        return x @ x.t()

    f(torch.ones(2, 2))
    assert seen == [True]
    seen.clear()
    with torch.no_grad():
        assert untransformed()
        _under_transforms(f, torch.ones(2, 2, 2)[0])
    assert len(seen) >= 6 and not any(seen)
    assert untransformed()


def _layer(n, k, bias, int8, g):
    lin = nn.Linear(k, n, bias=bias).bfloat16().cuda()
    with torch.no_grad():
        lin.weight.copy_(0.05 * torch.randn(n, k, generator=g))
        if bias:
            lin.bias.copy_(torch.randn(n, generator=g))
    w = lin.weight.double()
    if int8:
        lin = WOQLinear(lin, QuantizationConfig())
        q, s = lin.qweight.q, lin.qweight.scales
        w = (q.double() * s.double().repeat_interleave(2048)[:n * k]).view(n,
                                                                          k)
    b = lin.bias.double() if bias else 0.0
    return lin, lambda x: x.double() @ w.t() + b


def _close(got, want):
    # fp32 sums rounded to bf16 once
    err = (got.double() - want).abs()
    lim = 2.0 ** -8 * want.abs() + 2.0 ** -16 * want.abs().max()
    assert (err <= lim).all(), (err / lim).max()


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("sizes", [((37,), 256), ((6144,), 512),
                                   ((14336,), 256), ((256, 24, 40), 3072)])
@torch.no_grad()
def test_rows_linear_gpu(int8, m, sizes):
    ns, k = sizes
    g = torch.Generator().manual_seed(m)
    both = [_layer(n, k, i % 2 == 0, int8, g) for i, n in enumerate(ns)]
    x = torch.randn(1, m, k, generator=g).bfloat16().cuda()
    got = rows_linear(x, [b[0] for b in both])
    if m > (64 if int8 else 32):
        assert got is None
        return
    for (lin, want), y in zip(both, got):
        assert y.shape == (1, m, y.shape[-1])
        _close(y, want(x))
    if int8:
        _close(both[0][0](x), both[0][1](x))
    h = both[0][0].register_forward_hook(lambda *a: None)
    assert rows_linear(x, (both[0][0],)) is None
    h.remove()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [33, 48, 49, 64, 65, 80, 96, 112, 127, 128, 129,
                               200, 225, 256, 257])
@pytest.mark.parametrize("sizes", [((4, 132, 124), 256), ((100, 36), 512),
                                   ((1024, 256, 256), 1280),
                                   ((128,), 131072)])
@torch.no_grad()
def test_batch_linear_gpu(m, sizes):
    ns, k = sizes
    g = torch.Generator().manual_seed(m)
    both = [_layer(n, k, i % 2 == 0, False, g) for i, n in enumerate(ns)]
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    assert rows_linear(x, [b[0] for b in both]) is None
    got = tile_linear(x, [b[0] for b in both])
    for (lin, want), y in zip(both, got):
        _close(y, want(x))
    assert rows_linear(x, [both[0][0]] * 2, SWIGLU) is None


@pytest.mark.gpu
@pytest.mark.parametrize("m", [32, 33])
@torch.no_grad()
def test_longest_contractions_gpu(m):
    """Past what the tiled kernel takes, 33 rows and more are the module's own."""
    lin = nn.Linear(L.INPUTS + 256, 4, bias=False, device="cuda",
                    dtype=torch.bfloat16)
    x = torch.randn(m, L.INPUTS + 256, device="cuda").bfloat16()
    assert (rows_linear(x, (lin,)) is not None) == (m <= 32)
    assert m <= 32 or tile_linear(x, (lin,)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("m", [1, 16, 17, 32, 50])
@torch.no_grad()
def test_rows_swiglu_gpu(int8, m):
    g = torch.Generator().manual_seed(m)
    (gate, fg), (up, fu) = (_layer(1000, 512, False, int8, g)
                            for _ in range(2))
    x = torch.randn(m, 512, generator=g).bfloat16().cuda()
    got = rows_linear(x, (gate, up), SWIGLU)
    if m > 32 and not int8:
        assert got is None
        return
    y, = got
    _close(y, torch.nn.functional.silu(fg(x)) * fu(x))


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@torch.no_grad()
def test_under_transforms_gpu(int8):
    """A layer's call as a model makes it, and a quantized layer's own (whose
    dequantization no tangent transform and no trace has ever passed)."""
    lin, want = _layer(64, 256, False, int8, torch.Generator().manual_seed(0))
    x = torch.randn(4, 256, device="cuda").bfloat16()
    assert rows_linear(x, (lin,)) is not None
    lin.requires_grad_(False)      # constants of a trace

    def call(x):
        y = rows_linear(x, (lin,))
        return lin(x) if y is None else y[0]

    got = _under_transforms(lin if int8 else call, x, all=not int8)
    assert got.pop("flops") == 2 * 4 * 64 * 256
    for name, y in got.items():
        scale = {"vmap": 1, "jvp": 2, "dual": 2, "make_fx": 3, "trace": 3}[name]
        err = y.double() - scale * want(x)
        # weights rounded to bf16 on this way round, and inputs 3 * x
        assert err.norm() <= 0.01 * scale * want(x).norm(), name


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@torch.no_grad()
def test_replaced_forward_gpu(int8):
    lin, _ = _layer(64, 256, False, int8, torch.Generator().manual_seed(0))
    x = torch.randn(2, 256, device="cuda").bfloat16()
    want = rows_linear(x, (lin,))[0]
    lin.forward = lambda x: 0 * x
    assert rows_linear(x, (lin,)) is None
    del lin.forward
    assert torch.equal(rows_linear(x, (lin,))[0], want)
    if int8:
        w = 2 * lin.qweight.dequantized()
        lin.qweight.dequantized = lambda: w
        assert rows_linear(x, (lin,)) is None
        _close(lin(x), x.double() @ w.double().t())


@pytest.mark.gpu
@torch.no_grad()
def test_model_with_and_without_rows_linear(monkeypatch):
    """A decoding step's logits by either way, through a whole model."""
    from deepspeed_amd.models import llama
    torch.manual_seed(0)
    cfg = llama.LlamaConfig(vocab_size=1000, hidden_size=512,
                            intermediate_size=768, num_layers=2, num_heads=4,
                            num_kv_heads=2, max_seq_len=64,
                            attention_bias=True)
    model = llama.LlamaForCausalLM(cfg).bfloat16().cuda().eval()
    ids = torch.randint(0, 1000, (3, 7), device="cuda")
    a = model(ids).float()
    monkeypatch.setattr(llama, "rows_linear", lambda *a, **k: None)
    b = model(ids).float()
    assert (a - b).norm() < 0.02 * b.norm()
