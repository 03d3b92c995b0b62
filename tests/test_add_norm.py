"""RMS norm of a residual stream with a sublayer's output added: which calls
take the fused kernel, and both ways against fp64."""

import pytest
import torch

from deepspeed_amd.models import llama
from deepspeed_amd.ops.linear import unhooked
from deepspeed_amd.ops.norms import RMSNorm, add_rms_norm, rms_norm


def test_cpu_is_add_then_norm():
    torch.manual_seed(0)
    x, r, w = torch.randn(3, 5, 16), torch.randn(3, 5, 16), torch.randn(16)
    y, s = add_rms_norm(x, r, w, 1e-5)
    assert torch.equal(s, r + x) and torch.equal(y, rms_norm(r + x, w, 1e-5))


def test_hooked_or_replaced_layers_see_their_calls():
    """A hook on a norm or a layer, or another module in its place, gets what
    it got: one tensor in, one out, and the same loss."""
    torch.manual_seed(0)
    model = llama.LlamaForCausalLM(llama.llama_tiny())
    ids = torch.randint(0, 512, (2, 9))
    want = model(ids, labels=ids)
    seen = []
    norm = model.model.layers[1].post_attention_layernorm
    assert unhooked(norm)
    h1 = norm.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    h2 = model.model.layers[0].register_forward_hook(
        lambda m, i, o: seen.append(o.shape))
    assert torch.equal(model(ids, labels=ids), want)
    assert len(seen) == 2
    h1.remove(), h2.remove()

    class Other(torch.nn.Module):
        def forward(self, x):
            return norm(x)

    model.model.layers[1].post_attention_layernorm = Other()
    assert torch.equal(model(ids, labels=ids), want)


@pytest.mark.parametrize("where", ["module", "class"])
@pytest.mark.parametrize("grad", [False, True])
def test_replaced_forwards_are_taken(where, grad, monkeypatch):
    """A forward set on a layer, a norm or a projection, or on its class."""
    torch.manual_seed(0)
    model = llama.LlamaForCausalLM(llama.llama_tiny())
    ids = torch.randint(0, 512, (2, 9))
    layer = model.model.layers[1]
    for mod in (layer, layer.input_layernorm, model.model.norm,
                layer.self_attn.q_proj, layer.mlp.down_proj, model.lm_head):
        with monkeypatch.context() as m, torch.set_grad_enabled(grad):
            want, calls = model(ids), []
            old = type(mod).forward

            def forward(self, x, *a, **k):
                calls.append(0)
                assert not k.keys() - {"positions", "kv_cache"}
                y = old(self, x, *a, **k)
                return 2 * y if self is mod else y

            if where == "class":
                m.setattr(type(mod), "forward", forward)
            else:
                m.setitem(mod.__dict__, "forward", forward.__get__(mod))
            assert not unhooked(mod) and not unhooked(mod, internal_ok=True)
            got = model(ids)
            assert calls and not torch.equal(got, want)
        assert unhooked(mod)


def test_torchs_linear_replaced(monkeypatch):
    model = llama.LlamaForCausalLM(llama.llama_tiny())
    lin = model.lm_head
    monkeypatch.setattr(torch.nn.Linear, "forward", lambda self, x: x)
    assert not unhooked(lin)
    x = torch.randn(2, 64)
    assert lin(x) is x


@pytest.mark.parametrize("name", ["", ".input_layernorm", ".mlp.up_proj"])
def test_compiled_modules_run_compiled(name):
    torch.manual_seed(0)
    model = llama.LlamaForCausalLM(llama.llama_tiny())
    ids = torch.randint(0, 512, (2, 9))
    want = model(ids)
    mod = model.get_submodule("model.layers.0" + name)
    graphs = []
    mod.compile(backend=lambda g, _: graphs.append(g) or g.forward)
    assert not unhooked(mod)
    torch.testing.assert_close(model(ids), want)
    assert graphs


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,h", [(1, 8), (3, 2040), (7, 2048), (1030, 4096),
                                    (5000, 1024), (9, 8192), (4, 8200),
                                    (3, 16384), (5, 20), (2, 16392)])
@pytest.mark.parametrize("used", ["both", "norm", "sum"])
def test_add_norm_gpu(dtype, rows, h, used):
    g = torch.Generator().manual_seed(rows + h)

    def rand(*shape):
        return torch.randn(shape, generator=g).to(dtype).cuda()

    x, r, w = rand(rows, h).requires_grad_(), rand(rows, h), rand(h)
    r.requires_grad_(), w.requires_grad_()
    dy, ds = rand(rows, h), rand(rows, h)
    norm = RMSNorm(h, eps=1e-5)
    norm.weight = torch.nn.Parameter(w.detach().clone())
    y, s = norm(x, residual=r)
    eps = torch.finfo(dtype).eps
    xd, rd, wd = (t.detach().double().requires_grad_() for t in (x, r, w))
    sd = xd + rd
    yd = sd * torch.rsqrt(sd.square().mean(-1, keepdim=True) + 1e-5) * wd
    # a rounding or two of values that are sums of two
    lim = 2 * eps * (1 + yd.abs())
    assert ((y.double() - yd).abs() <= lim).all()
    assert ((s.double() - sd).abs() <= eps * (1 + sd.abs())).all()
    loss = sum((a * b).sum() for a, b, n in ((y, dy, "norm"), (s, ds, "sum"))
               if used in ("both", n))
    want = sum((a * b.double()).sum() for a, b, n in ((yd, dy, "norm"),
                                                      (sd, ds, "sum"))
               if used in ("both", n))
    loss.backward()
    want.backward()
    if used == "sum":
        assert torch.equal(x.grad, ds) and torch.equal(r.grad, ds)
        return
    assert torch.equal(x.grad, r.grad)
    top = xd.grad.abs().amax(-1, keepdim=True) + 1
    assert ((x.grad.double() - xd.grad).abs() <= 4 * eps * top).all()
    got = norm.weight.grad.double()
    # the sum is rounded to 16 bits before the backward reads it again
    assert (got - wd.grad).norm() <= 2 * eps * (wd.grad.norm() + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 4, 1029])
def test_norm_weight_gradient_repeats(rows):
    torch.manual_seed(0)
    x = torch.randn(rows, 1024, device="cuda").bfloat16()
    dy = torch.randn_like(x)
    grads = []
    for _ in range(3):
        w = torch.ones(1024, device="cuda").bfloat16().requires_grad_()
        rms_norm(x, w).backward(dy)
        grads.append(w.grad)
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])


@pytest.mark.parametrize("which", ["fwd", "bias", "bwd", "dy"])
def test_kernels_refuse_other_types(which):
    """A weight, bias or gradient in another type than x's would be read past its
    end, or as other numbers."""
    _C = pytest.importorskip("deepspeed_amd.ops._C")
    x, w = torch.zeros(2, 64), torch.zeros(64)
    bf16 = torch.zeros(64, dtype=torch.bfloat16)
    inv = torch.zeros(2)
    with pytest.raises(RuntimeError, match="types"):
        if which == "fwd":
            _C.norm_fwd(x, bf16, None, 1e-5, False)
        elif which == "bias":
            _C.norm_fwd(x, w, bf16, 1e-5, True)
        elif which == "bwd":
            _C.norm_bwd(x, x, bf16, inv, None, False)
        else:
            _C.norm_bwd(x.bfloat16(), x, w, inv, None, False)


@pytest.mark.parametrize("device", [
    "cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", ["rms", "add", "layer"])
@pytest.mark.parametrize("x_type", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("w_type", [torch.float32, torch.bfloat16])
def test_weights_of_another_type(kind, x_type, w_type, device):
    """The norm in x's type, the gradients each in its own."""
    from deepspeed_amd.ops.norms import layer_norm
    g = torch.Generator().manual_seed(0)
    x, r, dy = (torch.randn(5, 512, generator=g).to(device, x_type)
                for _ in range(3))
    w, b = (torch.randn(512, generator=g).to(device, w_type)
            for _ in range(2))
    ps = [x, w, b] if kind == "layer" else [x, w]
    for p in ps:
        p.requires_grad_()

    def norm(x, w, b=None, r=r, own=True):
        if not own:
            if kind == "layer":
                return torch.nn.functional.layer_norm(x, (512,), w, b, 1e-5)
            x = x + r.double() if kind == "add" else x
            return x * torch.rsqrt(x.square().mean(-1, keepdim=True)
                                   + 1e-5) * w
        if kind == "layer":
            return layer_norm(x, w, b, 1e-5)
        return add_rms_norm(x, r, w, 1e-5)[0] if kind == "add" else \
            rms_norm(x, w, 1e-5)

    y = norm(*ps)
    got = [y, *torch.autograd.grad(y, ps, dy)]
    assert [t.dtype for t in got] == [x_type] + [p.dtype for p in ps]
    qs = [p.detach().double().requires_grad_() for p in ps]
    y = norm(*qs, own=False)
    for a, c in zip(got, [y, *torch.autograd.grad(y, qs, dy.double())]):
        # fp32 within, rounded to the result's type; the sum of add to x's, too
        half = torch.bfloat16 in (a.dtype, x_type)
        assert (a.double() - c).norm() <= \
            (2.0 ** -7 if half else 2.0 ** -18) * c.norm()
