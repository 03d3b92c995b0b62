"""Serving steps whose decoder layers run as native calls: the same outputs and
cache as the modules give one by one (GPU), and what keeps the modules called
(CPU)."""

import pytest
import torch
import torch.nn as nn

from deepspeed_amd.inference.ragged import PagedKVCache
from deepspeed_amd.linear.optimized_linear import (QuantizationConfig,
                                                   WOQLinear)
from deepspeed_amd.models import llama


def _model(device, bias=False, int8=False):
    torch.manual_seed(0)
    cfg = llama.LlamaConfig(vocab_size=500, hidden_size=512,
                            intermediate_size=768, num_layers=3, num_heads=4,
                            num_kv_heads=2, max_seq_len=512,
                            attention_bias=bias)
    model = llama.LlamaForCausalLM(cfg).to(device, torch.bfloat16).eval()
    model.requires_grad_(False)
    if bias:
        for p in model.named_parameters():
            if p[0].endswith("bias"):
                p[1].normal_()
    if int8:
        for m in list(model.modules()):
            for name, lin in list(m.named_children()):
                if isinstance(lin, nn.Linear):
                    setattr(m, name, WOQLinear(lin, QuantizationConfig()))
    return model, cfg


def test_operands():
    """A hook, a replaced forward, another class anywhere in the layer: its
    modules are called."""
    model, _ = _model("cpu")
    layer = model.model.layers[0]
    assert llama._operands(layer, 1) is not None
    for m in (layer.self_attn, layer.mlp, layer.input_layernorm,
              layer.self_attn.o_proj, layer.mlp.down_proj):
        h = m.register_forward_hook(lambda *a: None)
        assert llama._operands(layer, 1) is None
        h.remove()
        m.forward = lambda x: x
        assert llama._operands(layer, 1) is None
        del m.forward
    # the norms' calls do not take place, so neither would their hooks
    for norm in (layer.input_layernorm, layer.post_attention_layernorm):
        def fetch(*a):
            return None
        fetch._ds_internal = True
        h = norm.register_forward_pre_hook(fetch)
        assert llama._operands(layer, 1) is None
        h.remove()
    own = type("Own", (llama.LlamaMLP,), {})
    layer.mlp.__class__ = own
    assert llama._operands(layer, 1) is None
    layer.mlp.__class__ = llama.LlamaMLP
    layer.chain = lambda *a: a
    assert llama._operands(layer, 1) is None
    del layer.chain
    layer.mlp.up_proj = nn.Linear(512, 768, bias=False)
    assert llama._operands(layer, 1) is None
    model, _ = _model("cpu", int8=True)
    assert llama._operands(model.model.layers[0], 64) is not None
    assert llama._operands(model.model.layers[0], 65) is None


def test_plan_is_the_caches_own():
    """With methods of another kind, a mask of the caller's or outside a step
    there is no plan."""
    x = torch.zeros(1, 1, 512)
    cache = PagedKVCache(1, 1, 2, 64, 128)
    assert cache.layers_plan(x, 4, 2) is None
    cache.begin_step([0], 1)
    cache.last_mask = None
    assert cache.layers_plan(x, 4, 2) is None
    sub = type("Sub", (PagedKVCache,), {})(1, 1, 2, 64, 128)
    sub.begin_step([0], 1)
    assert sub.layers_plan(x, 4, 2) is None


@pytest.mark.parametrize("where", ["weight", "bias", "scales", "norm",
                                   "delta"])
def test_refused(where):
    """Before anything is launched: tensors on another device, whichever product
    reads them, and an fp32 delta that is no layer's sums in parts."""
    _C = pytest.importorskip("deepspeed_amd.ops._C")
    bf16 = dict(dtype=torch.bfloat16)
    ws = [torch.zeros(512, 512, **bf16) for _ in range(7)]
    norms, bs, scales = [torch.zeros(512, **bf16)] * 2, [None] * 7, []
    delta = None
    if where == "weight":
        ws[3] = ws[3].to("meta")
    elif where == "bias":
        bs[2] = torch.zeros(512, device="meta", **bf16)
    elif where == "scales":
        scales = [torch.zeros(128)] * 6 + [torch.zeros(128, device="meta")]
    elif where == "norm":
        norms = [norms[0], norms[1].to("meta")]
    else:
        delta = torch.zeros(1, 20, 512)
    pool, plan = torch.zeros(1, 4, 64, 128, **bf16), torch.zeros(
        99, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="delta" if where == "delta" else
                       "on different devices"):
        _C.paged_decoder_layer(
            torch.zeros(1, 20, 512, **bf16), delta, norms, 1e-6, 1e-6, ws,
            scales, bs, 2048, torch.zeros(64, 64), torch.zeros(64, 64), None,
            20, pool, pool, plan[:20], plan, 1, 1, 1, False, 1, 1.0,
            False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "bias", "int8"])
@pytest.mark.parametrize("positions", [False, True])
@torch.no_grad()
def test_same_as_modules_gpu(kind, positions, monkeypatch):
    model, cfg = _model("cuda", kind == "bias", kind == "int8")
    # prompt portions, single tokens, both packed; rows on either side of each
    # kernel's line
    steps = [([0], 20, None), ([1], 33, None), ([2], 130, None),
             ([0, 1, 2], 1, None), ([2] * 2 + [0] * 30, 1,
                                    [0, 1] + list(range(30))), ([1], 1, None)]
    calls = []
    native = llama.get_ext().paged_decoder_layer

    class Ext:
        def __getattr__(self, name):
            return getattr(ext, name)

        def paged_decoder_layer(self, *a):
            calls.append(1)
            return native(*a)

    ext = llama.get_ext()
    monkeypatch.setattr(llama, "get_ext", Ext)
    out = []
    for own in (True, False):
        if not own:
            monkeypatch.setattr(llama.LlamaModel, "_paged_plan",
                                lambda *a: None)
        g = torch.Generator().manual_seed(1)
        cache = PagedKVCache(3, 3, 2, 512, 128, dtype=torch.bfloat16,
                             device="cuda")
        got = []
        for slots, n, offsets in steps:
            if offsets is not None and not positions:
                continue            # rows of one slot stand at their own places
            ids = torch.randint(0, 500, (len(slots), n), generator=g)
            start = cache.lens[slots]
            if offsets is not None:
                start = start + torch.tensor(offsets)
            pos = (start[:, None] + torch.arange(n)).int().cuda()
            cache.begin_step(slots, n, offsets=offsets)
            got.append(model(ids.cuda(), positions=pos if positions else None,
                             kv_cache=cache))
            assert cache.last_decoded == (n == 1)
            cache.end_step()
        out.append(got + cache.k + cache.v)
    rows = [len(s) * n for s, n, o in steps if positions or o is None]
    want = sum(3 for r in rows if kind != "int8" or r <= 64)
    assert len(calls) == want
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads", [(2, 1), (32, 8), (36, 18),
                                            (56, 8)])
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("int8", [False, True])
@torch.no_grad()
def test_append_with_the_products_gpu(heads, kv_heads, rows, int8, monkeypatch):
    """q, k and v turned and written by their products, bit by bit as behind
    them: one and two pairs of tiles a wave, a tile and several a workgroup; and
    these near fp32."""
    torch.manual_seed(rows)
    cfg = llama.LlamaConfig(vocab_size=64, hidden_size=heads * 128,
                            intermediate_size=256, num_layers=1,
                            num_heads=heads, num_kv_heads=kv_heads,
                            max_seq_len=256, attention_bias=True)
    model = llama.LlamaForCausalLM(cfg).to("cuda", torch.bfloat16).eval()
    attn = model.model.layers[0].self_attn
    for lin in (attn.q_proj, attn.k_proj, attn.v_proj):
        lin.bias.data.normal_()
    refs = [(lin.weight.float(), lin.bias.float())
            for lin in (attn.q_proj, attn.k_proj, attn.v_proj)]
    if int8:
        for m in (attn, model.model.layers[0].mlp):
            for name, lin in list(m.named_children()):
                setattr(m, name, WOQLinear(lin, QuantizationConfig()))
    ids = torch.randint(0, 64, (rows, 1), device="cuda")
    pos = torch.arange(rows, device="cuda", dtype=torch.int32)[:, None] + 3
    calls, native = [], llama.get_ext().paged_decoder_layer
    monkeypatch.setattr(llama.get_ext(), "paged_decoder_layer",
                        lambda *a: calls.append(1) or native(*a))
    out = []
    for own in (True, False):
        if not own:
            monkeypatch.setattr(llama.LlamaModel, "_paged_plan",
                                lambda *a: None)
        cache = PagedKVCache(1, rows, kv_heads, 256, 128,
                             dtype=torch.bfloat16, device="cuda")
        for s in range(rows):
            cache.begin_step([s], 3 + s)
            cache.end_step()
        cache.begin_step(list(range(rows)), 1)
        got = model(ids, positions=pos, kv_cache=cache)
        cache.end_step()
        out.append((got, cache.k[0], cache.v[0]))
    assert len(calls) == 1
    for a, b in zip(*out):
        assert torch.equal(a, b)
    # the pool's rows against fp32 products
    norm = model.model.layers[0].input_layernorm
    h = norm(model.model.embed_tokens(ids))[:, 0].float()
    k, v = ((h @ w.t() + b).view(rows, kv_heads, 128) for w, b in refs[1:])
    inv = cfg.rope_theta ** (-torch.arange(64, device="cuda") / 64.0)
    c, s = (f(pos * inv)[:, None] for f in (torch.cos, torch.sin))
    k1, k2 = k[..., :64], k[..., 64:]
    k = torch.cat([k1 * c - k2 * s, k2 * c + k1 * s], -1)
    for pool, want in ((out[0][1], k), (out[0][2], v)):
        rows_of = torch.stack([
            pool[cache.block_table[r][(3 + r) // cache.block_size], :,
                 (3 + r) % cache.block_size].float() for r in range(rows)])
        # bf16 outputs, and int8 weights within half a step of max / 127
        bound = 0.02 if int8 else 0.006
        assert (rows_of - want).norm() <= bound * want.norm()


class _Strided(llama.LlamaDecoderLayer):
    """Hands on a stream that lies across."""

    def forward(self, *a):
        y = super().forward(*a)
        return y.transpose(1, 2).contiguous().transpose(1, 2)


class _Offset(llama.LlamaMLP):
    """Its output starts off 16 bytes."""

    def forward(self, x):
        y = super().forward(x)
        return torch.cat([y.new_zeros(1), y.flatten()])[1:].view_as(y)


class _Masked(llama.LlamaDecoderLayer):
    """Sets the step's mask for the layers behind it: nothing but itself."""

    def forward(self, x, cos, sin, positions, kv_cache):
        y = super().forward(x, cos, sin, positions, kv_cache)
        kv_cache.last_mask = torch.eye(
            x.shape[1], dtype=torch.bool, device=x.device)[None, None]
        return y


class _Fp32(llama.LlamaDecoderLayer):
    def forward(self, *a):
        return super().forward(*a).float()


@pytest.mark.gpu
@pytest.mark.parametrize("own", [_Strided, _Offset, _Masked, _Fp32])
@torch.no_grad()
def test_behind_other_classes_gpu(own, monkeypatch):
    """What a layer or MLP of another class hands on reaches the layers behind it
    as if there were modules only, or is refused as there."""
    def attention(q, k, v, causal=True, attn_mask=None):
        # masked attention by the library's batched products has faulted GPUs
        assert attn_mask is not None
        return sdpa(*(t.float().cpu() for t in (q, k, v)), causal,
                    attn_mask.cpu()).to(q)

    sdpa = llama.sdpa_gqa
    monkeypatch.setattr(llama, "sdpa_gqa", attention)
    model, _ = _model("cuda")
    part = model.model.layers[1]
    part = part.mlp if issubclass(own, llama.LlamaMLP) else part
    part.__class__ = own
    ids = torch.randint(0, 500, (1, 20), device="cuda")
    out = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(llama.LlamaModel, "_paged_plan",
                                lambda *a: None)
        cache = PagedKVCache(3, 1, 2, 512, 128, dtype=torch.bfloat16,
                             device="cuda")
        cache.begin_step([0], 20)
        if own is _Fp32:
            with pytest.raises(RuntimeError, match="same dtype"):
                model(ids, kv_cache=cache)
            continue
        out.append(model(ids, kv_cache=cache))
    assert own is _Fp32 or torch.equal(*out)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "bias"])
def test_sums_in_parts_gpu(kind, monkeypatch):
    """Long contractions are split, and what reads their sums next adds them up."""
    x = torch.zeros(20, 2048, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(2048, 2048, device="cuda", dtype=torch.bfloat16)
    with torch.profiler.profile() as prof:
        llama.get_ext().tile_linear(x, [w], [None], 0)
        torch.cuda.synchronize()
    assert any("tile_merge" in e.key for e in prof.key_averages())

    class Wide(llama.LlamaConfig):
        def __init__(self, **kw):
            for name in ("hidden_size", "intermediate_size", "num_heads"):
                kw[name] *= 4
            super().__init__(**kw)

    monkeypatch.setattr(llama, "LlamaConfig", Wide)
    test_same_as_modules_gpu(kind, True, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads", [(8, 4), (16, 8), (18, 6), (24, 6)])
@pytest.mark.parametrize("rows", [1, 9, 32])
@pytest.mark.parametrize("int8", [False, True])
def test_append_up_to_a_round_gpu(heads, kv_heads, rows, int8, monkeypatch):
    """Bit by bit also where the products alone have a tile of 16 features a
    workgroup and those that append pairs of them: up to 256 tiles, and more."""
    test_append_with_the_products_gpu(heads, kv_heads, rows, int8, monkeypatch)
