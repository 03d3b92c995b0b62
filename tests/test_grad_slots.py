"""Weights' gradients written to their places in ZeRO's flat buffers: the same
values as added up there, for weights of one layer, of several, tied ones and
ones that no gradient reaches, over passes with and without accumulation."""

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from deepspeed_amd.ops import linear as L
from .common import run_distributed


class Net(torch.nn.Module):
    def __init__(self, device="cpu"):
        super().__init__()
        torch.manual_seed(3)

        def layer(bias=False):
            return torch.nn.Linear(64, 64, bias=bias).to(device)
        self.one, self.biased, self.twice = layer(), layer(True), layer()
        self.tied, self.around, self.out = layer(), layer(), layer()
        self.spare = layer()

    @staticmethod
    def apply_(mod, x):
        return torch.tanh(L._Linears.apply(x, False, mod.weight, mod.bias))

    def forward(self, x, labels):
        x = self.apply_(self.one, x)
        x = self.apply_(self.twice, self.apply_(self.twice, x))
        x = self.apply_(self.biased, x + self.tied.weight[:4].mean(0))
        x = self.apply_(self.tied, x)
        # beside its own product, one in a pass of its own
        x = checkpoint(lambda y: torch.tanh(y @ self.around.weight), x,
                       use_reentrant=True) + self.apply_(self.around, x)
        # written, and then not handed on
        dead = L._Linears.apply(x.detach(), False, self.spare.weight, None)
        return (self.apply_(self.out, x).float() - labels).square().mean() + \
            0.0 * dead.detach().sum()


def _grads(stage, gas, own, device="cpu", rows=4):
    import deepspeed_amd
    engine, opt, _, _ = deepspeed_amd.initialize(model=Net(device), config={
        "train_micro_batch_size_per_gpu": rows,
        "gradient_accumulation_steps": gas, "bf16": {"enabled": True},
        "zero_optimization": {"stage": stage},
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}})
    named = list(engine.module.named_parameters())
    if not own:
        opt.drop_slots()
    given = []
    for name, p in named:
        slot = L.slot_of(p)
        assert (slot is not None) == own
        if slot is not None:
            class Seen(L.GradSlot):
                __slots__ = ("name",)

                def take(self):
                    out = super().take()
                    if out is not None:
                        given.append(self.name)
                    return out
            seen = Seen(p, slot.view)
            seen.name = name
            opt._slots = [(q, seen if q is p else s, b)
                          for q, s, b in opt._slots]
    places = {n: p.grad.data_ptr() for n, p in named}
    g = torch.Generator().manual_seed(0)
    out = []
    for _ in range(2 * gas):
        x = torch.randn(rows, 64, generator=g).bfloat16().to(device)
        y = torch.randn(rows, 64, generator=g).to(device)
        loss = engine(x, labels=y)
        if len(out) == 1:       # seen by the caller: added up
            h = dict(named)["out.weight"].register_hook(lambda t: t * 2)
        engine.backward(loss)
        out.append({n: p.grad.clone() for n, p in named})
        if len(out) == 1 + 1:
            h.remove()
        for n, p in named:
            assert p.grad.data_ptr() == places[n], n
        engine.step()
    out.append({n: p.detach().clone() for n, p in named})
    assert not any(s.open or s.void or s.uses for _, s, _ in opt._slots)
    engine.destroy()
    return out, given


def _check(rank, world, stage, gas):
    got, given = _grads(stage, gas, True)
    want, _ = _grads(stage, gas, False)
    for a, b in zip(got, want):
        for n in b:
            # gradients of three sources are added in another order
            exact = "around" not in n
            assert torch.allclose(a[n].float(), b[n].float(),
                                  rtol=0 if exact else 2.0 ** -6,
                                  atol=0 if exact else 1e-4), n
    assert not got[0]["spare.weight"].any()
    # not: a first layer's (without its input's gradient the weight is not kept),
    # one of two products, and one whose gradient a hook sees
    first = ["out.weight", "around.weight", "tied.weight", "biased.weight"]
    second = first[1:] if gas == 1 else first
    assert given == first + second, given


@pytest.mark.parametrize("world", [1, 2])
@pytest.mark.parametrize("stage,gas", [(1, 1), (2, 1), (2, 2)])
def test_same_gradients(world, stage, gas):
    run_distributed(_check, world_size=world, args=(stage, gas))


def _seen(rank, world):
    """What reads the parameters' gradients in the backward finds the buffers."""
    import deepspeed_amd
    engine, opt, _, _ = deepspeed_amd.initialize(model=Net(), config={
        "train_micro_batch_size_per_gpu": 4, "bf16": {"enabled": True},
        "zero_optimization": {"stage": 2},
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}})
    named = dict(engine.module.named_parameters())
    # those used outside of their products as well come to theirs at the end
    places = {n: p.grad.data_ptr() for n, p in named.items()
              if n not in ("tied.weight", "around.weight")}
    seen = []

    def read(grad):
        assert all(named[n].grad.data_ptr() == places[n] for n in places)
        seen.append({n: named[n].grad.clone() for n in places})

    apply_ = engine.module.apply_

    def watched(mod, x):
        y = apply_(mod, x)
        y.register_hook(read)
        return y

    engine.module.apply_ = watched
    g = torch.Generator().manual_seed(0)
    for _ in range(2):
        x = torch.randn(4, 64, generator=g).bfloat16()
        loss = engine(x, labels=torch.randn(4, 64, generator=g))
        del seen[:]
        engine.backward(loss)
        assert len(seen) == 7
        # nothing has arrived at first; the last layer's is there when the one
        # before it is reached, and stays
        assert not any(v.any() for v in seen[0].values())
        for s in seen[1:]:
            assert torch.equal(s["out.weight"], named["out.weight"].grad)
        engine.step()
    engine.destroy()


def test_gradients_are_seen_in_the_backward():
    run_distributed(_seen, world_size=1)


def _saved(rank, world, path):
    import deepspeed_amd
    from torch.multiprocessing.reductions import StorageWeakRef
    engine, opt, _, _ = deepspeed_amd.initialize(
        model=torch.nn.Linear(1000, 1000), config={
            "train_micro_batch_size_per_gpu": 1, "bf16": {"enabled": True},
            "zero_optimization": {"stage": 2},
            "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}})
    lin = engine.module
    named = dict(lin.named_parameters())
    assert all(L.slot_of(p) is not None for p in named.values())
    torch.save(named, path)
    back = torch.load(path, weights_only=True)
    for n, p in named.items():
        assert torch.equal(back[n], p) and L.slot_of(back[n]) is None
    torch.save(lin.state_dict(keep_vars=True), path)
    assert list(torch.load(path, weights_only=True)) == list(named)
    # without its owner a place is gone, and with it the buffer
    flat = StorageWeakRef(opt.buckets[0].grad_flat.untyped_storage())
    engine.destroy()
    assert all(L.slot_of(p) is None for p in named.values())
    del engine, opt
    lin.zero_grad(set_to_none=True)
    import gc
    gc.collect()
    assert flat.expired()


def test_saved_parameters_hold_no_places(tmp_path):
    run_distributed(_saved, world_size=1, args=(str(tmp_path / "m.pt"),))


def test_place_of_another_parameter():
    """A place is its parameter's, and gone with its owner."""
    a, b = (torch.nn.Parameter(torch.zeros(4)) for _ in range(2))
    slot, key = L.GradSlot(a, torch.zeros(4)), id(a)
    assert L.slot_of(a) is slot and L.slot_of(b) is None
    newer = L.GradSlot(a, torch.zeros(4))
    del slot
    assert L.slot_of(a) is newer
    del a       # the id stays the parameter's while there is a place
    assert L.slot_of(newer.weight) is newer and id(newer.weight) == key
    del newer
    assert key not in L._slots


@pytest.mark.gpu
def test_same_gradients_gpu(monkeypatch):
    """By the tiled kernel, its split sums and the library."""
    import os
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29547")
    for rows in (4, 200, 3000):
        got, given = _grads(2, 1, True, "cuda", rows)
        want, _ = _grads(2, 1, False, "cuda", rows)
        assert len(given) == 7
        for n in want[0]:
            if "around" not in n:
                assert torch.equal(got[0][n], want[0][n]), n


def _model_grads(own, gas, tied, tokens, frozen=False):
    """Gradients and weights of a model's steps; the second batch has none of the
    first one's tokens, so that rows of the table are to be zero again."""
    import deepspeed_amd
    from deepspeed_amd.models import llama
    torch.manual_seed(0)
    cfg = llama.LlamaConfig(vocab_size=512, hidden_size=256,
                            intermediate_size=512, num_layers=2, num_heads=2,
                            num_kv_heads=1, max_seq_len=4096,
                            tie_embeddings=tied)
    model = llama.LlamaForCausalLM(cfg).cuda()
    if frozen:
        model.model.norm.weight.requires_grad_(False)
    engine, opt, _, _ = deepspeed_amd.initialize(model=model, config={
        "train_micro_batch_size_per_gpu": 3,
        "gradient_accumulation_steps": gas, "bf16": {"enabled": True},
        "zero_optimization": {"stage": 2}, "gradient_clipping": 1.0,
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}})
    named = dict(engine.module.named_parameters())
    taken = []
    if not own:
        opt.drop_slots()
    else:
        class Seen(L.GradSlot):
            __slots__ = ("name",)

            def take(self):
                out = super().take()
                if out is not None:
                    taken.append(self.name)
                return out

        slots = {}
        for n, p in named.items():
            if L.slot_of(p) is not None:
                slots[p] = Seen(p, L.slot_of(p).view)
                slots[p].name = n
        opt._slots = [(p, slots[p], b) for p, _, b in opt._slots]
    g = torch.Generator().manual_seed(1)
    out = []
    for i in range(3 * gas):
        lo = 256 * (i % 2)
        ids = torch.randint(lo, lo + 256, (3, tokens // 3), generator=g).cuda()
        engine.backward(engine(ids, labels=ids))
        out.append({n: p.grad.clone() for n, p in named.items()
                    if p.grad is not None})
        engine.step()
    out.append({n: p.detach().clone() for n, p in named.items()})
    engine.destroy()
    return out, set(taken)


@pytest.mark.gpu
@pytest.mark.parametrize("gas,tied,tokens,frozen", [
    (1, False, 600, False), (2, False, 600, False), (1, True, 600, False),
    (1, False, 9000, False), (1, False, 600, True)])
def test_places_of_a_model_gpu(gas, tied, tokens, frozen):
    """Embedding, norms and layers, each in its place, as added up there: over
    accumulation, with a tied head, with a head in several chunks."""
    import os
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29548")
    got, taken = _model_grads(True, gas, tied, tokens, frozen)
    want, none = _model_grads(False, gas, tied, tokens, frozen)
    assert not none
    norms = {n for n in got[-1] if "norm" in n}
    if frozen:
        norms.remove("model.norm.weight")
    assert norms <= taken
    # several uses of one weight are added up
    assert ("model.embed_tokens.weight" in taken) == (not tied)
    assert ("lm_head.weight" in taken) == (not tied and tokens <= 8192)
    for a, b in zip(got, want):
        assert a.keys() == b.keys()
        for n in b:
            # one rounding to bf16 either way, but where two are added up first
            if tied and "embed" in n or tokens > 8192 and "lm_head" in n:
                assert torch.allclose(a[n].float(), b[n].float(),
                                      rtol=2.0 ** -6, atol=1e-3), n
            elif gas == 1 and not tied:
                assert torch.equal(a[n], b[n]), n
            else:
                assert (a[n].float() - b[n].float()).norm() <= \
                    2.0 ** -6 * b[n].float().norm(), n


@pytest.mark.gpu
@pytest.mark.parametrize("rows,h", [(3, 8), (700, 1024), (40, 8192), (5, 9000),
                                    (9, 33)])
@pytest.mark.parametrize("dres", [False, True])
def test_norm_gradient_in_its_type_gpu(rows, h, dres):
    """As the fp32 one rounded, by the rows kernel and the general one."""
    from deepspeed_amd.ops import _C
    g = torch.Generator().manual_seed(h)
    x, dy, r = (torch.randn(rows, h, generator=g).bfloat16().cuda()
                for _ in range(3))
    w = torch.randn(h, generator=g).bfloat16().cuda()
    inv = torch.rand(rows, generator=g).cuda()
    r = r if dres else None
    dx, dw, _ = _C.norm_bwd(dy, x, w, inv, None, False, r)
    into = torch.empty_like(w)
    dx2, dw2, _ = _C.norm_bwd(dy, x, w, inv, None, False, r, into)
    assert dw2.data_ptr() == into.data_ptr()
    # the general kernel adds rows up with atomics, in any order
    exact = h % 8 == 0 and h <= 8192
    assert torch.equal(dx, dx2)
    torch.testing.assert_close(dw2, dw.bfloat16(), rtol=0 if exact else 2.0**-7,
                               atol=0 if exact else 1e-4)
