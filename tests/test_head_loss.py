"""The head's loss over chunks of rows as one node (ops/cross_entropy.py)."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from deepspeed_amd.models.llama import chunked_cross_entropy
from deepspeed_amd.ops import cross_entropy, linear


@pytest.mark.gpu
@pytest.mark.parametrize("n,rows", [(300, 128), (512, 256), (257, 256),
                                    (6400, 3200), (6144, 3200), (9000, 8192)])
@pytest.mark.parametrize("v", [1000, 1088])
@pytest.mark.parametrize("frozen", [None, "x", "w"])
def test_against_fp32_gpu(n, rows, v, frozen):
    """Whole and ragged chunks; products of the library and of the kernels, with
    and without transposed copies; one of the gradients not asked for."""
    g = torch.Generator(device="cuda").manual_seed(n + v)
    h = 1024 if rows > 3000 else 256
    x = torch.randn(1, n, h, device="cuda", generator=g).bfloat16()
    head = linear.Linear(h, v, bias=False).to("cuda", torch.bfloat16)
    head.weight.data.normal_(0.0, 0.05, generator=g)
    labels = torch.randint(0, v, (n,), device="cuda", generator=g)
    labels[::7] = -100
    x.requires_grad_(frozen != "x")
    head.weight.requires_grad_(frozen != "w")
    assert cross_entropy.head_loss_fits(head, x.view(n, h))
    loss = chunked_cross_entropy(x, head, labels, rows)
    loss.backward()
    xr, wr = (t.detach().float().requires_grad_() for t in (x, head.weight))
    # logits, as they are kept, are rounded to bf16
    logits = xr[0] @ wr.t()
    logits = logits + (logits.detach().bfloat16().float() - logits.detach())
    want = torch.nn.functional.cross_entropy(logits, labels)
    want.backward()
    # fp32 sums over bf16 logits, some of which the order of a product's sums
    # rounds the other way; gradients through bf16 ones: 2^-9 a rounding
    assert abs(loss.item() - want.item()) <= 1e-4 * want.item()
    for t, r in ((x, xr), (head.weight, wr)):
        if not t.requires_grad:
            assert t.grad is None
            continue
        err = (t.grad.float() - r.grad).norm() / r.grad.norm()
        assert err < 2 ** -7


@pytest.mark.gpu
def test_same_as_chunk_by_chunk_gpu(monkeypatch):
    """Loss bit by bit, gradients but for their roundings; a hooked head and one of
    another class are called."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(2, 300, 256, device="cuda", generator=g).bfloat16()
    head = linear.Linear(256, 640, bias=False).to("cuda", torch.bfloat16)
    labels = torch.randint(0, 640, (600,), device="cuda", generator=g)
    out = []
    for own in (True, False):
        if not own:
            monkeypatch.setattr(cross_entropy, "head_loss_fits",
                                lambda *a: False)
        leaf = x.detach().clone().requires_grad_()
        head.weight.grad = None
        loss = chunked_cross_entropy(leaf, head, labels, 256)
        loss.backward()
        out.append((loss.detach(), leaf.grad, head.weight.grad))
    assert torch.equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        assert (a.float() - b.float()).norm() <= 2 ** -7 * b.float().norm()
    monkeypatch.undo()
    flat = x.view(600, 256).requires_grad_()
    seen = []
    hook = head.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    assert not cross_entropy.head_loss_fits(head, flat)
    chunked_cross_entropy(flat[None], head, labels, 256)
    assert seen == [(256, 640), (256, 640), (88, 640)]
    hook.remove()
    other = torch.nn.Linear(256, 640, bias=False).to("cuda", torch.bfloat16)
    assert not cross_entropy.head_loss_fits(other, flat)
    with torch.no_grad():
        assert not cross_entropy.head_loss_fits(head, flat)


@pytest.mark.gpu
def test_weights_of_other_forms_gpu():
    """A weight of another number of inputs is refused, by several chunks as by one
    and by the kernels themselves; one that is not contiguous is taken."""
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(1, 600, 256, device="cuda", generator=g).bfloat16()
    labels = torch.randint(0, 640, (600,), device="cuda", generator=g)
    head = linear.Linear(512, 640, bias=False).to("cuda", torch.bfloat16)
    for rows in (256, 600):
        with pytest.raises(RuntimeError):
            chunked_cross_entropy(x, head, labels, rows)
    for w in (head.weight, head.weight.view(-1)):
        for op in (cross_entropy.get_ext().tile_linear,
                   lambda x, w, b, m: cross_entropy.get_ext().rows_linear(
                       x[:8], w, [], b, 0, m)):
            with pytest.raises(RuntimeError, match="weight"):
                op(x[0], [w.detach()], [None], 0)
    head = linear.Linear(256, 640, bias=False).to("cuda", torch.bfloat16)
    out = []
    for w in (head.weight.detach(), head.weight.detach().t().contiguous().t()):
        head.weight = torch.nn.Parameter(w)
        leaf = x.clone().requires_grad_()
        loss = chunked_cross_entropy(leaf, head, labels, 256)
        loss.backward()
        out.append((loss.detach(), leaf.grad, head.weight.grad))
    assert not w.is_contiguous()
    # sums in another order round some bf16 logits and gradients the other way
    assert abs(out[0][0] - out[1][0]) <= 1e-4 * out[0][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert (a.float() - b.float()).norm() <= 2 ** -7 * a.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [128, 300])
@pytest.mark.parametrize("frozen", [None, "x", "w"])
def test_second_derivatives_gpu(rows, frozen):
    """Products of the Hessian and a vector, by several chunks and by one."""
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(1, 300, 256, device="cuda", generator=g).bfloat16()
    head = linear.Linear(256, 640, bias=False).to("cuda", torch.bfloat16)
    head.weight.data.normal_(0.0, 0.05, generator=g)
    labels = torch.randint(0, 640, (300,), device="cuda", generator=g)
    labels[::7] = -100
    x.requires_grad_(frozen != "x")
    head.weight.requires_grad_(frozen != "w")
    leaves = [t for t in (x, head.weight) if t.requires_grad]
    ways = [torch.randn(t.shape, device="cuda", generator=g).bfloat16()
            for t in leaves]

    def products(loss, leaves, ways):
        first = torch.autograd.grad(loss, leaves, create_graph=True)
        return torch.autograd.grad(
            sum((f.float() * v.float()).sum() for f, v in zip(first, ways)),
            leaves)
    first = torch.autograd.grad(chunked_cross_entropy(x, head, labels, rows),
                                leaves, create_graph=True)
    both = torch.autograd.grad(first, leaves, [torch.stack([v, -v]) for v in ways],
                               is_grads_batched=True)
    got = products(chunked_cross_entropy(x, head, labels, rows), leaves, ways)
    xr, wr = (t.detach().float().requires_grad_(t.requires_grad)
              for t in (x, head.weight))
    want = products(torch.nn.functional.cross_entropy(xr[0] @ wr.t(), labels),
                    [t for t in (xr, wr) if t.requires_grad], ways)
    # logits, two gradients of theirs, a product each: four roundings of 2^-9,
    # of which the chunks' sums take another
    for a, b, t in zip(got, want, both):
        for a in (a, t[0], -t[1]):
            assert (a.float() - b).norm() <= 2 ** -6 * b.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [128, 300])
def test_watched_backward_gpu(rows):
    """A mode about the backward alone sees the products."""
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(1, 300, 256, device="cuda", generator=g).bfloat16()
    x.requires_grad_()
    head = linear.Linear(256, 640, bias=False).to("cuda", torch.bfloat16)
    labels = torch.randint(0, 640, (300,), device="cuda", generator=g)
    loss = chunked_cross_entropy(x, head, labels, rows)
    leaves = [x, head.weight]
    want = torch.autograd.grad(loss, leaves, retain_graph=True)
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.overloadpacket)
            return func(*args, **(kwargs or {}))
    with Watch():
        got = torch.autograd.grad(loss, leaves)
    assert seen.count(torch.ops.aten.mm) == 2 * -(-300 // rows)
    # gradients rounded in other places and added up in bf16
    for a, w in zip(got, want):
        assert (a.float() - w.float()).norm() <= 2 ** -7 * w.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,v,rows", [(4096, 1024, 16000, 1024),
                                        (16384, 2048, 16064, 4096)])
@pytest.mark.parametrize("frozen", [None, "x", "w", "both"])
def test_memory_gpu(monkeypatch, frozen, n, h, v, rows):
    """No more of it than by calls of the head, at the most and between forward and
    backward; hooks on what is saved are given no more at a time."""
    x = torch.randn(1, n, h, device="cuda").bfloat16()
    head = linear.Linear(h, v, bias=False).to("cuda", torch.bfloat16)
    labels = torch.randint(0, v, (n,), device="cuda")
    x.requires_grad_(frozen not in ("x", "both"))
    head.weight.requires_grad_(frozen not in ("w", "both"))

    def step():
        # hidden states whose owner lets them go, as a norm's output
        y = x * 1
        return chunked_cross_entropy(y, head, labels, rows)

    def memory(offloaded):
        x.grad = head.weight.grad = None
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        if offloaded:
            with torch.autograd.graph.save_on_cpu():
                loss = step()
        else:
            loss = step()
        most = [torch.cuda.max_memory_allocated() - before]
        held = torch.cuda.memory_allocated() - before
        torch.cuda.reset_peak_memory_stats()
        if loss.requires_grad:
            loss.backward()
        most.append(torch.cuda.max_memory_allocated() - before)
        return (held, *most)
    got = []
    for fits in (cross_entropy.head_loss_fits, lambda *a: False):
        monkeypatch.setattr(cross_entropy, "head_loss_fits", fits)
        memory(False)       # the library's workspace
        got.append([memory(False), memory(True)])
    # gradients of x are made in their places, those of calls piece by piece
    for a, b in zip(sum(got[0], ()), sum(got[1], ())):
        assert a <= b + 2 * h * rows + (1 << 16), got


def _moments(stage, gas):
    """First moments of two steps of an engine over a model whose head's loss takes
    several chunks, and the calls of ``head_loss``."""
    import deepspeed_amd
    from deepspeed_amd.models import llama
    torch.manual_seed(0)
    cfg = llama.LlamaConfig(vocab_size=512, hidden_size=256,
                            intermediate_size=512, num_layers=2, num_heads=2,
                            num_kv_heads=1, max_seq_len=4096)
    model = llama.LlamaForCausalLM(cfg).cuda()
    engine, opt, _, _ = deepspeed_amd.initialize(model=model, config={
        "train_micro_batch_size_per_gpu": 3,
        "gradient_accumulation_steps": gas, "bf16": {"enabled": True},
        "zero_optimization": {"stage": stage},
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}}})
    g = torch.Generator().manual_seed(1)
    out, seen = [], []
    own = cross_entropy.head_loss

    def spy(head, x, labels, rows):
        seen.append(tuple(head.weight.shape))   # filled in by then
        return own(head, x, labels, rows)
    cross_entropy.head_loss = spy
    try:
        for _ in range(2 * gas):
            ids = torch.randint(0, 512, (3, 3000), generator=g).cuda()
            loss = engine(ids, labels=ids)
            engine.backward(loss)
            engine.step()
            out.append(loss.detach().view(1))
    finally:
        cross_entropy.head_loss = own
    for part in opt.layout_manifest():
        flat = opt.param_groups[part["group_idx"]]["params"][0]
        first = opt.state[flat]["exp_avg"]
        for _, at, n, _ in part["params"]:
            at += part["master_offset"]
            out.append(first[at:at + n].clone())
    engine.destroy()
    return out, seen


@pytest.mark.gpu
@pytest.mark.parametrize("stage,gas", [(2, 1), (2, 2), (3, 1), (3, 2)])
def test_engine_with_several_chunks_gpu(stage, gas, monkeypatch):
    """Losses and gradients as by calls of the head: its place in the flat buffer
    closed, and with the hooks of partitioned weights about it."""
    monkeypatch.setenv("MASTER_ADDR", "127.0.0.1")
    monkeypatch.setenv("MASTER_PORT", "29549")
    got, seen = _moments(stage, gas)
    assert seen == [(512, 256)] * 2 * gas
    monkeypatch.setattr(cross_entropy, "head_loss_fits", lambda *a: False)
    want, seen = _moments(stage, gas)
    assert not seen and len(got) == len(want)
    # the second step's weights and losses follow from gradients rounded otherwise
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        assert (a.float() - b.float()).norm() <= 2.0 ** -6 * b.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("frozen", [None, "x", "w"])
@pytest.mark.parametrize("n", [5600, 11000])
def test_memory_of_uneven_chunks_gpu(monkeypatch, frozen, n):
    """A last chunk that is shorter is the first to go."""
    test_memory_gpu(monkeypatch, frozen, n, 1000, 32064, 4096)
