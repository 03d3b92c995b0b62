"""The Llama-family path as users of this framework run it: training steps
through the engine, whole-prompt forwards through the inference engine, and
serving steps over the paged key/value cache.

``listed`` names the cases, ``draw`` gives more of the same ranges. Models are
the geometries of ``deepspeed_amd.models`` with fewer layers, so that a pass
stays short; one layer is what repeats in the full models. Weights are random
with the standard deviation of the models' own initialisation; the matrices of
queries and keys have half of it, which keeps the rounding of bf16 queries and
keys from being the largest error in a random model's softmax.
"""

import dataclasses
import math
import os

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

import deepspeed_amd
from deepspeed_amd.inference.ragged import PagedKVCache
from deepspeed_amd.models import llama

GEOMETRY = {
    "llama3-8b": llama.llama3_8b,
    "mistral-7b": llama.mistral_7b,
    "qwen2-7b": llama.qwen2_7b,
    "phi3-mini": llama.phi3_mini,
    "llama-mini": llama.llama_mini,
}
LR, BETAS, EPS, DECAY, CLIP = 1e-4, (0.9, 0.95), 1e-8, 0.1, 1.0
GROUP = 2048        # weights per scale of int8 serving (the engine's default)
DEVICE = "cuda"


def listed():
    return [
        # a development or fine-tuning step of a small model: launches count
        dict(name="train mini 2x512", kind="train", model="llama-mini",
             layers=2, batch=2, seq=512, zero=2),
        # the headline training workload, at a small and at its own micro batch
        dict(name="train 8b 2x4096", kind="train", model="llama3-8b",
             layers=2, batch=2, seq=4096, zero=3),
        dict(name="train 8b 8x4096", kind="train", model="llama3-8b",
             layers=2, batch=8, seq=4096, zero=3),
        # packed fine-tuning batches of odd length, heads of 96, no grouping
        dict(name="train phi3 4x1000", kind="train", model="phi3-mini",
             layers=2, batch=4, seq=1000, zero=2),
        # scoring a long prompt: the whole-prompt forward without a cache
        dict(name="prompt 8b 1x4096", kind="prompt", model="llama3-8b",
             layers=4, batch=1, seq=4096),
        # a batch of prompts padded to an odd length, biased projections and
        # seven query heads to a key head
        dict(name="prompt qwen2 3x777", kind="prompt", model="qwen2-7b",
             layers=4, batch=3, seq=777),
        # continuous batching: a portion of a long prompt behind kept history
        dict(name="portion 8b 1024+1500", kind="portion", model="llama3-8b",
             layers=4, slots=1, seq=1024, context=1500, weights="bf16"),
        # a single chat, one token at a time
        dict(name="decode 8b 1x500", kind="decode", model="llama3-8b",
             layers=4, slots=1, context=500, weights="bf16"),
        # a busy server, and one with long documents
        dict(name="decode 8b 32x2000", kind="decode", model="llama3-8b",
             layers=4, slots=32, context=2000, weights="bf16"),
        dict(name="decode 8b 8x16000", kind="decode", model="llama3-8b",
             layers=4, slots=8, context=16000, weights="bf16"),
        # decoding requests and a prompt portion packed into one step
        dict(name="packed 8b 24+200", kind="packed", model="llama3-8b",
             layers=4, slots=25, seq=200, context=1000, weights="bf16"),
        # weight-only int8 serving
        dict(name="decode int8 8b 8x1000", kind="decode", model="llama3-8b",
             layers=4, slots=8, context=1000, weights="int8"),
    ]


def _between(rng, lo, hi):
    """A whole number between ``lo`` and ``hi``, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "prompt", "prompt",
                       "portion", "decode", "decode", "decode", "packed"])
    served = rng.choice(["llama3-8b", "mistral-7b"])
    if kind == "train":
        model = rng.choice(list(GEOMETRY))
        seq = _between(rng, 128, 4096)
        return dict(kind=kind, model=model, layers=rng.randint(1, 2),
                    batch=rng.randint(1, max(1, min(8, 16384 // seq))),
                    seq=seq, zero=rng.choice([2, 3]))
    if kind == "prompt":
        seq = _between(rng, 64, 4096)
        return dict(kind=kind, model=rng.choice(list(GEOMETRY)), layers=4,
                    batch=rng.randint(1, max(1, min(8, 8192 // seq))), seq=seq)
    weights = rng.choice(["bf16", "bf16", "bf16", "int8"])
    if kind == "portion":
        return dict(kind=kind, model=served, layers=4, slots=1,
                    seq=_between(rng, 64, 1024), context=_between(rng, 64, 4000),
                    weights=weights)
    if kind == "packed":
        return dict(kind=kind, model=served, layers=4,
                    slots=rng.randint(3, 32), seq=_between(rng, 32, 256),
                    context=_between(rng, 64, 2000), weights=weights)
    slots = _between(rng, 1, 64)
    return dict(kind=kind, model=served, layers=4, slots=slots,
                context=_between(rng, 32, min(16000, 128000 // slots)),
                weights=weights)


# ------------------------------------------------------------------- inputs

def _config(case):
    cfg = GEOMETRY[case["model"]]()
    need = case.get("seq", 0) + 2 * case.get("context", 0) + 64
    return dataclasses.replace(cfg, num_layers=case["layers"],
                               max_seq_len=max(cfg.max_seq_len, need))


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _weights(cfg, g):
    """bf16 weights by the model's parameter names, in a fixed order."""
    def matrix(*shape, part=1.0):
        w = torch.empty(shape, dtype=torch.bfloat16, device=DEVICE)
        return w.normal_(0.0, part * cfg.initializer_range, generator=g)

    def gain(n):
        x = torch.randn(n, device=DEVICE, generator=g)
        return (1.0 + 0.1 * x).to(torch.bfloat16)

    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    w = {"model.embed_tokens.weight": matrix(cfg.vocab_size, h)}
    for n in range(cfg.num_layers):
        at = "model.layers.%d." % n
        w[at + "input_layernorm.weight"] = gain(h)
        for name, rows, part in (("q", cfg.num_heads, 0.5),
                                 ("k", cfg.num_kv_heads, 0.5),
                                 ("v", cfg.num_kv_heads, 1.0)):
            w[at + "self_attn.%s_proj.weight" % name] = \
                matrix(rows * d, h, part=part)
            if cfg.attention_bias:
                w[at + "self_attn.%s_proj.bias" % name] = \
                    matrix(rows * d, part=10.0)
        w[at + "self_attn.o_proj.weight"] = matrix(h, cfg.num_heads * d)
        w[at + "post_attention_layernorm.weight"] = gain(h)
        w[at + "mlp.gate_proj.weight"] = matrix(i, h)
        w[at + "mlp.up_proj.weight"] = matrix(i, h)
        w[at + "mlp.down_proj.weight"] = matrix(h, i)
    w["model.norm.weight"] = gain(h)
    w["lm_head.weight"] = matrix(cfg.vocab_size, h)
    return w


def _tokens(cfg, g, *shape):
    return torch.randint(0, cfg.vocab_size, shape, device=DEVICE, generator=g)


def _labels(case, ids):
    """Next tokens; the ends of all rows but the first are padding."""
    labels = ids[:, 1:].clone()
    for b in range(1, labels.shape[0]):
        labels[b, labels.shape[1] - 7 * b:] = -100
    return labels


def _lengths(case):
    """Kept tokens of each request: spread around the case's context."""
    n = case["slots"]
    if n == 1:
        return [case["context"]]
    return [max(1, int(case["context"] * (0.5 + (i * 7 % n) / (n - 1))))
            for i in range(n)]


def _history(cfg, lengths, g):
    """Kept keys and values: for each layer and request [kv heads, len, dim]."""
    std = cfg.initializer_range * math.sqrt(cfg.hidden_size)

    def rows(n, part):
        x = torch.randn(cfg.num_kv_heads, n, cfg.head_dim, device=DEVICE,
                        generator=g, dtype=torch.float32)
        return (part * std * x).to(torch.bfloat16)
    return [[(rows(n, 0.5), rows(n, 1.0)) for n in lengths]
            for _ in range(cfg.num_layers)]


def _model(cfg, weights):
    with torch.device(DEVICE):
        model = llama.LlamaForCausalLM(cfg)
    model = model.to(torch.bfloat16)
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
    return model


class _Training(dict):
    """A training run's state, which gives the engine back at its end."""

    def __del__(self):
        self["engine"].destroy()


def _prepare_train(case, seed):
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29543")
    cfg, g = _config(case), _generator(seed)
    model = _model(cfg, _weights(cfg, g))
    engine, _, _, _ = deepspeed_amd.initialize(model=model, config={
        "train_micro_batch_size_per_gpu": case["batch"],
        "gradient_accumulation_steps": 1,
        "bf16": {"enabled": True},
        "gradient_clipping": CLIP,
        "steps_per_print": 10 ** 9,
        "zero_optimization": {"stage": case["zero"], "overlap_comm": True},
        "optimizer": {"type": "AdamW",
                      "params": {"lr": LR, "betas": list(BETAS), "eps": EPS,
                                 "weight_decay": DECAY}},
    })
    ids = _tokens(cfg, g, case["batch"], case["seq"] + 1)
    return _Training(engine=engine, ids=ids[:, :-1].contiguous(),
                     labels=_labels(case, ids).contiguous())


def _prepare_served(case, seed):
    cfg, g = _config(case), _generator(seed)
    model = _model(cfg, _weights(cfg, g))
    engine = deepspeed_amd.init_inference(
        model, dtype=torch.int8 if case.get("weights") == "int8"
        else torch.bfloat16)
    if case["kind"] == "prompt":
        return {"engine": engine,
                "ids": _tokens(cfg, g, case["batch"], case["seq"])}
    lengths = _lengths(case)
    cache = PagedKVCache(
        cfg.num_layers, case["slots"], cfg.num_kv_heads, cfg.max_seq_len,
        cfg.head_dim, dtype=torch.bfloat16, device=DEVICE,
        num_blocks=sum(n // 64 + 1 for n in lengths)
        + case["slots"] + case.get("seq", 0) // 64)
    # requests grow side by side, so their blocks lie among each other's
    for at in range(0, max(lengths), 512):
        for s, n in enumerate(lengths):
            if at < n:
                cache.begin_step([s], min(512, n - at))
                cache.end_step()
    for layer, rows in enumerate(_history(cfg, lengths, g)):
        for s, both in enumerate(rows):
            blocks = torch.tensor(cache.block_table[s], device=DEVICE)
            for pool, x in zip((cache.k[layer], cache.v[layer]), both):
                pad = len(blocks) * cache.block_size - x.shape[1]
                x = F.pad(x, (0, 0, 0, pad)).view(
                    x.shape[0], len(blocks), cache.block_size, x.shape[2])
                pool[blocks] = x.transpose(0, 1)
    state = {"engine": engine, "cache": cache, "lens": cache.lens.clone(),
             "offsets": None, "q_len": 1, "slots": list(range(case["slots"]))}
    rows, seq = case["slots"], 1
    start = torch.tensor(lengths, dtype=torch.int32, device=DEVICE)
    if case["kind"] == "portion":
        rows, seq = 1, case["seq"]
        state["q_len"] = seq
        positions = start[:, None] + torch.arange(
            seq, dtype=torch.int32, device=DEVICE)[None]
    elif case["kind"] == "packed":
        # one token of every request but the last, a portion of the last
        more = case["seq"]
        last = case["slots"] - 1
        state["slots"] = list(range(last)) + [last] * more
        state["offsets"] = [0] * last + list(range(more))
        rows = last + more
        positions = start[state["slots"]] + torch.tensor(
            state["offsets"], dtype=torch.int32, device=DEVICE)
        positions = positions[:, None]
    else:
        positions = start[:, None]
    state["positions"] = positions.contiguous()
    state["ids"] = _tokens(cfg, g, rows, seq)
    return state


def prepare(case, seed):
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    return _prepare_served(case, seed)


# ---------------------------------------------------------------------- run

def _views(engine):
    """The fp32 weights and first moments by parameter name, as views of the
    optimizer's flat state."""
    opt = engine.optimizer
    master, moment = {}, {}
    for part in opt.layout_manifest():
        flat = opt.param_groups[part["group_idx"]]["params"][0]
        first = opt.state[flat]["exp_avg"]
        for name, off, n, shape in part["params"]:
            lo = part["master_offset"] + off
            master[name] = flat.data[lo:lo + n].view(shape)
            moment[name] = first[lo:lo + n].view(shape)
    return {"master": master, "exp_avg": moment}


def run(state):
    engine, ids = state["engine"], state["ids"]
    if "labels" in state:
        loss = engine(ids, labels=state["labels"])
        engine.backward(loss)
        engine.step()
        if "views" not in state:      # the optimizer's state is there now
            state["views"] = _views(engine)
        return {"loss": loss.detach(), **state["views"]}
    cache = state.get("cache")
    if cache is None:
        return {"logits": engine(ids)}
    # every pass takes the same step: a rejected draft is rolled back like this
    cache.lens.copy_(state["lens"])
    if state["offsets"] is None:
        cache.begin_step(state["slots"], state["q_len"])
    else:
        cache.begin_step(state["slots"], state["q_len"],
                         offsets=state["offsets"])
    logits = engine(ids, positions=state["positions"], kv_cache=cache)
    cache.end_step()
    return {"logits": logits, "keys": cache.k[-1], "values": cache.v[-1]}


# --------------------------------------------------------------------- work

def _sizes(cfg):
    """Numbers in the matrices of all layers, in the head and elsewhere."""
    h, d = cfg.hidden_size, cfg.head_dim
    layer = h * d * (2 * cfg.num_heads + 2 * cfg.num_kv_heads) \
        + 3 * h * cfg.intermediate_size
    return cfg.num_layers * layer, h * cfg.vocab_size, h


def work(case):
    cfg = _config(case)
    layers, head, h = _sizes(cfg)
    kept = 2 * cfg.num_kv_heads * cfg.head_dim * cfg.num_layers  # per token
    score = 4.0 * cfg.num_heads * cfg.head_dim * cfg.num_layers  # per pair
    if case["kind"] in ("train", "prompt"):
        B, S = case["batch"], case["seq"]
        T, pairs = B * S, B * S * (S + 1) / 2
        if case["kind"] == "train":
            # per weight: read for the products, fp32 master and both moments
            # read and written, the bf16 weight written
            return {"bytes": (layers + 2 * head) * 28.0 + T * 16.0,
                    "flops": 6.0 * (layers + head) * T + 3.0 * score * pairs}
        return {"bytes": (layers + head + T * h) * 2.0
                + T * (8.0 + 2.0 * cfg.vocab_size),
                "flops": 2.0 * (layers + head) * T + score * pairs}
    lengths = _lengths(case)
    if case["kind"] == "portion":
        new = [case["seq"]]
    elif case["kind"] == "packed":
        new = [1] * (case["slots"] - 1) + [case["seq"]]
    else:
        new = [1] * case["slots"]
    T = sum(new)
    pairs = sum(m * n + m * (m + 1) / 2 for n, m in zip(lengths, new))
    per = 1.0 + 4.0 / GROUP if case["weights"] == "int8" else 2.0
    return {"bytes": (layers + head) * per + T * h * 2.0
            + (sum(lengths) + T) * kept * 2.0
            + T * (12.0 + 2.0 * cfg.vocab_size),
            "flops": 2.0 * (layers + head) * T + score * pairs}


def tolerance(case):
    # bf16 activations and gradients through the layers. Two attention kernels
    # in turn (another order of the sums, another place of the rounding) give
    # gradients and logits that differ by up to 0.014, and by up to 0.17 of
    # the root mean square at the worst of the values; both are 0.014 off
    # exact(). The second pass starts from weights whose first Adam update
    # turned on the sign of gradients next to nothing.
    return {"rel": 0.03, "max": 0.7}


# -------------------------------------------------------------------- exact

def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _turn(cfg, x, positions):
    """Rotary embedding of x [T, heads, dim] at ``positions`` [T]."""
    half = cfg.head_dim // 2
    inv = cfg.rope_theta ** (-torch.arange(0, half, dtype=torch.float64,
                                           device=x.device) / half)
    a = positions.double()[:, None] * inv
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _one_head(q, k, v, first):
    """Causal attention of q [T, dim] at positions ``first``.. over all k."""
    score = q @ k.t() / math.sqrt(q.shape[-1])
    at = first + torch.arange(q.shape[0], device=q.device)
    hidden = torch.arange(k.shape[0], device=q.device)[None] > at[:, None]
    return torch.softmax(score.masked_fill(hidden, -math.inf), -1) @ v


def _attend(q, k, v, first):
    """q [T, heads, dim] over k, v [kept + T, kv heads, dim]."""
    group = q.shape[1] // k.shape[1]
    return torch.stack(
        [checkpoint(_one_head, q[:, j], k[:, j // group], v[:, j // group],
                    first, use_reentrant=False) if q.requires_grad else
         _one_head(q[:, j], k[:, j // group], v[:, j // group], first)
         for j in range(q.shape[1])], 1)


def _hidden(cfg, w, ids, starts, history=None):
    """Last hidden rows [T, h] of the sequences ``ids`` (a list of 1-d
    tensors) that follow ``starts`` kept tokens each."""
    x = w["model.embed_tokens.weight"][torch.cat(ids)]
    cuts = [len(i) for i in ids]
    where = torch.cat([s + torch.arange(n, device=x.device)
                       for s, n in zip(starts, cuts)])

    def layer(x, n):
        at = "model.layers.%d." % n
        y = _norm(x, w[at + "input_layernorm.weight"], cfg.rms_eps)

        def proj(name, heads):
            return F.linear(y, w[at + "self_attn.%s_proj.weight" % name],
                            w.get(at + "self_attn.%s_proj.bias" % name)).view(
                                -1, heads, cfg.head_dim)
        q = _turn(cfg, proj("q", cfg.num_heads), where).split(cuts)
        k = _turn(cfg, proj("k", cfg.num_kv_heads), where).split(cuts)
        v = proj("v", cfg.num_kv_heads).split(cuts)
        o = []
        for j, s in enumerate(starts):
            kk, vv = k[j], v[j]
            if history is not None:
                old = [t.double().transpose(0, 1) for t in history[n][j]]
                kk, vv = torch.cat([old[0], kk]), torch.cat([old[1], vv])
            o.append(_attend(q[j], kk, vv, s))
        x = x + F.linear(torch.cat(o).flatten(1),
                         w[at + "self_attn.o_proj.weight"])
        y = _norm(x, w[at + "post_attention_layernorm.weight"], cfg.rms_eps)
        return x + F.linear(F.silu(F.linear(y, w[at + "mlp.gate_proj.weight"]))
                            * F.linear(y, w[at + "mlp.up_proj.weight"]),
                            w[at + "mlp.down_proj.weight"])

    for n in range(cfg.num_layers):
        x = layer(x, n)
    return _norm(x, w["model.norm.weight"], cfg.rms_eps)


def _int8(w):
    """The values that groupwise symmetric int8 weights stand for."""
    rows = F.pad(w.float().flatten(), (0, -w.numel() % GROUP)).view(-1, GROUP)
    top = rows.abs().amax(1, keepdim=True)
    scale = torch.where(top > 0, top / 127.0, torch.ones_like(top))
    q = torch.round(rows / scale).clamp(-127, 127).double() * scale.double()
    return q.flatten()[:w.numel()].view(w.shape)


def _exact_train(case, cfg, w, g):
    ids = _tokens(cfg, g, case["batch"], case["seq"] + 1)
    labels = _labels(case, ids)
    w = {k: v.double().requires_grad_() for k, v in w.items()}
    x = _hidden(cfg, w, list(ids[:, :-1]), [0] * case["batch"])
    flat = labels.reshape(-1)

    def part(rows, lab):
        return F.cross_entropy(F.linear(rows, w["lm_head.weight"]), lab,
                               reduction="sum")
    total = sum(checkpoint(part, x[i:i + 2048], flat[i:i + 2048],
                           use_reentrant=False)
                for i in range(0, len(flat), 2048))
    loss = total / (flat != -100).sum()
    names = list(w)
    grads = torch.autograd.grad(loss, [w[n] for n in names])
    with torch.no_grad():
        norm = torch.sqrt(sum(t.square().sum() for t in grads))
        cut = (norm / CLIP).clamp(min=1.0)
        master, first = {}, {}
        for n, t in zip(names, grads):
            t = t / cut
            first[n] = (1.0 - BETAS[0]) * t
            master[n] = w[n].detach() * (1.0 - LR * DECAY) \
                - LR * t / (t.abs() + EPS)
    return {"loss": loss.detach(), "master": master, "exp_avg": first}


def exact(case, seed):
    if work(case)["flops"] > 4e14:
        return None
    cfg, g = _config(case), _generator(seed)
    w = _weights(cfg, g)
    if case["kind"] == "train":
        return _exact_train(case, cfg, w, g)
    with torch.no_grad():
        if case.get("weights") == "int8":
            w = {k: _int8(v) if "proj" in k or "lm_head" in k else v
                 for k, v in w.items()}
        w = {k: v.double() for k, v in w.items()}
        if case["kind"] == "prompt":
            ids = _tokens(cfg, g, case["batch"], case["seq"])
            x = _hidden(cfg, w, list(ids), [0] * case["batch"])
            return {"logits": F.linear(x, w["lm_head.weight"]).view(
                case["batch"], case["seq"], -1)}
        lengths = _lengths(case)
        history = _history(cfg, lengths, g)
        if case["kind"] == "portion":
            ids = list(_tokens(cfg, g, 1, case["seq"]))
        elif case["kind"] == "packed":
            flat = _tokens(cfg, g, case["slots"] - 1 + case["seq"], 1)[:, 0]
            ids = list(flat.split([1] * (case["slots"] - 1) + [case["seq"]]))
        else:
            ids = list(_tokens(cfg, g, case["slots"], 1))
        x = _hidden(cfg, w, ids, lengths, history)
        logits = F.linear(x, w["lm_head.weight"])
        shape = (1, -1) if case["kind"] == "portion" else (-1, 1)
        return {"logits": logits.view(*shape, cfg.vocab_size),
                "keys": None, "values": None}
