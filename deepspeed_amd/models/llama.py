"""Llama-family decoder (Llama-3 shapes) built on the CDNA4 fused ops.

This is the framework's flagship training model for the headline benchmark
(Llama-3-8B ZeRO-3 bf16 on MI355X). Random-init weights,
synthetic data; architecture matches Llama-3 (GQA attention, RoPE
theta=500000, SwiGLU MLP, RMSNorm, tied-off lm_head).

Hot ops: RMSNorm / RoPE / SwiGLU are the hand-written HIP kernels in
``deepspeed_amd.ops``, and so is attention (flash forward and backward, paged
serving) wherever its kernels apply, else torch SDPA; linear layers are
``ops.linear``'s, with the library's products where these are faster.
"""

from dataclasses import dataclass

import torch
import torch.nn as nn
import torch.nn.functional as F

from ..ops import linear as _linear
from ..ops._loader import get_ext
from ..ops.attention import rope_flash_attention
from ..ops.embedding import Embedding
from ..ops.linear import (SWIGLU, Linear, all_unhooked, call, movable,
                          rows_linear, tile_linear, unhooked)
from ..ops.norms import RMSNorm
from ..ops.rope import apply_rope, rope_tables
from ..ops.swiglu import swiglu


@dataclass
class LlamaConfig:
    vocab_size: int = 128256
    hidden_size: int = 4096
    intermediate_size: int = 14336
    num_layers: int = 32
    num_heads: int = 32
    num_kv_heads: int = 8
    max_seq_len: int = 8192
    rope_theta: float = 500000.0
    rms_eps: float = 1e-5
    tie_embeddings: bool = False
    initializer_range: float = 0.02
    attention_bias: bool = False  # qwen2-style qkv bias
    # llama3-style rope_scaling dict: {factor, low_freq_factor,
    # high_freq_factor, original_max_position_embeddings}
    rope_scaling: dict = None

    @property
    def head_dim(self):
        return self.hidden_size // self.num_heads


def llama3_8b():
    return LlamaConfig()


def llama3_1_8b():
    """Llama-3.1-8B: llama3 rope scaling unlocks 128k context on the
    3-8B geometry (frequencies verified bit-exact vs HF transformers'
    _compute_llama3_parameters)."""
    return LlamaConfig(max_seq_len=131072, rope_scaling={
        "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
        "original_max_position_embeddings": 8192})


def llama3_70b():
    return LlamaConfig(hidden_size=8192, intermediate_size=28672,
                       num_layers=80, num_heads=64, num_kv_heads=8)


def llama_tiny():
    """Small config for CPU tests."""
    return LlamaConfig(vocab_size=512, hidden_size=64, intermediate_size=128,
                       num_layers=2, num_heads=4, num_kv_heads=2,
                       max_seq_len=128)


def phi3_mini():
    """Phi-3-mini 3.8B shapes (small-model ZeRO-2 path).
    Phi-3's decoder is Llama-architecture (RoPE, SwiGLU, RMSNorm) with MHA
    (no GQA) and a 32k vocab."""
    return LlamaConfig(vocab_size=32064, hidden_size=3072,
                       intermediate_size=8192, num_layers=32, num_heads=32,
                       num_kv_heads=32, max_seq_len=4096, rope_theta=10000.0,
                       tie_embeddings=False)


def mistral_7b():
    """Mistral-7B shapes (llama architecture; the 4k-window sliding
    attention is omitted — full causal attention is a superset and the
    paged KV cache caps context by max_seq_len)."""
    return LlamaConfig(vocab_size=32000, hidden_size=4096,
                       intermediate_size=14336, num_layers=32, num_heads=32,
                       num_kv_heads=8, max_seq_len=8192, rope_theta=10000.0)


def qwen2_7b():
    """Qwen2-7B shapes: Llama architecture + qkv bias, 152k vocab
    (reference inference/v2/model_implementations/qwen_v2)."""
    return LlamaConfig(vocab_size=152064, hidden_size=3584,
                       intermediate_size=18944, num_layers=28, num_heads=28,
                       num_kv_heads=4, max_seq_len=32768,
                       rope_theta=1000000.0, attention_bias=True)


def qwen2_mini():
    return LlamaConfig(vocab_size=512, hidden_size=64, intermediate_size=128,
                       num_layers=2, num_heads=4, num_kv_heads=2,
                       max_seq_len=128, attention_bias=True)


def llama_mini():
    """~0.5B for single-GPU smoke runs."""
    return LlamaConfig(vocab_size=32000, hidden_size=1024,
                       intermediate_size=2816, num_layers=8, num_heads=16,
                       num_kv_heads=4, max_seq_len=4096)


@movable
class LlamaAttention(nn.Module):
    def __init__(self, cfg: LlamaConfig):
        super().__init__()
        self.cfg = cfg
        self.num_heads = cfg.num_heads
        self.num_kv_heads = cfg.num_kv_heads
        self.head_dim = cfg.head_dim
        h = cfg.hidden_size
        ab = cfg.attention_bias
        self.q_proj = Linear(h, cfg.num_heads * self.head_dim, bias=ab)
        self.k_proj = Linear(h, cfg.num_kv_heads * self.head_dim, bias=ab)
        self.v_proj = Linear(h, cfg.num_kv_heads * self.head_dim, bias=ab)
        self.o_proj = Linear(cfg.num_heads * self.head_dim, h, bias=False)

    def _out(self, o):
        y = rows_linear(o, (self.o_proj,)) or tile_linear(o, (self.o_proj,))
        return call(self.o_proj, o) if y is None else y[0]

    def forward(self, x, cos, sin, positions=None, kv_cache=None,
                attention_fn=None):
        B, S, _ = x.shape
        mods = self.q_proj, self.k_proj, self.v_proj
        qkv = rows_linear(x, mods) or tile_linear(x, mods)
        if qkv is None:
            qkv = [call(m, x) for m in mods]
        q = qkv[0].view(B, S, self.num_heads, self.head_dim)
        k = qkv[1].view(B, S, self.num_kv_heads, self.head_dim)
        v = qkv[2].view(B, S, self.num_kv_heads, self.head_dim)
        if attention_fn is None and hasattr(kv_cache, "rope_attention"):
            # paged pool: rotation, cache write and attention over the block
            # lists in three launches; None -> ineligible, paths below
            o = kv_cache.rope_attention(self.layer_idx, q, k, v, cos, sin,
                                        positions)
            if o is not None:
                kv_cache.last_decoded = S == 1
                return self._out(o.reshape(B, S, -1))
        sp = getattr(self, "sp_group", None)
        if kv_cache is None and attention_fn is None and sp is None:
            # hand-written CDNA4 kernels, [B, S, H, D] throughout
            o = rope_flash_attention(q, k, v, cos, sin, positions)
            if o is not None:
                return self._out(o.reshape(B, S, -1))
        q = apply_rope(q, cos, sin, positions)
        k = apply_rope(k, cos, sin, positions)

        if sp is not None and kv_cache is None:
            # Ulysses: all-to-all scatters heads / gathers the sequence so
            # each rank runs full-sequence causal attention on H/P heads
            o = self._ulysses_attn(q, k, v)
            return self._out(o.reshape(B, S, -1))

        if (S == 1 and kv_cache is not None
                and hasattr(kv_cache, "decode_attention")
                and attention_fn is None):
            # paged flash-decode kernel over the block table (no padded
            # KV materialization); None -> ineligible, normal path below
            o = kv_cache.decode_attention(self.layer_idx, q, k, v)
            if o is not None:
                kv_cache.last_decoded = True
                return self._out(o.reshape(B, S, -1))

        # [B, H, S, D] for SDPA
        q = q.transpose(1, 2)
        k = k.transpose(1, 2)
        v = v.transpose(1, 2)
        attn_mask = None
        if kv_cache is not None:
            k, v = kv_cache.update(self.layer_idx, k, v)
            # ragged caches expose a per-sequence validity mask (slots in
            # one batch sit at different positions)
            attn_mask = getattr(kv_cache, "last_mask", None)
        if attention_fn is not None:
            o = attention_fn(q, k, v)
        else:
            # prefill (q spans the whole kv prefix) is causal; decode steps
            # (q_len < kv_len) attend to the full cached prefix
            o = sdpa_gqa(q, k, v,
                         causal=attn_mask is None and q.size(2) == k.size(2),
                         attn_mask=attn_mask)
        return self._out(o.transpose(1, 2).reshape(B, S, -1))


def _bshd_causal_attention(q, k, v):
    """Local attention in [b, s, H, d] layout (Ulysses local_attn)."""
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    return sdpa_gqa(q, k, v, causal=True).transpose(1, 2)


def enable_ulysses(model, sp_group=None):
    """Wire Ulysses sequence parallelism into every attention module.
    Requires num_heads % sp_world == 0 and num_kv_heads % sp_world == 0."""
    from ..parallel import groups
    from ..sequence import DistributedAttention
    sp_group = sp_group or groups.get_sequence_parallel_group()
    assert sp_group is not None, "initialize_sequence_parallel first"
    import torch.distributed as td
    P = td.get_world_size(sp_group)
    for mod in model.modules():
        if isinstance(mod, LlamaAttention):
            assert mod.num_heads % P == 0 and mod.num_kv_heads % P == 0, \
                f"heads {mod.num_heads}/{mod.num_kv_heads} not divisible " \
                f"by sp={P}"
            mod.sp_group = sp_group
            mod._ulysses_attn = DistributedAttention(_bshd_causal_attention,
                                                     sp_group)
    return model


def sdpa_gqa(q, k, v, causal=True, attn_mask=None):
    """SDPA with grouped-query support (expands KV if enable_gqa missing)."""
    try:
        return F.scaled_dot_product_attention(q, k, v, attn_mask=attn_mask,
                                              is_causal=causal,
                                              enable_gqa=True)
    except (TypeError, RuntimeError):
        rep = q.shape[1] // k.shape[1]
        if rep > 1:
            k = k.repeat_interleave(rep, dim=1)
            v = v.repeat_interleave(rep, dim=1)
        return F.scaled_dot_product_attention(q, k, v, attn_mask=attn_mask,
                                              is_causal=causal)


@movable
class LlamaMLP(nn.Module):
    def __init__(self, cfg: LlamaConfig):
        super().__init__()
        h, i = cfg.hidden_size, cfg.intermediate_size
        self.gate_proj = Linear(h, i, bias=False)
        self.up_proj = Linear(h, i, bias=False)
        self.down_proj = Linear(i, h, bias=False)

    def forward(self, x):
        mods = self.gate_proj, self.up_proj
        h = rows_linear(x, mods, SWIGLU) or tile_linear(x, mods, SWIGLU)
        if h is None:
            h = [swiglu(*(tile_linear(x, mods) or [call(m, x) for m in mods]))]
        mods = self.down_proj,
        y = rows_linear(h[0], mods) or tile_linear(h[0], mods)
        return call(self.down_proj, h[0]) if y is None else y[0]


def add_norm(norm, x, delta):
    """(norm of the residual stream x with a sublayer's output added, the new
    stream); one kernel where nothing watches or replaces the norm's call."""
    if delta is None:
        return norm(x), x
    if type(norm) is RMSNorm and unhooked(norm, internal_ok=True):
        return norm(delta, residual=x)
    x = x + delta
    return norm(x), x


@movable
class LlamaDecoderLayer(nn.Module):
    def __init__(self, cfg: LlamaConfig, layer_idx: int):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, eps=cfg.rms_eps)
        self.self_attn = LlamaAttention(cfg)
        self.self_attn.layer_idx = layer_idx
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, eps=cfg.rms_eps)
        self.mlp = LlamaMLP(cfg)

    def chain(self, x, delta, cos, sin, positions=None, kv_cache=None):
        """The layer on a residual stream x that still lacks the last
        sublayer's output ``delta`` (or None); returns it the same way, so that
        every add happens inside the norm behind it."""
        h, x = add_norm(self.input_layernorm, x, delta)
        h, x = add_norm(self.post_attention_layernorm, x,
                        self.self_attn(h, cos, sin, positions, kv_cache))
        return x, self.mlp(h)

    def forward(self, x, cos, sin, positions=None, kv_cache=None):
        x, delta = self.chain(x, None, cos, sin, positions, kv_cache)
        return x + delta


# What a native layer stands for: replaced, they are called.
_CHAIN, _OUT = LlamaDecoderLayer.chain, LlamaAttention._out


_ATTN = "q_proj", "k_proj", "v_proj", "o_proj"
_MLP = "gate_proj", "up_proj", "down_proj"


def _operands(layer, rows: int):
    """What a decoder layer brings to ``paged_decoder_layer``, or None where its
    modules are to be called: (norm weights, their eps, linear weights, scales,
    biases, group)."""
    attn, mlp = layer.self_attn, layer.mlp
    if type(attn) is not LlamaAttention or type(mlp) is not LlamaMLP or \
            not unhooked(attn) or not unhooked(mlp) or \
            "chain" in layer.__dict__ or "_out" in attn.__dict__ or \
            attn.head_dim != 128:
        return None
    H, parts = attn.num_heads * 128, layer._modules
    norms = parts.get("input_layernorm"), parts.get("post_attention_layernorm")
    mods = [attn._modules.get(name) for name in _ATTN]
    mods += [mlp._modules.get(name) for name in _MLP]
    kind = type(mods[0])
    if type(norms[0]) is not RMSNorm or type(norms[1]) is not RMSNorm or \
            any(type(m) is not kind for m in mods):
        return None
    scales, group = [], 0
    if kind is Linear or kind is nn.Linear:
        weights = [m._parameters.get("weight") for m in mods]
        if any(type(w) is not nn.Parameter for w in weights):
            return None
    elif hasattr(kind, "int8_rows") and rows <= _linear.ROWS_INT8:
        weights = []
        for m in mods:
            p = m.int8_rows(H if len(weights) < 6 else
                            weights[5].numel() // H)
            if p is None or p[2] % 256 or group not in (0, p[2]):
                return None
            group = p[2]
            weights.append(p[0])
            scales.append(p[1])
    else:
        return None
    if not all_unhooked((attn, mlp, *norms, *mods)):
        return None
    biases = [m._parameters["bias"] if "bias" in m._parameters else m.bias
              for m in mods]
    scaled = [n._parameters.get("weight") for n in norms]
    if any(w is None for w in scaled) or not get_ext().paged_layer_fits(
            scaled, weights, scales, biases, H, attn.num_kv_heads * 128):
        return None
    return (scaled, norms[0].eps, norms[1].eps, weights, scales, biases, group)


def _plain(x) -> bool:
    """A stream, or an output to be added to it, that native layers take."""
    return type(x) is torch.Tensor and x.is_cuda and \
        x.dtype is torch.bfloat16 and x.is_contiguous() and \
        x.data_ptr() % 16 == 0


class LlamaModel(nn.Module):
    def __init__(self, cfg: LlamaConfig):
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(
            [LlamaDecoderLayer(cfg, i) for i in range(cfg.num_layers)])
        self.norm = RMSNorm(cfg.hidden_size, eps=cfg.rms_eps)
        self.gradient_checkpointing = False

    def forward(self, input_ids, positions=None, kv_cache=None):
        x = self.embed_tokens(input_ids)
        cos, sin = rope_tables(self.cfg.head_dim, self.cfg.max_seq_len,
                               self.cfg.rope_theta, device=x.device,
                               rope_scaling=self.cfg.rope_scaling)
        recompute = (self.gradient_checkpointing and self.training
                     and torch.is_grad_enabled())
        if recompute:
            from ..runtime.activation_checkpointing import checkpoint
        delta = None
        plan = self._paged_plan(x, positions, kv_cache)
        layers = list(self.layers)

        def operands(i):
            if plan is None or i == len(layers) or \
                    type(layers[i]) is not LlamaDecoderLayer or \
                    not unhooked(layers[i]):
                return None
            return _operands(layers[i], x.shape[0] * x.shape[1])

        after, native = operands(0), True
        for i, layer in enumerate(layers):
            # behind modules, which may hand on or change anything, all is
            # looked at anew
            behind = native
            ops = after if behind else operands(i)
            if not behind and ops and not (
                    (delta is None or _plain(delta) and delta.shape == x.shape)
                    and self._paged_plan(x, positions, kv_cache) is plan):
                ops = None
            native = ops is not None
            after = operands(i + 1) if native else None
            if recompute:
                x = checkpoint(lambda x_, l=layer: l(x_, cos, sin, positions,
                                                     kv_cache), x)
            elif native:
                at = layer.self_attn.layer_idx
                x, delta = get_ext().paged_decoder_layer(
                    x, delta, *ops, cos, sin, positions, x.shape[1],
                    kv_cache.k[at], kv_cache.v[at], plan.dst, plan.meta,
                    plan.items, plan.runs, plan.merges, plan.any_merge,
                    plan.nq, 128 ** -0.5, behind, after is not None)
                kv_cache.last_decoded = x.shape[1] == 1
            elif type(layer) is LlamaDecoderLayer and unhooked(layer):
                x, delta = layer.chain(x, delta, cos, sin, positions,
                                       kv_cache)
            else:
                x = x if delta is None else x + delta
                x, delta = layer(x, cos, sin, positions, kv_cache), None
        return add_norm(self.norm, x, delta)[0]

    def _paged_plan(self, x, positions, kv_cache):
        """The plan of a serving step whose layers may run as native calls of
        nine launches each, or None. A step of few tokens is bound by the host
        otherwise (one request, four layers: 740 us of host time for 640 us of
        kernels)."""
        cfg = self.cfg
        if not hasattr(kv_cache, "layers_plan") or torch.is_grad_enabled() or \
                not _plain(x) or not x.numel() or \
                x.shape[-1] != cfg.num_heads * 128 or x.shape[-1] > 16384 or \
                get_ext() is None or torch.is_autocast_enabled() or \
                torch.compiler.is_compiling() or \
                LlamaDecoderLayer.chain is not _CHAIN or \
                LlamaAttention._out is not _OUT or \
                rows_linear is not _linear.rows_linear or \
                tile_linear is not _linear.tile_linear:
            return None
        return kv_cache.layers_plan(x, cfg.num_heads, cfg.num_kv_heads,
                                    positions)

    def gradient_checkpointing_enable(self):
        self.gradient_checkpointing = True


class LlamaForCausalLM(nn.Module):
    def __init__(self, cfg: LlamaConfig):
        super().__init__()
        self.cfg = cfg
        self.model = LlamaModel(cfg)
        self.lm_head = Linear(cfg.hidden_size, cfg.vocab_size, bias=False)
        if cfg.tie_embeddings:
            self.lm_head.weight = self.model.embed_tokens.weight
        self.apply(self._init_weights)

    def _init_weights(self, module):
        std = self.cfg.initializer_range
        if isinstance(module, nn.Linear):
            module.weight.data.normal_(0.0, std)
            if module.bias is not None:
                module.bias.data.zero_()
        elif isinstance(module, nn.Embedding):
            module.weight.data.normal_(0.0, std)

    def forward(self, input_ids, labels=None, positions=None, kv_cache=None):
        hidden = self.model(input_ids, positions, kv_cache)
        if labels is not None:
            # chunked fp32 cross-entropy: avoids materializing the full
            # [B*S, vocab] fp32 logits (vocab=128256 -> ~2 GB per 4k tokens).
            # Routed through the lm_head MODULE so ZeRO-3 fetch hooks fire.
            return chunked_cross_entropy(hidden, self.lm_head, labels)
        mods = self.lm_head,
        logits = rows_linear(hidden, mods) or tile_linear(hidden, mods)
        return call(self.lm_head, hidden) if logits is None else logits[0]

    def num_parameters(self):
        return sum(p.numel() for p in self.parameters())


def chunked_cross_entropy(hidden, lm_head, labels, chunk_tokens=8192):
    """loss = CE(lm_head(hidden), labels), computed in token chunks so the
    fp32 logits never exceed chunk_tokens x vocab. With DS_AMD_FUSED_CE=1
    the per-chunk softmax+nll runs as the fused bf16 HIP kernel and no
    fp32 logits are materialized at all."""
    from ..ops.cross_entropy import (fused_cross_entropy_mean,
                                     fused_cross_entropy_sum, head_loss_fits)
    B, S, H = hidden.shape
    hidden = hidden.reshape(-1, H)
    labels = labels.reshape(-1)
    n = hidden.shape[0]
    if 0 < n <= chunk_tokens:
        if labels.shape[0] > n:
            labels = labels[:n]
        return fused_cross_entropy_mean(call(lm_head, hidden), labels)
    if n and labels.shape[0] >= n and labels.dtype is torch.long and \
            head_loss_fits(lm_head, hidden):
        total, count = lm_head(hidden, loss=(labels[:n].contiguous(),
                                             chunk_tokens))
        return total / count.clamp(min=1)
    total = hidden.new_zeros((), dtype=torch.float32)
    count = hidden.new_zeros((), dtype=torch.float32)
    for s in range(0, n, chunk_tokens):
        e = min(s + chunk_tokens, n)
        logits = call(lm_head, hidden[s:e])
        l, c = fused_cross_entropy_sum(logits, labels[s:e])
        total = total + l
        count = count + c
    return total / count.clamp(min=1)
