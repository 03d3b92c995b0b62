"""Flash attention on the matrix cores (csrc/attention.hip), forward and
backward: heads of 64, 96 and 128, any sequence length, grouped key heads, bf16.
Elsewhere callers take torch's scaled_dot_product_attention."""

import math
import os
from typing import Optional

import torch

from ._loader import get_ext
from .linear import _plain_autograd, untransformed


def _eligible(q: torch.Tensor, k: torch.Tensor) -> bool:
    return (get_ext() is not None and q.is_cuda
            and q.dtype is torch.bfloat16 and k.dtype is torch.bfloat16
            and q.dim() == 4 and k.dim() == 4
            and q.size(-1) == k.size(-1) and q.size(-1) in (64, 96, 128)
            and q.size(1) == k.size(1) and q.size(2) % k.size(2) == 0
            and q.numel() > 0)


def flash_attn_available(q: torch.Tensor, k: torch.Tensor) -> bool:
    """Inference/prefill forward; DS_AMD_FLASH=0 opts out."""
    if os.environ.get("DS_AMD_FLASH", "1") == "0":
        return False
    return _eligible(q, k) and not torch.is_grad_enabled()


def flash_train_available(q: torch.Tensor, k: torch.Tensor) -> bool:
    """Training forward and backward (FlashAttnFunc); DS_AMD_FLASH_TRAIN=0
    opts out."""
    if os.environ.get("DS_AMD_FLASH_TRAIN", "1") == "0":
        return False
    return _eligible(q, k) and _plain_autograd()


def _rows(x: torch.Tensor) -> torch.Tensor:
    """x as the kernels read it: unit stride inside a head, 16-byte rows."""
    if x.stride(3) == 1 and x.data_ptr() % 16 == 0 and all(
            x.stride(d) % 8 == 0 and x.stride(d) >= 0 for d in range(3)) and \
            x.stride(1) < 1 << 24:
        return x
    return x.clone(memory_format=torch.contiguous_format)


def _scaled(q, scale):
    """(q, scale, factor of dq) with a positive scale: the kernels take maxima
    of unscaled scores. A scale of nought or no number goes into q."""
    scale = scale if scale is not None else 1.0 / math.sqrt(q.size(-1))
    if scale > 0:
        return q, scale, 1
    return (-q, -scale, -1) if scale < 0 else (q * scale, 1.0, scale)


def _vt_from_bshd(v):
    """[B, S, Hkv, D] -> [B, Hkv, D, S] via the tiled transpose kernel."""
    ext = get_ext()
    B, S, Hk, D = v.shape
    if ext is None or not v.is_cuda or v.dtype != torch.bfloat16:
        return v.permute(0, 2, 3, 1).contiguous()
    out = ext.transpose_bf16(v.contiguous(), B * Hk, S, D, Hk * D, Hk, D,
                             S * Hk * D)
    return out.view(B, Hk, D, S)


def _t_last2_bhsd(x):
    """[B, H, S, D] -> [B, H, D, S] via the tiled transpose kernel."""
    ext = get_ext()
    B, H, S, D = x.shape
    if ext is None or not x.is_cuda or x.dtype != torch.bfloat16:
        return x.transpose(-1, -2).contiguous()
    out = ext.transpose_bf16(x.contiguous(), B * H, S, D, D, 1, 0, S * D)
    return out.view(B, H, D, S)


def flash_attn_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                   causal: bool = True,
                   scale: Optional[float] = None) -> torch.Tensor:
    """q,k,v: [B, S, H(kv), D] bf16 -> o [B, S, H, D]. Inference/prefill
    only (no autograd)."""
    q, scale, _ = _scaled(q, scale)
    return get_ext().flash_attn_fwd(_rows(q), _rows(k), _rows(v), scale,
                                    causal, False)[0]


def sdpa_reference(q, k, v, causal=True, scale=None):
    """Plain fp32 reference in the same [B,S,H,D] layout (for tests)."""
    qt, kt, vt = (t.transpose(1, 2).float() for t in (q, k, v))
    rep = qt.shape[1] // kt.shape[1]
    if rep > 1:
        kt = kt.repeat_interleave(rep, dim=1)
        vt = vt.repeat_interleave(rep, dim=1)
    o = torch.nn.functional.scaled_dot_product_attention(
        qt, kt, vt, is_causal=causal, scale=scale)
    return o.transpose(1, 2).to(q.dtype)


def flash_attn_bwd(q, k, v, o, do, lse, causal=True, scale=None):
    """Backward pass in BHSD ([B,H(kv),S,D] bf16; lse [B,H,S] fp32).
    Returns (dq, dk, dv)."""
    q, scale, factor = _scaled(q, scale)
    dq, dk, dv = get_ext().flash_attn_bwd(
        *(_rows(t.transpose(1, 2)) for t in (q, k, v, o, do)),
        lse.contiguous().float(), scale, causal)
    dq = dq if factor == 1 else dq * factor
    return tuple(g.transpose(1, 2).contiguous() for g in (dq, dk, dv))


class FlashAttnFunc(torch.autograd.Function):
    """Training-path flash attention (BSHD in/out)."""

    @staticmethod
    def forward(ctx, q, k, v, causal, scale):
        q, scale, ctx.factor = _scaled(q, scale)
        q, k, v = _rows(q), _rows(k), _rows(v)
        o, lse = get_ext().flash_attn_fwd(q, k, v, scale, causal, True)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.causal, ctx.scale = causal, scale
        return o

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, do):
        q, k, v, o, lse = ctx.saved_tensors
        dq, dk, dv = get_ext().flash_attn_bwd(q, k, v, o, _rows(do), lse,
                                              ctx.scale, ctx.causal)
        return (dq if ctx.factor == 1 else dq * ctx.factor), dk, dv, None, None


class RopeFlashFunc(torch.autograd.Function):
    """Causal attention of unrotated q, k [B, S, H(kv), D]: one launch rotates
    both, and the gradients on their way back in place."""

    @staticmethod
    def forward(ctx, q, k, v, cos, sin, positions):
        ext = get_ext()
        q, k = ext.rope(q.contiguous(), k.contiguous(), cos, sin, positions,
                        False)
        v = _rows(v)
        ctx.scale = 1.0 / math.sqrt(q.size(-1))
        o, lse = ext.flash_attn_fwd(q, k, v, ctx.scale, True, True)
        ctx.save_for_backward(q, k, v, o, lse, cos, sin, positions)
        return o

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, do):
        q, k, v, o, lse, cos, sin, positions = ctx.saved_tensors
        ext = get_ext()
        dq, dk, dv = ext.flash_attn_bwd(q, k, v, o, _rows(do), lse, ctx.scale,
                                        True)
        ext.rope(dq, dk, cos, sin, positions, True, True)
        return dq, dk, dv, None, None, None


def rope_flash_attention(q, k, v, cos, sin, positions=None):
    """Rotary embedding and causal attention, [B, S, H(kv), D] bf16; None where
    the kernels do not apply."""
    grad = torch.is_grad_enabled()
    if not (flash_train_available(q, k) if grad else
            flash_attn_available(q, k) and untransformed()) or (
            positions is None and cos.size(0) < q.size(1)) or (
            positions is not None and positions.dtype != torch.int32):
        return None
    if positions is not None:
        positions = positions.contiguous()
    if grad:
        return RopeFlashFunc.apply(q, k, v, cos, sin, positions)
    q, k = get_ext().rope(q.contiguous(), k.contiguous(), cos, sin, positions,
                          False)
    return flash_attn_fwd(q, k, v)


def flash_attn_func(q, k, v, causal=True, scale=None):
    """Differentiable flash attention, [B,S,H(kv),D] bf16."""
    return FlashAttnFunc.apply(q, k, v, causal, scale)
