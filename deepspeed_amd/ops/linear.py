"""Linear layers of a few rows (decoding): the weight-streaming kernel of
csrc/rows_linear.hip in place of a library GEMM, with several layers of one
input in one launch and the gate's activation or the residual in its epilogue.

``rows_linear`` takes the modules themselves and returns None wherever calling
them is the thing to do: with gradients, hooks, autocast, other types, sharded
or replaced modules, or more rows than the kernel is the faster one for."""

import torch
import torch.nn as nn
from torch.nn.modules import module as _module

from ._loader import get_ext

# Most rows: at 64 the library's product takes half the kernel's time (N 14336:
# 26.6 to 49.8 us); with int8 weights it needs them dequantized first (85 us).
ROWS, ROWS_INT8 = 32, 64

PLAIN, SWIGLU = 0, 1


def unhooked(mod: nn.Module) -> bool:
    """No hook sees the module's call: its work may move elsewhere."""
    return not (mod._forward_hooks or mod._forward_pre_hooks
                or mod._backward_hooks or mod._backward_pre_hooks
                or _module._global_forward_hooks
                or _module._global_forward_pre_hooks
                or _module._global_backward_hooks
                or _module._global_backward_pre_hooks)


def rows_linear(x: torch.Tensor, mods, mode: int = PLAIN, residual=None,
                hooks_ran: bool = False):
    """Outputs of the linear modules ``mods`` on x [..., K], a list: one each,
    or with ``SWIGLU`` silu(first) * second. ``residual`` is added to the first
    output. ``hooks_ran``: called from inside the module's own call. None when
    ineligible."""
    if torch.is_grad_enabled() or not x.is_cuda or \
            x.dtype is not torch.bfloat16 or type(x) is not torch.Tensor:
        return None
    K = x.shape[-1]
    M = x.numel() // K if K else 0
    if not 1 <= M <= ROWS_INT8 or K % 256 or get_ext() is None or \
            torch.is_autocast_enabled() or torch.compiler.is_compiling():
        return None
    from ..linear.optimized_linear import WOQLinear
    kind = type(mods[0])
    weights, scales, biases, group = [], [], [], 0
    for m in mods:
        if type(m) is not kind or not (hooks_ran or unhooked(m)):
            return None
        if kind is nn.Linear:
            w = m.weight
            if M > ROWS or w.dtype is not torch.bfloat16 or \
                    type(w) is not nn.Parameter or w.shape[1:] != (K,):
                return None
        elif kind is WOQLinear:
            p = m.qweight
            w, group = p.q, p.cfg.group_size
            if p.cfg.q_bits != 8 or group % 256 or \
                    group != mods[0].qweight.cfg.group_size or \
                    p.shape[1:] != (K,) or \
                    w.numel() != p.shape[0] * K or not unhooked(p):
                return None
            scales.append(p.scales)
        else:
            return None
        b = m.bias
        if not w.is_cuda or not w.is_contiguous() or w.data_ptr() % 16 or (
                b is not None and (b.dtype is not torch.bfloat16
                                   or not b.is_contiguous())):
            return None
        weights.append(w)
        biases.append(b)
    if residual is not None and (residual.dtype is not torch.bfloat16 or
                                 not residual.is_contiguous()):
        return None
    x2 = x.reshape(M, K).contiguous()
    if x2.data_ptr() % 16:
        return None
    out = get_ext().rows_linear(x2, weights, scales, biases, residual, group,
                                mode)
    return [o.view(*x.shape[:-1], o.shape[-1]) for o in out]
