"""Embedding whose table's gradient is the framework's kernel
(csrc/embedding.hip): only the rows of the batch's tokens are moved, into the
place where the optimizer reads the gradient if that is known."""

import torch
import torch.nn as nn

from ._loader import get_ext
from .linear import _batched, _plain_autograd, untransformed, uses

# Most tokens, rows and columns of the kernel's tables.
TOKENS, ROWS, COLUMNS = 32768, (1 << 30) - 1, 1 << 20


def fits(tokens: int, rows: int, columns: int) -> bool:
    """Whether the kernel takes the gradient of a table. Its places, 4 bytes for
    each row and 256 tokens and a bit more (80 MB for 152064 rows and 32768
    tokens), may take as much memory as the gradient itself: ten million rows of
    64 would want 5.3 GB of it beside one of 1.3."""
    blocks = -(-tokens // 256)
    return 0 < tokens <= TOKENS and 0 < rows <= ROWS and \
        0 < columns <= COLUMNS and columns % 8 == 0 and \
        4 * (blocks + -(-blocks // 32)) <= 2 * columns


class _Embed(torch.autograd.Function):
    """Kept for the backward are the tokens, and of the weight its shape and
    ``GradSlot``."""

    @staticmethod
    def forward(ctx, ids, weight, padding):
        ctx.save_for_backward(ids)
        ctx.shape, ctx.padding = weight.shape, padding
        ctx.slot = uses(weight)
        return nn.functional.embedding(ids, weight)

    @staticmethod
    def backward(ctx, dy):
        ids, = ctx.saved_tensors
        V, H = ctx.shape
        if torch.is_grad_enabled() or not untransformed() or _batched(dy) or \
                dy.dtype is not torch.bfloat16:
            return None, torch.ops.aten.embedding_dense_backward(
                dy, ids, V, ctx.padding, False), None
        dy = dy.reshape(-1, H).contiguous()
        if dy.data_ptr() % 16:
            dy = dy.clone()
        return None, get_ext().embedding_bwd(
            ids.reshape(-1).contiguous(), dy, V, ctx.padding,
            ctx.slot and ctx.slot.take()), None


_TORCHS = nn.Embedding.forward


class Embedding(nn.Embedding):
    """nn.Embedding with the backward of ``_Embed`` on a GPU."""

    def forward(self, ids):
        w = self.weight
        if torch.is_grad_enabled() and type(w) is nn.Parameter and \
                w.requires_grad and w.is_cuda and \
                w.dtype is torch.bfloat16 and w.dim() == 2 and \
                w.is_contiguous() and \
                type(ids) is torch.Tensor and ids.dtype is torch.long and \
                ids.device == w.device and fits(ids.numel(), *w.shape) and \
                self.max_norm is None and not self.sparse and \
                not self.scale_grad_by_freq and get_ext() is not None and \
                _plain_autograd() and nn.Embedding.forward is _TORCHS:
            return _Embed.apply(ids, w, -1 if self.padding_idx is None
                                else self.padding_idx)
        return super().forward(ids)
