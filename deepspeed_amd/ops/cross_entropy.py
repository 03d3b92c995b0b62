"""Fused cross-entropy (bf16 logits, no fp32 materialization).

See csrc/cross_entropy.hip. The autograd wrapper recomputes nothing: the
forward saves (logits, labels, lse) and the backward emits bf16 dlogits in
one elementwise pass. The default of the chunked-CE loss path on a GPU
(DS_AMD_FUSED_CE=0 opts out); the torch fallback defines the semantics and
runs everywhere."""

import os

import torch

from ._loader import get_ext


class _FusedCE(torch.autograd.Function):
    """(sum of the rows' losses, labels that count), or with ``mean`` their
    quotient; what torch makes of it takes ten launches more."""

    @staticmethod
    def forward(ctx, logits, labels, ignore_index, mean=False):
        total, count, quotient, lse = get_ext().ce_loss(logits, labels,
                                                        ignore_index)
        ctx.save_for_backward(logits, labels, lse, count if mean else None)
        ctx.ignore_index = ignore_index
        if mean:
            return quotient
        ctx.mark_non_differentiable(count)
        return total, count

    @staticmethod
    def backward(ctx, g, _gcount=None):
        logits, labels, lse, count = ctx.saved_tensors
        d = get_ext().ce_bwd(logits, labels, lse, g.contiguous().float(),
                             ctx.ignore_index, count)
        return d, None, None, None


def fused_ce_available(logits) -> bool:
    """Default ON: the fused kernel computes loss+lse from bf16 logits and
    emits bf16 dlogits in one pass — no [tokens, vocab] fp32 materialization,
    no cunn_SoftMax pair. DS_AMD_FUSED_CE=0 opts out."""
    return (os.environ.get("DS_AMD_FUSED_CE", "1") != "0"
            and get_ext() is not None and logits.is_cuda
            and logits.dtype == torch.bfloat16)


def fused_cross_entropy_sum(logits, labels, ignore_index=-100):
    """Returns (summed loss, valid-token count) like the chunked-CE inner
    loop expects. Falls back to the fp32 torch path when ineligible."""
    if fused_ce_available(logits):
        return _FusedCE.apply(logits.contiguous(), labels.contiguous(),
                              ignore_index)
    lf = logits.float()
    loss = torch.nn.functional.cross_entropy(lf, labels,
                                             ignore_index=ignore_index,
                                             reduction="sum")
    return loss, (labels != ignore_index).sum().float()


def fused_cross_entropy_mean(logits, labels, ignore_index=-100):
    """The mean over the labels that count (0 without any)."""
    if fused_ce_available(logits):
        return _FusedCE.apply(logits.contiguous(), labels.contiguous(),
                              ignore_index, True)
    loss, count = fused_cross_entropy_sum(logits, labels, ignore_index)
    return loss / count.clamp(min=1)
