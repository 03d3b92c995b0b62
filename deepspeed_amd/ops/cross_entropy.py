"""Fused cross-entropy (bf16 logits, no fp32 materialization).

See csrc/cross_entropy.hip. The autograd wrapper recomputes nothing: the
forward saves (logits, labels, lse) and the backward emits bf16 dlogits in
one elementwise pass. The default of the chunked-CE loss path on a GPU
(DS_AMD_FUSED_CE=0 opts out); the torch fallback defines the semantics and
runs everywhere."""

import os

import torch

from . import linear
from ._loader import get_ext


_saved_hooks = torch._C._autograd._top_saved_tensors_default_hooks


def _dlogits(logits, labels, lse, g, ignore_index, count=None):
    """Gradient of the logits of a sum of losses, or with ``count`` of their mean;
    by torch's own operations where it is differentiated itself."""
    if not torch.is_grad_enabled():
        return get_ext().ce_bwd(logits, labels, lse, g.contiguous().float(),
                                ignore_index, count)
    live = (labels != ignore_index)[:, None]
    p = torch.softmax(logits.float(), -1)
    d = p.scatter_add(1, torch.where(live, labels[:, None], 0),
                      p.new_full((len(p), 1), -1.0))
    g = g.float() if count is None else g.float() / count.clamp(min=1)
    return torch.where(live, d * g, 0).to(logits.dtype)


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
        d = _dlogits(logits, labels, lse, g, ctx.ignore_index, count)
        return d, None, None, None


class _HeadLoss(torch.autograd.Function):
    """(sum of the rows' losses, labels that count) of the logits x W^T, in chunks
    of rows. As one node: gradients of x are made in their places, W is transposed
    once or twice and the library's products add the chunks' gradients of W up
    (those of the kernels, ``own_dw``, are added in bf16), where slices and calls of
    a head each clear, fill and add up gradients of all rows and of W (32768 rows of
    4096, 128256 features in four chunks: 3.4 of 162 ms). The logits
    are outputs too: where the gradients are differentiated themselves, what they
    owe to the logits comes back here. Kept is what a chunk's calls would keep, and
    let go as early: a frozen head holds no input, and each chunk's logits go when
    their gradient, one chunk's at a time, is made."""

    @staticmethod
    def forward(ctx, x, weight, labels, rows, ignore_index):
        ctx.rows, ctx.ignore_index = rows, ignore_index
        ctx.set_materialize_grads(False)
        total, count, lses, outputs = None, None, [], []
        for xs, ys in zip(x.split(rows), labels.split(rows)):
            linear.uses(weight)     # a use each: W's place is not for their sum
            logits = linear._forward(xs, [weight], [None])[0]
            t, c, _, lse = get_ext().ce_loss(logits, ys, ignore_index)
            total = t if total is None else total + t
            count = c if count is None else count + c
            lses.append(lse)
            outputs.append(logits)
        need_x, need_w = ctx.needs_input_grad[:2]
        ctx.save_for_backward(x if need_w else None, weight if need_x else None,
                              labels, *lses, *outputs)
        ctx.mark_non_differentiable(count)
        return (total, count, *outputs)

    @staticmethod
    def backward(ctx, g, _gcount, *more):
        x, w, labels, *kept = ctx.saved_tensors
        rows, (need_x, need_w) = ctx.rows, ctx.needs_input_grad[:2]
        n = len(more)
        lses, outputs = kept[:n], kept[n:]
        del kept
        ys = labels.split(rows)
        xs = x.split(rows) if need_w else [None] * n

        def gradient(i):
            logits, outputs[i], d = outputs[i], None, more[i]
            if g is None:
                return torch.zeros_like(logits) if d is None else d
            own = _dlogits(logits, ys[i], lses[i], g, ctx.ignore_index)
            return own if d is None else own + d
        # differentiable products where the gradient itself is differentiated,
        # torch's own where something watches them
        if torch.is_grad_enabled() or not linear.untransformed() or any(
                d is not None and linear._batched(d) for d in more):
            ds = [gradient(i) for i in range(n)]
            dx = torch.cat([d @ w for d in ds]) if need_x else None
            dw = sum(d.t() @ p for d, p in zip(ds, xs)) if need_w else None
            return dx, dw, None, None, None
        ctx.maybe_clear_saved_tensors()     # unless the graph is to stay
        dx = dw = turned = None
        gone = 0
        # a shorter chunk first: its gradient is beside all of the logits
        for i in range(n) if len(ys[-1]) == rows else (n - 1, *range(n - 1)):
            d = gradient(i).contiguous()
            T, at = len(d), slice(i * rows, (i + 1) * rows)
            gone += T
            if need_x:
                to, K = None if dx is None else dx[at], w.shape[1]
                if linear.own_dx(T, w.shape[:1], K) and linear._aligned(d, w):
                    part = linear._dx([d], [w], True)
                elif linear.backward_plan(T, *w.shape)[0]:
                    if turned is None:
                        turned = linear._transposed(w)
                    part = torch.mm(d, turned.t(), out=to)
                else:
                    part = torch.mm(d, w, out=to)
                # kept where the logits that are gone have left room for it
                if 2 * w.numel() + len(labels) * K > gone * len(w):
                    turned = None
            if dw is not None:
                linear.add_dw(dw, xs[i], d)
            elif need_w:
                dw = linear._dw(xs[i], [d], True, [None])[0]
            del d
            if need_x:
                if dx is None:      # not beside all of the logits
                    dx = w.new_empty(len(labels), K)
                if part is not to:
                    dx[at] = part
                del part
        return dx, dw, None, None, None


def head_loss(head, x, labels, rows, ignore_index=-100):
    """(sum of the rows' losses, labels that count) of ``head``, a ``linear.Linear``
    that is being called. Its weight is looked at here, behind the hooks that may
    have filled it in. What the node is not for goes a chunk at a time: weights of
    another form or number of inputs, which torch's product takes or refuses,
    nothing to differentiate, and hooks on what is saved, which then get a chunk's
    logits back when these are needed."""
    w = head.weight
    if linear._differentiable(x, (w,)) and head.bias is None and \
            (x.requires_grad or w.requires_grad) and _saved_hooks(False) is None:
        return _HeadLoss.apply(x, w, labels, rows, ignore_index)[:2]
    total = count = 0
    for xs, ys in zip(x.split(rows), labels.split(rows)):
        t, c = fused_cross_entropy_sum(linear.Linear.forward(head, xs, True), ys,
                                       ignore_index)
        total, count = total + t, count + c
    return total, count


def head_loss_fits(head, x) -> bool:
    """A head without bias of the framework's own, watched by its own hooks at
    most, and rows with gradients: one that takes ``loss``."""
    return (type(head) is linear.Linear and head.bias is None
            and linear.unhooked(head, internal_ok=True)
            and x.is_contiguous() and linear._differentiable(x, ())
            and type(head.weight) is torch.nn.Parameter
            and head.weight.dtype is torch.bfloat16
            and fused_ce_available(x))


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
