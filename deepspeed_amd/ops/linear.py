"""Linear layers.

``Linear`` is torch's, with the backward of ``_Linears``.

``rows_linear``, for a few rows (decoding), and ``tile_linear``, for any more:
the framework's kernels (csrc/rows_linear.hip, csrc/tile_linear.hip) in place of
a library GEMM, with several layers of one input in one launch and the gate's
activation in the epilogue.

Both take the modules themselves and return None wherever calling them is the
thing to do: with gradients (but for several layers of ``tile_linear``), hooks,
autocast, function transforms, tangents or traces, other types, sharded or
replaced modules."""

import weakref

import torch
import torch.nn as nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _module

from ._loader import get_ext

# Most rows that ``rows_linear`` takes: bf16 (more are for ``tile_linear``), and
# int8 (past it the weights are dequantized first).
ROWS, ROWS_INT8 = 32, 64

PLAIN, SWIGLU = 0, 1

# What the library's bf16 products reach for the input's gradient, with the
# weight as stored and transposed (FLOP/s: 1140 to 1425 and 1500 to 1660 over
# 8192 rows), and the transposing kernel (bytes/s, seconds a launch).
DGRAD, DGRAD_T = 1220e12, 1530e12
STREAM, LAUNCH = 5e12, 5e-6

# Largest layers of csrc/tile_linear.hip: a lane's offset in a tile is 32 bits, up
# to 255 rows of 2 bytes a feature (of the output's gradient) or input and a row's
# 128 bytes.
FEATURES, INPUTS = 1 << 23, 1 << 22


def backward_plan(T: int, N: int, K: int):
    """Which operands to transpose in the backward of a layer [N, K] over T
    rows: (weight, for the input's gradient; gradient, input, for the
    weight's). A product reads an operand along the contracted axis faster than
    across it, and transposing costs a read and a write.

    Weight: the library's times jump by up to 1.9 between neighbouring numbers of
    rows (128256 x 4096: 2560 rows 2245 us, 2561 3724), so a rule by rows holds
    on balance only. Over 15 weights of 3072 x 3072 to 152064 x 3584 (us as
    stored and transposed, the copy included): below some 3100 rows large ones
    mostly lose (14336 x 4096: 2560 rows 264 / 271, 3000 285 / 296; 4096 x
    14336: 2700 345 / 399; 128256 x 4096: 2700 3820 / 4378, 3000 2560 / 2585;
    8192 x 8192: 3000 337 / 347), from there on two in three gain (14336 x 4096:
    3111 496 / 390, 3500 324 / 327, 4000 351 / 342, 8192 704 / 640; 128256 x
    4096: 3111 4088 / 3224, 4000 3190 / 2973; 4096 x 4096: 3500 117 / 108; but
    4096 x 14336: 3500 404 / 448, 4000 400 / 370; 32064 x 3072: 3500 904 / 968,
    4000 632 / 626). Small ones wait for the copy to be worth it.
    Gradient of the weight: both operands lie across. Transposing the narrower
    is within 7% of the best choice over all sizes measured (8192 rows: 14336 x
    4096 993 / 756, both 741; 4096 x 14336 994 / 785, both 734; 128256 x 4096
    7178 / 6247, both 6364). Outputs under 256 tiles of 256 x 256 and fewer
    rows stay: there the library splits the contraction over more of the chip
    in its own layout (3072 x 3072 over 32768 rows 598 / 994, 14336 x 4096 over
    1000 rows 160 / 161). So do, from 16384 rows, outputs that nearly fill a
    second round of the 256 CUs (tiles, over 16384 rows: 384 752 / 702, 400 904 /
    1017, 416 1022 / 1056, 448 984 / 1052 and 927 / 1091, 480 1008 / 998, 512 951
    / 790); over 8192 rows they gain a fifth, between the two some gain and some
    lose."""
    flops = 2.0 * T * N * K
    w = T >= 3100 and flops / DGRAD_T + 4.0 * N * K / STREAM + LAUNCH < \
        flops / DGRAD
    tiles = -(-N // 256) * -(-K // 256)
    big = N * K >= 1 << 24 and T >= 2048 and not (
        T >= 16384 and 384 < tiles < 512)
    return w, big and N < K, big and N >= K


def _tiles(T: int, ns) -> int:
    """Tiles of 256 x 256 of outputs [T, n]."""
    return -(-T // 256) * sum(-(-n // 256) for n in ns)


def own_dx(T: int, ns, K: int) -> bool:
    """Whether the input's gradient of layers [n, K] of ``ns`` features over T rows
    is csrc/tile_linear.hip's, which adds the layers up in one product (us, library
    with the copies of ``backward_plan`` and additions, and kernel).

    N 14336, K 4096, 1000 rows 148 / 121, 2300 290 / 259; 18944, K 3584, 2048 rows
    343 / 233; 32064, K 3072, 2559 rows 594 / 401; but 3072, K 8192, 1024 rows 51 / 52.
    From 2560 rows on the library is ahead past 7e10 products where the rows are whole
    tiles of 256 (14336, K 4096: 4096 rows 348 / 355, 8192 643 / 719; 4096, K 4096,
    8192 rows 192 / 207; 14336, K 3072, 8192 544 / 621; over 508 of these the kernel
    takes 0.96 all the same, since the library's times jump between neighbouring
    layers), but for features many times the inputs up to 1.7e11.
    Elsewhere the kernel is, by 7% in the geometric mean (128256, K 3072, 4000 rows
    4175 / 2727; 3072, K 8192 155 / 158), but not where it has a bit more than a round
    of tiles (14336, K 2048, 10000 rows 458 / 600), if there are not too many features.
    Several layers, over 1200: 0.75 of the library's time, whose additions count for
    less the more features there are (4096 + 2 of 1024, K 4096: 8192 rows 422 / 339; 3
    of 3072, K 8192: 4096 rows 550 / 443; whole tiles of rows and 2 of 14336, K 4096:
    4096 rows 715 / 694, 8192 1316 / 1402; 2 of 8192, K 3072, 8192 667 / 697; a bit more
    than a round of tiles: 2 of 11008, K 2048, 10000 rows 729 / 882)."""
    if T <= ROWS or T >= 1 << 30 or K % 8 or K > INPUTS:
        return False
    for n in ns:
        if n % 64 or n < 192 or n > FEATURES:
            return False
    if T < 2560:
        return True
    work, tiles = T * sum(ns) * K, _tiles(T, (K,))
    uneven = T % 256 != 0 and (not 256 < tiles < 400 or
                               (len(ns) == 1 and ns[0] >= 28672))
    if len(ns) > 1:
        return uneven or sum(ns) <= 4 * K or (
            work < 22e10 and max(ns) * K < 1 << 25)
    if max(ns) * K < 1 << 25 and work < (17e10 if ns[0] >= 16 * K else 7e10):
        return True
    return uneven


def own_dw(T: int, N: int, K: int) -> bool:
    """Whether the gradient of a weight [N, K] over T rows is
    csrc/tile_linear.hip's (us, library with the copies of ``backward_plan`` and
    kernel): 4096, K 4096, 4000 rows 138 / 108; 14336, K 4096, 4000 rows 443 / 368,
    6144 576 / 528, 8192 759 / 737, 10000 1147 / 901, 32768 3544 / 2990; 3072, K 3072,
    4000 rows 108 / 78, 24576 447 / 419; 32064, K 8192, 16384 rows 6789 / 6191. Over
    1200 layers and rows from 2560 on 0.87 of the library's time, 1.09 at most. The
    library keeps where the two are closest, vocabularies over many whole tiles of
    rows (0.96 over 44; 128256, K 4096, 8192 rows 6460 / 6284, but of other numbers of
    rows 0.90)."""
    return T > 192 and N % 8 == 0 and K % 8 == 0 and T < 1 << 30 and \
        N <= FEATURES and K <= INPUTS and (
            T < 6144 or T % 256 != 0 or N < 65536 or N * K < 1 << 28)


def own_products(T: int, N: int, K: int):
    """Which products of the backward of a layer [N, K] over T rows are
    csrc/tile_linear.hip's: (the input's gradient, the weight's). It reads either
    operand across the contraction as fast as along it, without a transposed copy.
    """
    return own_dx(T, (N,), K), own_dw(T, N, K)


def one_dw(T: int, ns, K: int) -> bool:
    """Whether the weights' gradients of several layers over T rows are one launch.
    Not where that is a bit more than a round of the 256 CUs over operands past the
    256 MB that the chip caches: the second round is then as long as the first. Over
    400 layers and rows past that size one launch takes, of the time of one each, 1.10
    at up to 288 tiles, 1.12 to 320, 1.03 to 352, 0.99 to 400, 0.89 to 480 and 0.9 from
    there (us, one launch, one each, library: 4096 + 2 of 1024, K 4096, 384 tiles: 14000
    rows 597 / 526 / 765, 32768 1456 / 1185 / 1499; 3 of 3072, K 2048, 288 tiles: 10000
    363 / 355 / 453, 16384 602 / 556 / 709; 4096 + 2 of 512, K 4096, 320 tiles: 16384
    612 / 539 / 714; but 4096 + 2 of 1536, 448 tiles: 16384 739 / 758 / 925; 5120 + 2 of
    1024, K 5120, 560 tiles: 16384 971 / 1035 / 1531)."""
    if 2 * T * (K + sum(ns)) <= 1 << 28:
        return True
    return not 256 < sum(-(-n // 256) for n in ns) * -(-K // 256) < 400


def own_forward(T: int, ns, K: int, mode: int = PLAIN) -> bool:
    """Whether the forward product of layers of ``ns`` features is
    csrc/tile_linear.hip's. Over 20 layers of 1024 x 1024 to 128256 x 4096 and 33 to
    8192 rows the kernel takes 0.65 of the library's time in the geometric mean (us,
    library and kernel: gate and up 14336, K 4096, 224 rows 86 + activation / 57;
    4096, K 14336, 1024 rows 114 / 104; 3584, K 18944, 2331 rows 495 / 256).

    From 2560 rows on, over 1000 layers and rows: 0.95 of the library's time for one
    layer, but where 256 x 256 tiles fill whole rounds of the 256 CUs and contractions
    are long, the library is ahead (4096 rows: N 4096, K 14336 351 / 385; 8192 rows: N
    14336, K 4096 644 / 675; else N 3072, K 4096, 4096 rows 81 / 78, 8192 127 / 120 at K
    3072), and from 65536 features on whole tiles of rows are within 2% either way
    (128256, K 4096, 4096 rows 3016 / 2961). K from 16384 on, over 1400: 0.84 of it, but
    for features in 4096s, which the library's tiles fill best: 4096 of them 0.83
    (4352 rows, K 16384 869 / 456) but in whole rounds (4096 rows, K 16384 354 / 384), 8192
    0.96 and 12288 0.98 but of whole tiles of rows (both 1.00), more 1.02 (8192 rows N
    24576, K 16384 4198 / 4533).
    Several layers, over 1200: 0.80 (3 of 3072, K 3072, 8192 rows 372 / 340; 2 of 11008,
    K 4096, 8192 rows 1306 / 976), but whole tiles of rows of large ones are the
    library's (2 of 8192, K 14336, 4096 rows 1231 / 1286, though over 137 the kernel
    takes 0.87), as are, from 16384 of these on, many products (3 of 4096, K 4096:
    16384 rows 1084 / 1114); gate and up with their activation stay (14336, K 4096,
    8192 rows 1260 + activation / 1379)."""
    if T <= ROWS or K % 64 or not 192 <= K <= INPUTS or any(n % 4 for n in ns):
        return False
    if T < 2560 or mode == SWIGLU:
        return True
    if len(ns) == 1:
        if K >= 16384:
            return ns[0] % 4096 != 0 or (ns[0] < 16384 and T % 256 != 0) or (
                ns[0] < 8192 and _tiles(T, ns) % 256 != 0)
        return T % 256 != 0 or ns[0] < 65536 and (
            K < 3072 or _tiles(T, ns) % 256 != 0)
    return T % 256 != 0 or max(ns) * K < 1 << 26 and (
        T < 16384 or T * sum(ns) * K < 4e11)


def _aligned(*ts) -> bool:
    return all(t.data_ptr() % 16 == 0 for t in ts)


def _forward(x, weights, biases):
    """Outputs of the layers on x, by the kernel where that pays."""
    ns, K = [w.shape[0] for w in weights], x.shape[-1]
    x2 = x.reshape(-1, K).contiguous()
    if own_forward(x2.shape[0], ns, K) and _aligned(x2, *weights) and all(
            b is None or (b.dtype is torch.bfloat16 and b.is_contiguous())
            for b in biases):
        out = get_ext().tile_linear(x2, weights, biases, PLAIN)
        return [o.view(*x.shape[:-1], o.shape[-1]) for o in out]
    return [nn.functional.linear(x, w, b) for w, b in zip(weights, biases)]


def _dx(dys, weights, own: bool):
    """Sum of dy W over the layers."""
    T, K = dys[0].shape[0], weights[0].shape[1]
    sizes = [w.shape[0] for w in weights]
    if own and own_dx(T, sizes, K) and _aligned(*dys, *weights):
        return get_ext().tile_linear_dx(dys, weights)
    dx = None
    for dy, w in zip(dys, weights):
        b = _transposed(w).t() if own and backward_plan(T, *w.shape)[0] else w
        if dx is None:
            dx = dy @ b
        else:       # by the product itself: two reads and a write less
            dx = dx.addmm_(dy, b) if own else dx + dy @ b
    return dx


class GradSlot:
    """Where the gradient of a parameter belongs: ``view``, a part of its owner's
    flat buffer. While it is ``open`` (the owner's backward, nothing there yet; it
    holds the tensor that the parameter has as its gradient) the product of the
    parameter's one layer may be written into it. Autograd then keeps that very
    tensor as the gradient, where it added a new one to the buffer: two reads and a
    write of every weight's gradient, 20 us for 25M values.

    uses: forward products since the owner's last backward; a weight of several
    keeps to the addition. void: a product was given the place, whose parameter
    has no gradient until what that wrote arrives.

    Beside the parameter, not on it: what is on it is saved with it. It lives as
    long as its owner keeps it; since it keeps the parameter, that one's id is not
    another's."""

    __slots__ = ("view", "at", "uses", "open", "void", "weight", "__weakref__")

    def __init__(self, weight, view):
        self.view, self.at = view, view.data_ptr()
        self.uses = 0
        self.open, self.void = None, False
        self.weight = weight
        key = id(weight)
        _slots[key] = weakref.ref(
            self, lambda ref: _slots.get(key) is ref and _slots.pop(key))

    def take(self):
        """The place for a product that is made now, or None. Only from here on
        has the parameter no gradient: hooks that read it see the buffer until
        autograd goes on to it, which it does next (but where the weight is used
        outside of products as well: then when its last gradient is made)."""
        w = self.weight
        if self.open is None or self.uses != 1 or w.grad is not self.open:
            return None
        self.open, self.void = None, True
        w.grad = None
        return self.view.detach()


_slots = {}     # weak references by the id of the parameter


def slot_of(weight):
    """The parameter's ``GradSlot``, or None."""
    ref = _slots.get(id(weight))
    return None if ref is None else ref()


def uses(weight):
    """A product that may write the weight's gradient is being made; its slot."""
    ref = _slots.get(id(weight))
    slot = None if ref is None else ref()
    if slot is not None:
        slot.uses += 1
    return slot


def place(weight):
    """Where the weight's gradient may be written now, or None."""
    slot = slot_of(weight)
    return None if slot is None else slot.take()


def _dw(x, dys, own: bool, slots):
    """dy^T x of the layers, in their weights' places where these are open."""
    T, K = x.shape
    into = [s.take() if own and s else None for s in slots]
    ns = [dy.shape[1] for dy in dys]
    if own and all(own_dw(T, n, K) for n in ns) and _aligned(x, *dys):
        if len(ns) == 1 or one_dw(T, ns, K):
            return get_ext().tile_linear_dw(x, dys, into=into)
        return [get_ext().tile_linear_dw(x, [dy], into=[out])[0]
                for dy, out in zip(dys, into)]
    dws = []
    for dy, out in zip(dys, into):
        a, b = _across(x, dy) if own else (dy.t(), x)
        dws.append(a @ b if out is None else torch.mm(a, b, out=out))
    return dws


def _across(x, dy):
    """Operands of the library's dy^T x, laid out as ``backward_plan`` says."""
    _, dy_t, x_t = backward_plan(x.shape[0], dy.shape[1], x.shape[1])
    return (_transposed(dy) if dy_t else dy.t(),
            _transposed(x).t() if x_t else x)


def add_dw(dw, x, dy):
    """dw += dy^T x."""
    if own_dw(x.shape[0], *dw.shape) and _aligned(x, dy):
        dw += get_ext().tile_linear_dw(x, [dy], into=[None])[0]
    else:
        dw.addmm_(*_across(x, dy))


class _Linears(torch.autograd.Function):
    """x W^T + b of one to three layers on one input. The backward's products lie
    across their operands (dx = dy W across W, dW = dy^T x across both): those of
    ``own_products`` are csrc/tile_linear.hip's, with the input's gradient summed
    over the layers in the product; for the others operands are transposed where
    ``backward_plan`` says. Kept for the backward is what it needs: a frozen layer
    holds no input. ``own``: the forward product may be the kernel's as well.
    Weights' gradients go to their ``GradSlot``."""

    @staticmethod
    def forward(ctx, x, own, *params):
        weights, biases = params[::2], params[1::2]
        need = ctx.needs_input_grad
        ctx.save_for_backward(x if any(need[2::2]) else None,
                              *(w if need[0] else None for w in weights))
        ctx.shape, ctx.features = x.shape, [w.shape for w in weights]
        if len(weights) > 1:
            ctx.set_materialize_grads(False)
        ctx.slots = [uses(w) for w in weights]
        if own:
            out = _forward(x, weights, biases)
        else:
            out = [nn.functional.linear(x, w, b)
                   for w, b in zip(weights, biases)]
        return out[0] if len(out) == 1 else tuple(out)

    @staticmethod
    def backward(ctx, *dys):
        x, *weights = ctx.saved_tensors
        need = ctx.needs_input_grad
        K = ctx.shape[-1]
        grads = [None] * (2 * len(dys))
        used = range(len(dys))
        if len(dys) > 1 and any(dy is None for dy in dys):
            used = [i for i in used if dys[i] is not None]
            if not used:
                return None, None, *grads
            dys, weights = [dys[i] for i in used], [weights[i] for i in used]
        dys = [dy.reshape(-1, ctx.features[i][0]) for i, dy in zip(used, dys)]
        # differentiable products where the gradient itself is differentiated,
        # torch's own where something watches them
        own = (not torch.is_grad_enabled() and untransformed()
               and all(dy.dtype is torch.bfloat16 and not _batched(dy)
                       for dy in dys))
        if own:
            dys = [dy.contiguous() for dy in dys]
        dx = None
        if need[0]:
            dx = _dx(dys, weights, own).view(ctx.shape)
        some = [i for i in used if need[2 + 2 * i]]
        if some:
            x2 = x.reshape(-1, K)
            if own:
                x2 = x2.contiguous()
            theirs = dys if len(some) == len(dys) else \
                [dy for i, dy in zip(used, dys) if i in some]
            for i, dw in zip(some, _dw(x2, theirs, own,
                                       [need[0] and ctx.slots[i]
                                        for i in some])):
                grads[2 * i] = dw
        for i, dy in zip(used, dys):
            if need[3 + 2 * i]:
                grads[2 * i + 1] = dy.sum(0)
        return dx, None, *grads


class _Linear:
    """One layer with torch's forward product."""

    @staticmethod
    def apply(x, weight, bias):
        return _Linears.apply(x, False, weight, bias)


def _transposed(a: torch.Tensor) -> torch.Tensor:
    return get_ext().transpose_2d(a.contiguous())


# Gradients asked for in batches (``is_grads_batched``) have no memory of their own.
_batched = torch._C._functorch.is_legacy_batchedtensor
_interpreter = torch._C._functorch.peek_interpreter_stack
_modes = torch._C._len_torch_dispatch_stack
_trace = torch._C._get_tracing_state


def untransformed() -> bool:
    """No function transform, tangent, trace or dispatch mode is about: these
    see torch's own operations, and a kernel called directly passes them by."""
    return (_interpreter() is None and forward_ad._current_level < 0
            and _modes() == 0 and _trace() is None)


def _plain_autograd() -> bool:
    """Neither one of these nor autocast or a compiler is about: an autograd
    function without rules for them would stop them."""
    return (untransformed() and not torch.compiler.is_compiling()
            and not torch.is_autocast_enabled())


# The forward that each class had when its work was given another way round it.
_TORCHS = nn.Linear.forward
_FORWARD = {nn.Linear: _TORCHS}


def movable(cls):
    """Class decorator: ``unhooked`` may say yes to modules of this class."""
    _FORWARD[cls] = cls.forward
    return cls


def _differentiable(x, weights) -> bool:
    """``_Linears`` takes these with gradients: plain bf16 tensors on a GPU."""
    return (torch.is_grad_enabled() and x.is_cuda and x.dim() > 1
            and type(x) is torch.Tensor and x.dtype is torch.bfloat16
            and x.numel() > 0
            and all(type(w) is nn.Parameter and w.dtype is torch.bfloat16
                    and w.dim() == 2 and w.shape[1] == x.shape[-1]
                    and w.is_contiguous() for w in weights)
            and get_ext() is not None and _plain_autograd()
            and nn.Linear.forward is _TORCHS)


@movable
class Linear(nn.Linear):
    """nn.Linear with the backward of ``_Linears`` on a GPU, and with ``own`` its
    forward. ``loss``, labels and rows a chunk: ``head_loss`` in the place of
    outputs."""

    def forward(self, x, own: bool = False, loss=None):
        if loss is not None:
            from .cross_entropy import head_loss
            return head_loss(self, x, *loss)
        w = self.weight
        if _differentiable(x, (w,)):
            T = x.numel() // w.shape[1]
            if any(own_products(T, *w.shape)) or \
                    any(backward_plan(T, *w.shape)) or \
                    (own and own_forward(T, w.shape[:1], w.shape[1])):
                return _Linears.apply(x, own, w, self.bias)
        return super().forward(x)


def call(mod: nn.Module, x):
    """The module on x: a layer of this framework that at most the framework's
    own hooks watch may take its forward product itself."""
    if type(mod) is Linear and unhooked(mod, internal_ok=True):
        return mod(x, own=True)
    return mod(x)


def all_unhooked(mods) -> bool:
    """``unhooked`` of each of them."""
    if nn.Linear.forward is not _TORCHS or \
            _module._global_forward_hooks or \
            _module._global_forward_pre_hooks or \
            _module._global_backward_hooks or \
            _module._global_backward_pre_hooks:
        return False
    for mod in mods:
        cls = type(mod)
        if "forward" in mod.__dict__ or mod._compiled_call_impl is not None or \
                cls.forward is not _FORWARD.get(cls) or \
                mod._forward_hooks or mod._forward_pre_hooks or \
                mod._backward_hooks or mod._backward_pre_hooks:
            return False
    return True


def unhooked(mod: nn.Module, internal_ok: bool = False) -> bool:
    """No hook sees the module's call and no other forward takes it (one set on
    the module or on its class, or a compiled one): its work may move
    elsewhere. With ``internal_ok`` the call itself stays, in another form that
    the framework's own hooks (marked ``_ds_internal``) take as well."""
    cls = type(mod)
    if "forward" in mod.__dict__ or mod._compiled_call_impl is not None or \
            cls.forward is not _FORWARD.get(cls) or \
            nn.Linear.forward is not _TORCHS or \
            _module._global_forward_hooks or \
            _module._global_forward_pre_hooks or \
            _module._global_backward_hooks or \
            _module._global_backward_pre_hooks:
        return False
    if not (mod._forward_hooks or mod._forward_pre_hooks
            or mod._backward_hooks or mod._backward_pre_hooks):
        return True
    return internal_ok and all(
        getattr(h, "_ds_internal", False)
        for hooks in (mod._forward_hooks, mod._forward_pre_hooks,
                      mod._backward_hooks, mod._backward_pre_hooks)
        for h in hooks.values())


def rows_linear(x: torch.Tensor, mods, mode: int = PLAIN,
                hooks_ran: bool = False):
    """Outputs of the linear modules ``mods`` on x [..., K], a list: one each,
    or with ``SWIGLU`` silu(first) * second. ``hooks_ran``: called from inside
    the module's own call. None when ineligible."""
    if type(x) is not torch.Tensor or torch.is_grad_enabled() or \
            not x.is_cuda or x.dtype is not torch.bfloat16:
        return None
    K = x.shape[-1]
    M = x.numel() // K if K else 0
    if not 1 <= M <= ROWS_INT8 or K % 256 or get_ext() is None or \
            torch.is_autocast_enabled() or torch.compiler.is_compiling() or \
            not untransformed():
        return None
    kind = type(mods[0])
    weights, scales, biases, group = [], [], [], 0
    for m in mods:
        if type(m) is not kind or not (hooks_ran or unhooked(m)):
            return None
        if kind is Linear or kind is nn.Linear:
            w = m.weight
            if w.dtype is not torch.bfloat16 or \
                    type(w) is not nn.Parameter or w.shape[1:] != (K,):
                return None
        elif hasattr(kind, "int8_rows"):
            p = m.int8_rows(K)
            if p is None or p[2] % 256 or group not in (0, p[2]):
                return None
            w, scale, group = p
            scales.append(scale)
        else:
            return None
        b = m.bias
        if not w.is_cuda or not w.is_contiguous() or w.data_ptr() % 16 or (
                b is not None and (b.dtype is not torch.bfloat16
                                   or not b.is_contiguous())):
            return None
        weights.append(w)
        biases.append(b)
    if M > ROWS and not scales:
        return None
    x2 = x.reshape(M, K).contiguous()
    if x2.data_ptr() % 16:
        return None
    out = get_ext().rows_linear(x2, weights, scales, biases, group, mode)
    return [o.view(*x.shape[:-1], o.shape[-1]) for o in out]


def _with_gradients(x, mods):
    """Several layers of a training step's rows in one function, or None: their
    products are one launch each way and nothing adds the input's gradients up."""
    if len(mods) < 2 or not all(type(m) is Linear and unhooked(m)
                                for m in mods) or \
            not _differentiable(x, [m.weight for m in mods]):
        return None
    T, K = x.numel() // x.shape[-1], x.shape[-1]
    ns = [m.weight.shape[0] for m in mods]
    if not own_forward(T, ns, K) and not own_dx(T, ns, K) and \
            not any(own_dw(T, n, K) for n in ns):
        return None
    return _Linears.apply(x, True, *(p for m in mods
                                     for p in (m.weight, m.bias)))


def tile_linear(x: torch.Tensor, mods, mode: int = PLAIN):
    """``rows_linear`` for more than ``ROWS`` rows and torch's or the models' own
    bf16 layers, where ``own_forward`` says so."""
    if torch.is_grad_enabled():
        return _with_gradients(x, mods) if mode == PLAIN else None
    if type(x) is not torch.Tensor or \
            not x.is_cuda or x.dtype is not torch.bfloat16:
        return None
    K = x.shape[-1]
    M = x.numel() // K if K else 0
    if M <= ROWS or get_ext() is None or torch.is_autocast_enabled() or \
            torch.compiler.is_compiling() or not untransformed():
        return None
    weights, biases = [], []
    for m in mods:
        if type(m) not in (Linear, nn.Linear) or not unhooked(m):
            return None
        w, b = m.weight, m.bias
        if w.dtype is not torch.bfloat16 or type(w) is not nn.Parameter or \
                w.shape[1:] != (K,) or not w.is_cuda or \
                not w.is_contiguous() or w.data_ptr() % 16 or (
                    mode == SWIGLU and w.shape != mods[0].weight.shape) or (
                    b is not None and (b.dtype is not torch.bfloat16
                                       or not b.is_contiguous())):
            return None
        weights.append(w)
        biases.append(b)
    if not own_forward(M, [w.shape[0] for w in weights], K, mode):
        return None
    x2 = x.reshape(M, K).contiguous()
    if x2.data_ptr() % 16:
        return None
    out = get_ext().tile_linear(x2, weights, biases, mode)
    return [o.view(*x.shape[:-1], o.shape[-1]) for o in out]
