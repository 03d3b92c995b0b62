"""Linear layers of many rows: which calls take the kernel (CPU) and every tile
of the kernel against fp64 products, forward and backward (GPU)."""

import pytest
import torch
import torch.nn as nn

from deepspeed_amd.ops import linear as L
from deepspeed_amd.ops._loader import get_ext
from deepspeed_amd.ops.linear import SWIGLU, Linear, call, tile_linear

# rows, features and stages of the tiles, in the kernel's order
TILES = [(64, 64, 8), (64, 128, 6), (128, 64, 6), (128, 128, 5), (128, 256, 3),
         (192, 128, 4), (192, 256, 2), (256, 128, 3), (256, 192, 2),
         (256, 256, 2)]
WIDE = len(TILES) - 1


def test_calls_left_alone():
    lin = Linear(256, 16).bfloat16()
    x = torch.randn(40, 256).bfloat16()
    with torch.no_grad():
        assert tile_linear(x, (lin,)) is None      # on the CPU
    assert tile_linear(x, (lin, lin)) is None


def test_largest_of_the_widest_tile():
    """256 x 256 reaches its rows and outputs by 32 bits: 2^23 features of the
    output's gradient are one too many, as are 2^22 columns stored."""
    ext = get_ext()
    if ext is None:
        pytest.skip("the plan is the extension's")
    most = 1 << 23
    assert ext.tile_linear_plan([most - 64], 8192, 4096, 2)[0] == WIDE
    assert ext.tile_linear_plan([most], 8192, 4096, 2)[0] != WIDE
    assert ext.tile_linear_plan([4096, most], 8192, 4096, 2)[0] != WIDE
    assert ext.tile_linear_plan([most], 8192, 4096, 3)[0] == WIDE
    most = 1 << 22
    assert ext.tile_linear_plan([most - 8], 8192, 4096, 0)[0] == WIDE
    assert ext.tile_linear_plan([most], 8192, 4096, 0)[0] != WIDE
    assert ext.tile_linear_plan([4096], 8192, most - 8, 3)[0] == WIDE
    assert ext.tile_linear_plan([4096], 8192, most, 3)[0] != WIDE


def _inputs(m, ns, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def new(*shape, std=1.0):
        return (std * torch.randn(shape, device="cuda", generator=g)).bfloat16()
    return (new(m, k), [new(n, k, std=0.05) for n in ns],
            [new(n) if i % 2 == 0 else None for i, n in enumerate(ns)])


def _want(x, ws, bs, mode):
    y = [x.double() @ w.double().t() + (0 if b is None else b.double())
         for w, b in zip(ws, bs)]
    return [nn.functional.silu(y[0]) * y[1]] if mode == SWIGLU else y


def _close(got, want):
    # fp32 sums rounded to bf16 once
    err = (got.double() - want).abs()
    lim = 2.0 ** -8 * want.abs() + 2.0 ** -16 * want.abs().max()
    assert (err <= lim).all(), (err / lim).max()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("rows", [-1, 0, 1])        # beside a whole tile
@torch.no_grad()
def test_every_tile_gpu(tile, rows):
    from deepspeed_amd.ops import _C
    bm, bn, stages = TILES[tile]
    for ns, splits, mode in (((bn,), 1, 0), ((bn + 4, 4, bn - 4), 1, 0),
                             ((2 * bn + 8, bn - 8), 1, 0), ((bn + 12,), 3, 0),
                             ((bn // 2 + 4,) * 2, 1, 1), ((bn,) * 2, 1, 1)):
        if mode and (bm, bn) == (256, 192):
            continue
        # the fewest stages, one more, and a longer loop
        for steps in (stages, stages + 1, 2 * stages + 3):
            m, k = bm + rows, 64 * (steps * splits + (splits > 1))
            x, ws, bs = _inputs(m, ns, k, steps)
            got = _C.tile_linear(x, ws, bs, mode, tile, splits)
            for y, want in zip(got, _want(x, ws, bs, mode)):
                _close(y, want)
        with pytest.raises(RuntimeError):
            _C.tile_linear(x[:, :64 * (stages - 1)].contiguous(),
                           [w[:, :64 * (stages - 1)].contiguous()
                            for w in ws], bs, mode, tile, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [33, 64, 130, 257, 1000, 2331])
@torch.no_grad()
def test_modules_gpu(m):
    """The chosen tiles, through the modules: several tiles each way, splits."""
    for ns, k, mode in (((512, 128, 128), 1024, 0), ((260,), 4096, 0),
                        ((1800, 1800), 192, 1), ((5000,), 256, 0)):
        x, ws, bs = _inputs(m, ns, k, m)
        mods = []
        for w, b in zip(ws, bs):
            lin = Linear(k, w.shape[0], bias=b is not None, device="cuda",
                         dtype=torch.bfloat16)
            lin.weight.copy_(w)
            if b is not None:
                lin.bias.copy_(b)
            mods.append(lin)
        x = x.view(1, m, k)
        for y, want in zip(tile_linear(x, mods, mode),
                           _want(x, ws, bs, mode)):
            assert y.shape == (1, m, y.shape[-1])
            _close(y, want)
        h = mods[0].register_forward_hook(lambda *a: None)
        assert tile_linear(x, mods, mode) is None
        h.remove()


@pytest.mark.gpu
@torch.no_grad()
def test_refused_gpu():
    def call(m, k, n, dtype=torch.bfloat16):
        lin = Linear(k, n, bias=False, device="cuda", dtype=dtype)
        return tile_linear(torch.randn(m, k, device="cuda", dtype=dtype),
                           (lin,))
    assert call(40, 256, 64) is not None
    assert call(32, 256, 64) is None       # rows_linear's
    assert call(40, 256, 62) is None
    assert call(40, 224, 64) is None
    assert call(40, 128, 64) is None
    assert call(40, 256, 64, torch.float16) is None
    with torch.enable_grad():              # one layer is the module's own
        assert call(40, 256, 64) is None
        lin = Linear(256, 64, device="cuda", dtype=torch.bfloat16)
        x = torch.randn(40, 256, device="cuda", dtype=torch.bfloat16)
        assert "_Linears" in type(tile_linear(x, (lin, lin))[0].grad_fn
                                  ).__name__
        assert tile_linear(x, (lin, lin), SWIGLU) is None


def _limit(want, terms):
    # one rounding to bf16 of an fp32 sum
    return 2.0 ** -8 * want.abs() + 2.0 ** -20 * terms ** 0.5 * \
        want.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@torch.no_grad()
def test_every_tile_backward_gpu(tile):
    from deepspeed_amd.ops import _C
    bm, bn, stages = TILES[tile]
    for rows, more in ((-1, 8), (0, 0), (1, -8)):      # beside a whole tile
        for steps, splits in ((stages, 1), (stages + 1, 1),
                              (3 * stages + 4, 3)):
            # the input's gradient: over one layer, and over three
            for ns in ((64 * steps,), (64 * (steps - 1), 64), (64, 64 * steps,
                                                              128)):
                x, ws, _ = _inputs(bm + rows, ns, bn + more, steps)
                dys = [_inputs(bm + rows, (), n, n)[0] for n in ns]
                want = sum(d.double() @ w.double() for d, w in zip(dys, ws))
                err = (_C.tile_linear_dx(dys, ws, tile, splits).double()
                       - want).abs()
                assert (err <= _limit(want, sum(ns))).all()
            if bm == 64:        # its rows' halves are narrower than a block
                with pytest.raises(RuntimeError):
                    _C.tile_linear_dw(x, dys, tile, 1)
                continue
            # the weights': rows that end anywhere in a stage
            for end in (-63, -31, -8, -1, 0):
                m, ns = 64 * steps + end, (bm + more, 8, 2 * bm - 8)
                x, _, _ = _inputs(m, (), bn + more, steps)
                dys = [_inputs(m, (), n, n)[0] for n in ns]
                for got, d in zip(_C.tile_linear_dw(x, dys, tile, splits),
                                  dys):
                    want = d.double().t() @ x.double()
                    err = (got.double() - want).abs()
                    assert (err <= _limit(want, m)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [2, 3, 4, 5, 9])
@torch.no_grad()
def test_widest_tile_in_rounds_gpu(steps):
    """256 x 256: more tiles than the chip has CUs, over the shortest contractions
    and longer ones, in one part and in uneven ones."""
    from deepspeed_amd.ops import _C
    wide, k = WIDE, 64 * steps
    for m, ns, mode in ((4100, (4360,), 0), (2305, (6148, 516, 264), 0),
                        (2100, (4100, 4100), SWIGLU)):
        x, ws, bs = _inputs(m, ns, k, steps)
        for y, want in zip(_C.tile_linear(x, ws, bs, mode, wide, 1),
                           _want(x, ws, bs, mode)):
            _close(y, want)
    for splits in (2, 3):
        x, ws, bs = _inputs(2305, (4100, 516, 264), 64 * (splits * steps + 1), steps)
        for y, want in zip(_C.tile_linear(x, ws, bs, 0, wide, splits),
                           _want(x, ws, bs, 0)):
            _close(y, want)
    for splits in (1, 2):       # dx [4100, 4360] over two layers, dW of as many
        ns = (64 * splits * steps - 64, 64)
        _, ws, _ = _inputs(1, ns, 4360, steps)
        dys = [_inputs(4100, (), n, n)[0] for n in ns]
        want = sum(d.double() @ w.double() for d, w in zip(dys, ws))
        err = (_C.tile_linear_dx(dys, ws, wide, splits).double() - want).abs()
        assert (err <= _limit(want, sum(ns))).all()
        m = 64 * splits * steps - 3
        x, _, _ = _inputs(m, (), 4360, steps)
        dys = [_inputs(m, (), n, n)[0] for n in (4104, 264)]
        for got, d in zip(_C.tile_linear_dw(x, dys, wide, splits), dys):
            want = d.double().t() @ x.double()
            assert ((got.double() - want).abs() <= _limit(want, m)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile,bm,bn,least", [
    (6, 192, 256, 2), (8, 256, 192, 2), (10, 192, 192, 3)])
@pytest.mark.parametrize("more", [0, 1, 2, 3, 7])
@torch.no_grad()
def test_tiles_by_four_waves_gpu(tile, bm, bn, least, more):
    """Several tiles of rows: features that end anywhere in a lane's eight or six and
    in a tile, layers that end in one, gates, both gradients."""
    from deepspeed_amd.ops import _C
    steps = least + more
    k = 64 * steps
    for m, ns in ((bm + 1, (bn + 4,)), (2 * bm + 1, (3 * bn + 4, 4, bn - 4)),
                  (700, (1000, 2 * bn + 8)), (2600, (3076,))):
        x, ws, bs = _inputs(m, ns, k, steps)
        for biases in (bs, [None] * len(ns)):
            for y, want in zip(_C.tile_linear(x, ws, biases, 0, tile, 1),
                               _want(x, ws, biases, 0)):
                _close(y, want)
    if bn == 256:
        for m, n in ((bm + 1, 132), (700, 1004), (2600, 2056)):
            x, ws, bs = _inputs(m, (n, n), 64 * (23 + steps), steps)
            _close(_C.tile_linear(x, ws, bs, SWIGLU, tile, 1)[0],
                   _want(x, ws, bs, SWIGLU)[0])
    for m, ns, k in ((bm + 1, (64 * steps,), bn + 8),
                     (700, (64 * (steps - 1), 64), 2 * bn - 8),
                     (2600, (64, 64 * steps, 128), 3080)):
        _, ws, _ = _inputs(1, ns, k, steps)
        dys = [_inputs(m, (), n, n)[0] for n in ns]
        want = sum(d.double() @ w.double() for d, w in zip(dys, ws))
        err = (_C.tile_linear_dx(dys, ws, tile, 1).double() - want).abs()
        assert (err <= _limit(want, sum(ns))).all()
    for end, ns, k in ((-63, (bm,), bn), (-31, (bm - 8, 8, 2 * bm + 8), bn + 8),
                       (-8, (1000,), 2 * bn - 8), (0, (3080, 264), 3080)):
        m = 64 * steps + end
        x, _, _ = _inputs(m, (), k, steps)
        dys = [_inputs(m, (), n, n)[0] for n in ns]
        for got, d in zip(_C.tile_linear_dw(x, dys, tile, 1), dys):
            want = d.double().t() @ x.double()
            assert ((got.double() - want).abs() <= _limit(want, m)).all()


def test_short_gradients():
    """Those of few stages are the largest tile's by eight waves, where what was
    measured of the tiles by four has them behind."""
    ext = get_ext()
    if ext is None:
        pytest.skip("the plan is the extension's")
    plan, eight = ext.tile_linear_plan, len(TILES) + 1
    for m, n, k in ((4000, 512, 11008), (4000, 768, 14336), (6000, 512, 28672)):
        assert plan([n], m, k, 2)[0] == eight
    assert plan([1024], 4000, 3072, 2)[0] in (6, 8)
    for n, k in ((32064, 3072), (3072, 18944)):
        assert plan([n], 512, k, 3)[0] == eight
    assert plan([128256], 256, 4096, 3)[0] == WIDE
    for m in (200, 512):
        assert plan([3072], m, 8192, 3) == (6, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("tile,bm,bn,x,w", [
    (6, 192, 256, 8, 5), (8, 256, 192, 8, 8), (10, 192, 192, 4, 3)])
@torch.no_grad()
def test_short_gradients_gpu(tile, bm, bn, x, w):
    """Stages around those up to which eight waves take a tile, and one more for
    each state of the four waves' rings."""
    from deepspeed_amd.ops import _C
    for steps in (x, *range(x + 1, x + 7)):
        for m, n, k in ((bm + 1, 64 * steps, bn + 8), (700, 64 * steps, 2 * bn)):
            _, ws, _ = _inputs(1, (n,), k, steps)
            dys = [_inputs(m, (), n, n)[0]]
            want = dys[0].double() @ ws[0].double()
            err = (_C.tile_linear_dx(dys, ws, tile, 1).double() - want).abs()
            assert (err <= _limit(want, n)).all()
    for steps in (w, *range(w + 1, w + 4)):
        for k in (12288, 12296, 16384):
            m = 64 * steps - 3
            i, _, _ = _inputs(m, (), k, steps)
            d = _inputs(m, (), bm + 8, steps)[0]
            want = d.double().t() @ i.double()
            err = (_C.tile_linear_dw(i, [d], tile, 1)[0].double() - want).abs()
            assert (err <= _limit(want, m)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,ns,k,mode,tile", [
    (40, (20000,), 2048, 0, 0), (33, (9000, 9000), 4096, SWIGLU, 1),
    (100, (8200, 4100), 2048, 0, 3), (190, (16396,), 4096, 0, 6),
    (128, (8196,), 8192, 0, 3), (129, (8196,), 8192, 0, 6)])
@torch.no_grad()
def test_one_tile_of_rows_gpu(m, ns, k, mode, tile):
    """Rows of whole multiples of 4 KB: every workgroup begins elsewhere in them,
    and comes to all of them; up to 2 MB of x, and past them."""
    from deepspeed_amd.ops import _C
    x, ws, bs = _inputs(m, ns, k, m)
    for y, want in zip(_C.tile_linear(x, ws, bs, mode, tile, 1),
                       _want(x, ws, bs, mode)):
        _close(y, want)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, SWIGLU])
@pytest.mark.parametrize("tile", [1, 2, 4, 5, 7, 8, 9, 10, 11])
@torch.no_grad()
def test_weights_past_the_caches_gpu(tile, mode):
    """One tile of rows over 16 MB of W and a bit less: W's loads are another
    kind. A last tile of 4 features, gate and up ends in the wave's half."""
    from deepspeed_amd.ops import _C
    m = {1: 64, 2: 127, 4: 128, 5: 191, 10: 190}.get(tile, 255)
    if (tile == 8 and mode) or (tile == 11 and not mode):
        return      # no such kernels
    for k in (704, 640):
        ns = (6148, 6148) if mode else (8196, 3844)
        assert (sum(ns) * k >= 1 << 23) == (k == 704)
        x, ws, bs = _inputs(m, ns, k, m)
        for y, want in zip(_C.tile_linear(x, ws, bs, mode, tile, 1),
                           _want(x, ws, bs, mode)):
            _close(y, want)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [-1, 0, 1, None])
def test_square_tile_gpu(rows, monkeypatch):
    """192 x 192, as the tiles before it."""
    monkeypatch.setitem(globals(), "TILES", TILES + [(192, 192, 3)])
    if rows is None:
        test_every_tile_backward_gpu(len(TILES) - 1)
    else:
        test_every_tile_gpu(len(TILES) - 1, rows)


def test_short_contractions():
    """256 x 256 by eight waves where the contraction, or a part of it, is short."""
    ext = get_ext()
    if ext is None:
        pytest.skip("the plan is the extension's")
    plan = ext.tile_linear_plan
    eight = len(TILES) + 1
    assert plan([14336] * 2, 8192, 1536, SWIGLU)[0] == eight
    assert plan([14336] * 2, 8192, 1600, SWIGLU)[0] == WIDE
    assert plan([1024], 8192, 14336, 2)[0] == eight
    assert plan([512, 576], 8192, 14336, 2)[0] == WIDE
    assert plan([14336], 768, 14336, 3)[0] == eight
    assert plan([14336], 769, 14336, 3)[0] == WIDE
    assert plan([14336], 8192, 512, 0)[0] != eight
    for k in (2560, 4096, 8192):      # few columns, and powers of two
        assert plan([32000], 768, k, 3)[0] == WIDE


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [SWIGLU, 2])
def test_short_contractions_gpu(mode, monkeypatch):
    """256 x 256 by eight waves, as the tiles before it."""
    from deepspeed_amd.ops import _C
    eight = len(TILES) + 1
    monkeypatch.setitem(globals(), "TILES",
                        TILES + [(192, 192, 3), (256, 256, 2)])
    if mode != SWIGLU:
        return test_every_tile_backward_gpu(eight)
    for rows in (-1, 0, 1):
        for n in (132, 256):
            for steps in (2, 3, 7):
                x, ws, bs = _inputs(256 + rows, (n, n), 64 * steps, steps)
                _close(_C.tile_linear(x, ws, bs, SWIGLU, eight, 1)[0],
                       _want(x, ws, bs, SWIGLU)[0])
    with pytest.raises(RuntimeError):
        _C.tile_linear(x, ws, bs, 0, eight, 1)


@pytest.mark.gpu
def test_what_lies_past_the_last_row_gpu():
    """Rows past the end count for nothing, whatever the last one holds: each
    value of the weight's gradient comes from its own column."""
    from deepspeed_amd.ops import _C
    x, _, _ = _inputs(257, (), 256, 0)
    dy, _, _ = _inputs(257, (), 264, 1)
    x[-1, 5] = float("inf")
    dy[-1, 7] = 0.0
    got, = _C.tile_linear_dw(x, [dy])
    want = dy.double().t() @ x.double()
    finite = want.isfinite()
    assert torch.equal(finite, got.isfinite())
    assert torch.equal(want.isnan(), got.isnan())
    err = (got.double() - want)[finite].abs()
    assert (err <= _limit(want[finite], 257)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [40, 250, 1000, 2600])
@pytest.mark.parametrize("ns,k", [((512, 128, 128), 256), ((1000, 1000), 264),
                                  ((640,), 512)])
@pytest.mark.parametrize("frozen", [None, "input", 0])
def test_training_layers_gpu(m, ns, k, frozen):
    x, ws, bs = _inputs(m, ns, k, m)
    mods = []
    for w, b in zip(ws, bs):
        lin = Linear(k, len(w), bias=b is not None, device="cuda",
                     dtype=torch.bfloat16)
        with torch.no_grad():
            lin.weight.copy_(w)
            if b is not None:
                lin.bias.copy_(b)
        mods.append(lin)
    if frozen == 0:
        mods[0].weight.requires_grad_(False)
    x = x.view(2, m // 2, k).requires_grad_(frozen != "input")
    ys = tile_linear(x, mods) or [call(lin, x) for lin in mods]
    dys = [torch.randn_like(y) for y in ys]
    torch.autograd.backward(ys, dys)
    x2 = x.detach().reshape(-1, k).double()
    d2 = [d.reshape(-1, d.shape[-1]).double() for d in dys]
    for y, want in zip(ys, _want(x2, ws, bs, 0)):
        _close(y.detach().reshape(want.shape), want)
    if frozen != "input":
        want = sum(d @ w.double() for d, w in zip(d2, ws))
        got = x.grad.view(-1, k).double()
        # layers whose parts are added up outside are rounded one by one
        parts = sum((d @ w.double()).abs() for d, w in zip(d2, ws))
        assert ((got - want).abs() <= 2.0 ** -7 * parts
                + _limit(want, sum(ns))).all()
    for i, (lin, d) in enumerate(zip(mods, d2)):
        if frozen == i:
            assert lin.weight.grad is None
        else:
            want = d.t() @ x2
            err = (lin.weight.grad.double() - want).abs()
            assert (err <= _limit(want, m)).all()
        if lin.bias is not None:
            torch.testing.assert_close(lin.bias.grad.double(), d.sum(0),
                                       rtol=2.0 ** -7, atol=0.05)


@pytest.mark.gpu
def test_training_layers_watched_gpu():
    """Hooks, dispatch modes, batched and twice differentiated gradients go
    through torch's own products."""
    from torch.utils.flop_counter import FlopCounterMode
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(300, 256, device="cuda", generator=g).bfloat16()
    x.requires_grad_()
    mods = [Linear(256, 256, bias=False, device="cuda", dtype=torch.bfloat16)
            for _ in range(2)]
    a, b = tile_linear(x, mods)
    with FlopCounterMode(display=False) as mode:
        (a * b).sum().backward(retain_graph=True)
    assert mode.get_total_flops() == 4 * 2 * 300 * 256 * 256
    gx, = torch.autograd.grad((a.float() * b.float()).sum(), x,
                              create_graph=True)
    gx.float().sum().backward(retain_graph=True)
    v = torch.randn(3, 300, 256, device="cuda", generator=g).bfloat16()
    many, = torch.autograd.grad(a, x, v, is_grads_batched=True,
                                retain_graph=True)
    for got, d in zip(many, v):
        one, = torch.autograd.grad(a, x, d, retain_graph=True)
        assert (got.float() - one.float()).norm() <= 0.01 * one.float().norm()
    h = mods[0].register_forward_hook(lambda *a: None)
    assert tile_linear(x, mods) is None
    h.remove()
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: seen.append(t.shape) or t, lambda t: t):
        tile_linear(x, mods)
    assert seen == [x.shape, mods[0].weight.shape, mods[1].weight.shape]


def test_own_products():
    assert L.own_products(4000, 3072, 3072) == (True, True)
    assert L.own_products(8192, 14336, 4096) == (False, True)
    assert L.own_products(8192, 128256, 4096) == (False, False)
    assert L.own_products(1000, 1000, 512) == (False, True)
    assert L.own_products(1000, 1024, 516) == (False, False)
    assert L.own_products(32, 1024, 512) == (False, False)


def test_own_dx():
    """The input's gradient of many rows is the library's where that is ahead."""
    def one(t, n, k):
        return L.own_dx(t, (n,), k)
    assert one(2559, 128256, 4096) and not one(2560, 128256, 4096)
    assert one(4096, 4096, 4096) and not one(8192, 4096, 4096)
    assert one(2700, 3072, 8192) and not one(32768, 8192, 3072)
    assert one(5000, 32000, 1024) and not one(8192, 32000, 1024)
    assert one(32768, 1024, 1024)
    # several at once save the additions
    assert L.own_dx(32768, (4096, 1024, 1024), 4096)
    assert L.own_dx(32768, (3072,) * 3, 3072)
    assert L.own_dx(4096, (8192,) * 2, 3072)
    assert not L.own_dx(6000, (8192,) * 2, 3072)
    assert not L.own_dx(2560, (14336,) * 2, 4096)
    # what the kernel does not take
    for t, ns, k in ((32, (256,), 64), (1 << 30, (256,), 64), (64, (128,), 64),
                     (64, (256, 224), 64), (64, (256,), 68)):
        assert not L.own_dx(t, ns, k)


def test_own_forward():
    own = L.own_forward
    assert own(2559, (128256,), 4096) and not own(2560, (128256,), 4096)
    # long contractions, but for whole rounds of tiles
    assert own(8192, (3584,), 18944) and own(2560, (5120,), 16384)
    assert not own(8192, (4096,), 16384) and not own(2560, (8192,), 28672)
    assert own(2559, (4096,), 16384)
    # several layers
    assert own(12288, (4096, 1024, 1024), 4096)
    assert not own(16384, (4096, 1024, 1024), 4096)
    assert own(32768, (1024, 256, 256), 1024)
    assert not own(4096, (8192, 1024, 1024), 8192)
    assert own(32768, (14336, 14336), 4096, SWIGLU)
    for t, ns, k in ((32, (64,), 256), (64, (62,), 256), (64, (64,), 224),
                     (64, (64,), 128), (64, (64,), L.INPUTS + 64)):
        assert not own(t, ns, k) and not own(t, ns * 2, k, SWIGLU)


@pytest.mark.parametrize("own,other", [
    # whole tiles of rows, and one row more
    ((4097, (4096,), 4096), (4096, (4096,), 4096)),
    ((4097, (8192, 8192), 8192), (4096, (8192, 8192), 8192)),
    ((16385, (4096,) * 3, 4096), (16384, (4096,) * 3, 4096)),
    # whole rounds of tiles and contractions that are not short
    ((4096, (3840,), 4096), (4096, (4096,), 4096)),
    ((4096, (4096,), 3008), (4096, (4096,), 3072)),
    # long contractions: features in 4096s
    ((4096, (24640,), 16384), (4096, (24576,), 16384)),
    ((4097, (12288,), 16384), (4096, (12288,), 16384)),
    ((4097, (12288,), 16384), (4097, (16384,), 16384)),
    ((3840, (4096,), 16384), (4096, (4096,), 16384)),
    ((3840, (4096,), 16384), (3840, (8192,), 16384)),
    # vocabularies
    ((4096, (65280,), 4096), (4096, (65536,), 4096)),
    # the largest of several, their rows and their products
    ((4096, (8128, 8128), 8192), (4096, (8192, 8192), 8192)),
    ((16128, (4096,) * 3, 4096), (16384, (4096,) * 3, 4096)),
    ((16384, (2048,) * 2, 4096), (16384, (4096,) * 2, 4096)),
])
def test_lines_of_forward(own, other):
    assert L.own_forward(*own) and not L.own_forward(*other)


@pytest.mark.parametrize("own,other", [
    # whole tiles of rows, and one row more
    ((8193, (14336,), 4096), (8192, (14336,), 4096)),
    ((8193, (14336,) * 2, 4096), (8192, (14336,) * 2, 4096)),
    # a bit more than a round of tiles, but for many features
    ((8160, (14336,), 2048), (8200, (14336,), 2048)),
    ((12700, (14336,), 2048), (12500, (14336,), 2048)),
    ((10000, (28672,), 2048), (10000, (28608,), 2048)),
    ((8160, (11008,) * 2, 2048), (10000, (11008,) * 2, 2048)),
])
def test_lines_of_dx(own, other):
    assert L.own_dx(*own) and not L.own_dx(*other)


def test_lines_of_dw():
    """The library's: vocabularies over many whole tiles of rows."""
    assert L.own_dw(8193, 128256, 4096) and not L.own_dw(8192, 128256, 4096)
    assert L.own_dw(5888, 65536, 4096) and not L.own_dw(6144, 65536, 4096)
    assert L.own_dw(6144, 65528, 8192) and not L.own_dw(32768, 65536, 8192)
    assert L.own_dw(32768, 128256, 2048)


def test_both_copies_of_forward():
    """A serving step's native layer and the modules make the same products."""
    ext = get_ext()
    if ext is None:
        pytest.skip("the copy is the extension's")
    rows = [33, 2559, 2560, 2561, 3840, 4095, 4096, 8192, 16128, 16383, 16384,
            16385, 32768, 100000]
    widths = [4, 256, 1024, 3072, 4096, 4100, 8192, 12288, 16384, 28672, 65280,
              65532, 65536, 128256]
    inputs = [192, 1024, 3008, 3072, 4096, 8192, 16320, 16384, 28672, 1 << 22]
    seen = set()
    for t in rows:
        for n in widths:
            for ns in ((n,), (n, n), (n, 1024, 1024), (n,) * 3):
                for k in inputs:
                    for mode in (0, 1) if len(ns) == 2 else (0,):
                        want = L.own_forward(t, ns, k, mode)
                        assert ext.own_forward(t, ns, k, mode) == want, (t, ns, k)
                        seen.add((len(ns), want))
    assert len(seen) == 6


@pytest.mark.parametrize("t,ns,k,want", [
    (12288, (4096, 1024, 1024), 4096, [3]),
    (14000, (4096, 1024, 1024), 4096, [1, 1, 1]),
    (32768, (4096, 1536, 1536), 4096, [3]),
    (16384, (3072, 3072, 3072), 2048, [1, 1, 1]),
    (32768, (1024, 256, 256), 1024, [3]),
    (32768, (4096,), 4096, [1])])
def test_launches_of_weight_gradients(t, ns, k, want, monkeypatch):
    """Each gradient arrives at its own weight, in one launch or in several."""
    calls = []

    class Ext:
        @staticmethod
        def tile_linear_dw(x, dys, into):
            calls.append(len(dys))
            assert len(into) == len(dys)
            return [(dy.shape[1], out) for dy, out in zip(dys, into)]

    class Slot:
        def __init__(self, n):
            self.take = lambda: n

    monkeypatch.setattr(L, "get_ext", Ext)
    x = torch.empty(t, k, device="meta", dtype=torch.bfloat16)
    dys = [torch.empty(t, n, device="meta", dtype=torch.bfloat16) for n in ns]
    slots = [None if i == 1 else Slot(i) for i in range(len(ns))]
    assert L._dw(x, dys, True, slots) == [
        (n, None if i == 1 else i) for i, n in enumerate(ns)]
    assert calls == want


@pytest.mark.parametrize("used", [(0,), (2,), (0, 2), ()])
def test_unused_outputs_have_no_gradients(used):
    g = torch.Generator().manual_seed(0)
    mods = [nn.Linear(8, n) for n in (4, 6, 2)]
    x = torch.randn(3, 5, 8, generator=g).requires_grad_()
    ys = L._Linears.apply(x, False, *(p for m in mods
                                      for p in (m.weight, m.bias)))
    if not used:
        # nothing but a gradient of None arrives
        class Off(torch.autograd.Function):
            forward = staticmethod(lambda ctx, *ys: ys[0].detach().sum())
            backward = staticmethod(lambda ctx, g: (None,) * 3)
        Off.apply(*ys).backward()
    else:
        sum(ys[i].square().sum() for i in used).backward()
    got = [x.grad] + [p.grad for m in mods for p in (m.weight, m.bias)]
    x.grad = None
    for m in mods:
        m.zero_grad()
    if used:
        sum(mods[i](x).square().sum() for i in used).backward()
    want = [x.grad] + [p.grad for m in mods for p in (m.weight, m.bias)]
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            torch.testing.assert_close(a, b)


def test_largest_layers():
    """Past what a lane's 32 bits of offset reach the library has the products."""
    for n, k in ((L.FEATURES, 64), (64, L.INPUTS)):
        # the last of 256 rows, or of the 64 of a stage across the contraction
        assert 255 * 2 * max(n, k) + 128 < 2 ** 32
        assert any(L.own_products(256, n, k))
    assert L.own_products(256, L.FEATURES + 64, 64) == (False, False)
    assert L.own_products(256, 64, L.INPUTS + 64) == (False, False)
    assert L.own_products((1 << 30) - 1, 8, 8) == (False, True)
    assert L.own_products(1 << 30, 8, 8) == (False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [L.FEATURES, L.FEATURES + 64, 9_000_000])
def test_largest_layers_gpu(n):
    """Every row's gradient of the input from its own row of the output's."""
    from deepspeed_amd.ops import _C
    m, k = 256, 64
    lin = Linear(k, n, bias=False, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(m, k, device="cuda").bfloat16().requires_grad_()
    y = lin(x)
    assert ("_Linears" in type(y.grad_fn).__name__) == (n <= L.FEATURES)
    at = torch.arange(m, device="cuda") * 33203 % n
    dy = torch.zeros_like(y)
    dy[torch.arange(m, device="cuda"), at] = 1.0
    y.backward(dy)
    assert torch.equal(x.grad, lin.weight.detach()[at])
    assert torch.equal(lin.weight.grad[at], x.detach())
    if n > L.FEATURES:
        for call in (lambda: _C.tile_linear_dx([dy], [lin.weight.detach()]),
                     lambda: _C.tile_linear_dw(x.detach(), [dy])):
            with pytest.raises(RuntimeError, match="operands"):
                call()


@pytest.mark.gpu
@pytest.mark.parametrize("tile,bm,bn", [(6, 192, 256), (8, 256, 192),
                                        (10, 192, 192), (9, 256, 256)])
@torch.no_grad()
def test_rows_of_parts_of_lines_gpu(tile, bm, bn):
    """Gradients whose rows are whole 64 bytes or not, to the last column, either
    side of the stages up to which eight waves take these."""
    from deepspeed_amd.ops import _C
    for steps in (12, 13, 14):
        for k in (bn + 8, bn + 32, 2 * bn - 8, 2 * bn):
            n, m = 64 * steps, 64 * steps - 3
            _, ws, _ = _inputs(1, (n,), k, steps)
            dys = [_inputs(bm + 1, (), n, n)[0]]
            want = dys[0].double() @ ws[0].double()
            err = (_C.tile_linear_dx(dys, ws, tile, 1).double() - want).abs()
            assert (err <= _limit(want, n)).all()
            i, _, _ = _inputs(m, (), k, steps)
            d = _inputs(m, (), bm + 8, steps)[0]
            want = d.double().t() @ i.double()
            err = (_C.tile_linear_dw(i, [d], tile, 1)[0].double() - want).abs()
            assert (err <= _limit(want, m)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile,bm,bn", [(6, 192, 256), (8, 256, 192),
                                        (10, 192, 192), (9, 256, 256)])
@pytest.mark.parametrize("biased", [False, True])
@torch.no_grad()
def test_outputs_of_parts_of_lines_gpu(tile, bm, bn, biased):
    """Forward rows that are whole 64 bytes or not, to the last feature, and outputs
    that no cache holds."""
    from deepspeed_amd.ops import _C
    for m, n, k in ((bm + 1, bn + 4, 192), (2 * bm, 2 * bn - 8, 256),
                    (bm + 70, bn + 32, 320), (8300, 16200, 192)):
        x, ws, bs = _inputs(m, (n,), k, n)
        bs = bs if biased else [None]
        got = _C.tile_linear(x, ws, bs, 0, tile, 1)[0]
        rows = torch.cat([torch.arange(64), torch.arange(m - 64, m)]).cuda()
        _close(got[rows], _want(x[rows], ws, bs, 0)[0])
