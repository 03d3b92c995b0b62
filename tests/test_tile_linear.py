"""Linear layers of many rows: which calls take the kernel (CPU) and every tile
of the kernel against fp64 products (GPU)."""

import pytest
import torch
import torch.nn as nn

from deepspeed_amd.ops.linear import SWIGLU, Linear, tile_linear

# rows, features and stages of the tiles, in the kernel's order
TILES = [(64, 64, 8), (64, 128, 6), (128, 64, 6), (128, 128, 5), (128, 256, 3),
         (192, 128, 4), (192, 256, 2), (256, 128, 3), (256, 192, 2),
         (256, 256, 2)]


def test_calls_left_alone():
    lin = Linear(256, 16).bfloat16()
    x = torch.randn(40, 256).bfloat16()
    with torch.no_grad():
        assert tile_linear(x, (lin,)) is None      # on the CPU
    assert tile_linear(x, (lin,)) is None          # with gradients


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
