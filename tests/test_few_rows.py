"""Linear layers of up to 16 rows where chunks of inputs end unevenly among the
waves, features in a tile, and scales past what is kept in LDS, against fp64."""

import pytest
import torch

from deepspeed_amd.ops.linear import SWIGLU, rows_linear
from tests.test_rows_linear import _close, _layer


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("k", [256, 768, 1280, 2048, 2304, 4352, 65536, 65792])
@pytest.mark.parametrize("m", [1, 5, 16])
@torch.no_grad()
def test_few_rows_gpu(int8, k, m):
    g = torch.Generator().manual_seed(k + m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    # one tile a wave and two, gate and up
    for ns, mode in (((17,), 0), ((6145, 3, 16), 0), ((33, 33), SWIGLU)):
        if k > 5000 and ns[0] > 1000:
            ns = (33, 3)
        both = [_layer(n, k, i == 0, int8, g) for i, n in enumerate(ns)]
        got = rows_linear(x, [b[0] for b in both], mode)
        want = [f(x) for _, f in both]
        if mode == SWIGLU:
            want = [torch.nn.functional.silu(want[0]) * want[1]]
        for y, w in zip(got, want):
            _close(y, w)


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("n,k", [(6144, 4096), (8192, 4352), (9216, 1024),
                                 (9216, 4096), (32000, 256), (33000, 512)])
@pytest.mark.parametrize("m", [1, 8, 9])
@torch.no_grad()
def test_tiles_a_wave_gpu(int8, n, k, m):
    """One and two tiles on either side of their lines, with chunks that are a
    wave's whole parts and others."""
    g = torch.Generator().manual_seed(m)
    lin, want = _layer(n, k, False, int8, g)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    _close(rows_linear(x, (lin,))[0], want(x))


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("k", [2048, 3072, 4096])
@pytest.mark.parametrize("m", [1, 5, 16])
@torch.no_grad()
def test_workgroups_go_on_gpu(int8, k, m):
    """More tiles than CUs: one that begins the second round, rounds that end in
    part and whole, the last tile in part, and layers that end inside a tile."""
    g = torch.Generator().manual_seed(k + m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    for ns, mode in (((4100,), 0), ((8196,), 0), ((16384,), 0),
                     ((8200, 4100, 5000), 0), ((4100, 4100), SWIGLU),
                     ((8200, 8200), SWIGLU), ((8192, 8192), SWIGLU)):
        both = [_layer(n, k, i == 0, int8, g) for i, n in enumerate(ns)]
        got = rows_linear(x, [b[0] for b in both], mode)
        want = [f(x) for _, f in both]
        if mode == SWIGLU:
            want = [torch.nn.functional.silu(want[0]) * want[1]]
        for y, w in zip(got, want):
            _close(y, w)


@pytest.mark.gpu
@pytest.mark.parametrize("ns,k", [((1024,), 1024), ((4096, 1024, 1024), 1792),
                                  ((4096, 1024, 1028), 1792), ((512,), 2048),
                                  ((130, 64), 256)])
@pytest.mark.parametrize("m", [16, 17, 32])
@torch.no_grad()
def test_small_layers_of_up_to_32_rows_gpu(ns, k, m):
    g = torch.Generator().manual_seed(m)
    both = [_layer(n, k, i == 0, False, g) for i, n in enumerate(ns)]
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    for y, (_, want) in zip(rows_linear(x, [b[0] for b in both]), both):
        _close(y, want(x))


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("k", [256, 1792, 2304, 4352])
@pytest.mark.parametrize("m", [4, 8, 17, 24, 32])
@torch.no_grad()
def test_streams_gpu(int8, k, m):
    """Every number of tiles and waves: rings that are not filled once, waves
    without a chunk, tiles that end in part and several to a workgroup, with the
    bias of each layer."""
    g = torch.Generator().manual_seed(k + m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    for ns, mode in (((4096,), 0), ((4100, 1030, 20), 0), ((8190,), 0),
                     ((16500, 36), 0), ((4100, 4100), SWIGLU),
                     ((12300, 12300), SWIGLU)):
        both = [_layer(n, k, True, int8, g) for n in ns]
        got = rows_linear(x, [b[0] for b in both], mode)
        want = [f(x) for _, f in both]
        if mode == SWIGLU:
            want = [torch.nn.functional.silu(want[0]) * want[1]]
        for y, w in zip(got, want):
            _close(y, w)


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("m", [3, 20])
@torch.no_grad()
def test_past_the_streams_gpu(int8, m):
    """More inputs than a lane's offsets are for: the kernel that takes its operands
    straight to registers."""
    k = (1 << 22) + 256
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    for ns, mode in (((20, 4), 0), ((17, 17), SWIGLU)):
        both = [_layer(n, k, i == 0, int8, g) for i, n in enumerate(ns)]
        got = rows_linear(x, [b[0] for b in both], mode)
        want = [f(x) for _, f in both]
        if mode == SWIGLU:
            want = [torch.nn.functional.silu(want[0]) * want[1]]
        for y, w in zip(got, want):
            # fp32 sums of k / 8 terms a wave, two roundings with the gate
            lim = 2.0 ** (-7 if mode else -8) * w.abs() + 2.0 ** -12 * w.abs().max()
            assert ((y.double() - w).abs() <= lim).all()


@pytest.mark.gpu
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("k", [256, 512, 768])
@pytest.mark.parametrize("m", [1, 16, 17, 24, 25, 32])
@torch.no_grad()
def test_brief_layers_gpu(int8, k, m):
    """A tile less than a round and a whole one, either side of the rows and inputs up
    to which they go straight to registers; several layers, and of heads."""
    g = torch.Generator().manual_seed(k + m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    for ns in ((4068,), (4084,), (2000, 36, 4), (256, 128, 128)):
        both = [_layer(n, k, i == 0, int8, g) for i, n in enumerate(ns)]
        for y, (_, want) in zip(rows_linear(x, [b[0] for b in both]), both):
            _close(y, want(x))
