"""The gradient of an embedding's table where blocks of tokens, tables of blocks and
shared rows end, against fp64, and the module where its kernel is not taken."""

import pytest
import torch

from deepspeed_amd.ops.embedding import Embedding, fits


def test_on_the_cpu_and_its_second_derivative():
    torch.manual_seed(0)
    ids = torch.randint(0, 9, (3, 5))
    own, ref = Embedding(9, 8, padding_idx=2), torch.nn.Embedding(9, 8, 2)
    ref.load_state_dict(own.state_dict())
    for m in (own, ref):
        m(ids).square().sum().backward()
    assert torch.equal(own.weight.grad, ref.weight.grad)


def test_places_take_no_more_than_the_gradient():
    for tokens, rows, columns, want in (
            (32768, 152064, 3584, True), (4096, 32000, 1024, True),
            (32768, 10_000_000, 64, False), (32768, 100, 264, True),
            (32768, 100, 256, False), (256, 10, 8, True), (1000, 10, 8, False),
            (32769, 100, 4096, False), (0, 100, 4096, False),
            (8, 1 << 30, 8, False), (8, 100, (1 << 20) + 8, False),
            (8, 100, 12, False)):
        assert fits(tokens, rows, columns) == want, (tokens, rows, columns)
        if want:
            blocks = -(-tokens // 256)
            spans, has = rows * blocks, rows * -(-blocks // 32)
            assert 4 * (spans + has) <= 2 * rows * columns


@pytest.mark.gpu
@pytest.mark.parametrize("t", [1, 255, 256, 257, 1000, 8193, 32768])
@pytest.mark.parametrize("v,h", [(3, 8), (700, 520), (32000, 1024)])
def test_table_gradient_gpu(t, v, h):
    from deepspeed_amd.ops import _C
    g = torch.Generator().manual_seed(t + v)
    ids = torch.randint(0, v, (t,), generator=g).cuda()
    if t > 1000:
        ids[: t // 3] = v // 2          # shared by a workgroup's waves
        ids[100:131], ids[4000:4032] = 0, min(1, v - 1)
    dy = torch.randn(t, h, generator=g).bfloat16().cuda()
    for padding in (-1, v // 2):
        got = _C.embedding_bwd(ids, dy, v, padding)
        into = torch.zeros_like(got)
        assert _C.embedding_bwd(ids, dy, v, padding, into) is not None
        assert torch.equal(got, into)   # in the same order every time
        keep = ids != padding
        want = torch.zeros(v, h, dtype=torch.float64, device="cuda")
        want.index_add_(0, ids[keep], dy[keep].double())
        size = torch.zeros_like(want).index_add_(0, ids[keep],
                                                 dy[keep].double().abs())
        # fp32 sums of up to t terms, rounded once
        err = (got.double() - want).abs()
        assert (err <= 2.0 ** -8 * want.abs() + 2.0 ** -22 * size).all()


@pytest.mark.gpu
def test_module_gpu():
    torch.manual_seed(0)
    ids = torch.randint(0, 50, (2, 33), device="cuda")
    own = Embedding(50, 64, device="cuda", dtype=torch.bfloat16)
    ref = torch.nn.Embedding(50, 64, device="cuda", dtype=torch.bfloat16)
    ref.load_state_dict(own.state_dict())
    grads = []
    for m in (own, ref):
        y = m(ids)
        assert ("_Embed" in type(y.grad_fn).__name__) == (m is own)
        dy = torch.randn_like(y).requires_grad_()
        first, = torch.autograd.grad(y, m.weight, dy, create_graph=True)
        second, = torch.autograd.grad(first.float().square().sum(), dy)
        first2, = torch.autograd.grad(m(ids), m.weight, torch.ones_like(y))
        grads.append((first2, second.shape))
        if m is own:
            grads_dy = dy.detach(), second
        else:
            y = m(ids)
            dy = grads_dy[0].clone().requires_grad_()
            first, = torch.autograd.grad(y, m.weight, dy, create_graph=True)
            second, = torch.autograd.grad(first.float().square().sum(), dy)
            torch.testing.assert_close(second, grads_dy[1], rtol=2.0 ** -6,
                                       atol=1e-2)
    torch.testing.assert_close(grads[0][0], grads[1][0], rtol=2.0 ** -7, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [64, 512])
def test_narrow_tables_are_torchs_gpu(columns):
    ids = torch.randint(0, 300, (32768,), device="cuda")
    own = Embedding(300, columns, device="cuda", dtype=torch.bfloat16)
    y = own(ids)
    assert ("_Embed" in type(y.grad_fn).__name__) == (columns == 512)
    y.backward(torch.ones_like(y))
    want = torch.bincount(ids, minlength=300)[:, None]
    torch.testing.assert_close(own.weight.grad.float(),
                               want.expand(300, columns).float(),
                               rtol=2.0 ** -8, atol=0)
