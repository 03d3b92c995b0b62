"""Sum of squares over lists of gradients."""

import pytest
import torch

from deepspeed_amd.ops.grad_norm import sum_of_squares


def test_cpu_and_fp16():
    ts = [torch.randn(n) for n in (1, 7, 100)]
    want = sum(t.double().square().sum() for t in ts)
    assert abs(sum_of_squares(ts).double() - want) < 1e-5 * want
    big = [torch.full((1000,), 6e4, dtype=torch.float16)]
    assert torch.isinf(sum_of_squares(big))       # as a loss scale expects


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes", [(1,), (7, 0, 9), (32768, 32769, 8),
                                   (5_000_011,), tuple(range(1, 150)),
                                   (70_000_001, 3)])
def test_sum_of_squares_gpu(dtype, sizes):
    torch.manual_seed(0)
    flat = torch.randn(sum(sizes) + 1, device="cuda").to(dtype)[1:]
    ts = list(flat.split(list(sizes)))            # of any alignment
    got = sum_of_squares(ts)
    want = flat.double().square().sum()
    # each thread adds thousands of fp32 terms, rounding like their root
    assert abs(got.double() - want) <= 1e-5 * want
    assert torch.equal(got, sum_of_squares(ts))
    ts[-1][-1] = float("nan")
    assert torch.isnan(sum_of_squares(ts))
