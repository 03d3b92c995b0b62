"""Gated activations and int8 dequantization over every alignment and
remainder, against the same operations in fp32."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [1, 7, 8, 2049, 1_000_003])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("act", [0, 1])
def test_gated_act(dtype, n, offset, act):
    from deepspeed_amd.ops import _C
    torch.manual_seed(n)
    g, u, d = (torch.randn(n + offset, device="cuda").to(dtype)[offset:]
               for _ in range(3))
    gf, uf = (t.double().requires_grad_() for t in (g, u))
    a = torch.nn.functional.silu(gf) if act == 0 else \
        torch.nn.functional.gelu(gf, approximate="tanh")
    want = a * uf
    want.backward(d.double())
    tol = dict(rtol=2 * torch.finfo(dtype).eps, atol=2e-6)
    torch.testing.assert_close(_C.gated_act_fwd(g, u, act).double(),
                               want.detach(), **tol)
    dg, du = _C.gated_act_bwd(d, g, u, act)
    torch.testing.assert_close(dg.double(), gf.grad, **tol)
    torch.testing.assert_close(du.double(), uf.grad, **tol)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [1, 15, 16, 2048, 5000, 100_017])
@pytest.mark.parametrize("group", [16, 100, 2048])
@pytest.mark.parametrize("bits", [4, 8])
def test_dequantize(dtype, n, group, bits):
    from deepspeed_amd.ops.quantizer import (_torch_dequantize, dequantize,
                                             quantize)
    torch.manual_seed(n)
    x = torch.randn(n, device="cuda")
    q, s = quantize(x, group, bits)
    for off in (0, 1):
        at = torch.empty(q.numel() + off, dtype=q.dtype,
                         device="cuda")[off:].copy_(q)
        # The compiler may round the product once, to 16 bits, where torch
        # rounds it to 32 bits first: one unit in the last place apart.
        ulp = 0 if dtype == torch.float32 else torch.finfo(dtype).eps
        torch.testing.assert_close(
            dequantize(at, s, n, group, bits, dtype),
            _torch_dequantize(q, s, n, group, bits, dtype), rtol=ulp,
            atol=0 if dtype != torch.float16 else 2.0**-24)
