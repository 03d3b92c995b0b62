"""Fused Adam over flat shards of every alignment and remainder."""

import pytest
import torch

pytestmark = pytest.mark.gpu


LARGE = (1 << 25) + 5     # past the caches: the nontemporal kernel


@pytest.mark.parametrize("n,offset", [
    (n, offset) for n in (1, 3, 4, 5, 1023, 2048, 2053)
    for offset in (0, 1, 2)] + [(LARGE, 0), (LARGE, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16,
                                   torch.float32])
@pytest.mark.parametrize("adamw", [True, False])
def test_adam_flat(n, offset, dtype, adamw):
    from deepspeed_amd.ops import _C
    torch.manual_seed(n)

    def buf(dt):
        return torch.randn(n + offset, device="cuda").to(dt)[offset:]

    p, m, g = buf(torch.float32), buf(torch.float32), buf(dtype)
    v = buf(torch.float32).square_()
    p16 = torch.empty(n + offset, device="cuda",
                      dtype=torch.bfloat16)[offset:]
    pd, md, vd = p.double(), m.double(), v.double()
    gd = g.double() * 0.5
    if not adamw:
        gd = gd + 0.1 * pd
    md = 0.9 * md + 0.1 * gd
    vd = 0.95 * vd + 0.05 * gd * gd
    up = md / (1 - 0.9 ** 3) / ((vd / (1 - 0.95 ** 3)).sqrt() + 1e-8)
    if adamw:
        up = up + 0.1 * pd
    pd = pd - 0.01 * up
    _C.fused_adam_flat(p, g, m, v, p16, 0.01, 0.9, 0.95, 1e-8, 0.1, 3, 0.5,
                       adamw)
    # a dozen fp32 operations, of which sums may cancel: by the size of their
    # terms, of which the update can be the largest
    for a, b, terms in ((p, pd, 0.01 * up.abs() + pd.abs() + 1),
                        (m, md, md.abs() + gd.abs() + 1), (v, vd, vd + 1)):
        assert ((a.double() - b).abs() <= 4e-6 * terms).all()
    assert torch.equal(p16, p.bfloat16())
    q = p.clone()
    _C.fused_adam_flat(p, g, m, v, None, 0.01, 0.9, 0.95, 1e-8, 0.1, 4, 0.5,
                       adamw)
    assert not torch.equal(p, q)
