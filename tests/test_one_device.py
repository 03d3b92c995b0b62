"""Extension calls whose tensors lie on different devices are refused with a
message, by the shared check that also names the devices; the CPU and the meta
device stand for two GPUs."""

import pytest
import torch

from deepspeed_amd.ops._loader import get_ext

pytestmark = pytest.mark.skipif(get_ext() is None, reason="extension not built")
BF16, F32, I32 = torch.bfloat16, torch.float32, torch.int32


def _t(shape, dtype=BF16):
    return torch.zeros(shape, dtype=dtype)


Q, KV = _t((2, 4, 128)), _t((2, 2, 128))
POOL, TABLE = _t((3, 2, 64, 128)), _t((9, 64), F32)
QF, KF = _t((1, 8, 4, 64)), _t((1, 8, 2, 64))

# name, arguments, and which of them are tensors (or lists) to move
CALLS = [
    ("rows_linear", (_t((2, 256)), [_t((16, 256))], [], [_t(16)], 0, 0),
     (0, 1, 3)),
    ("rows_linear", (_t((2, 256)), [_t(4096, torch.int8)], [_t(16, F32)],
                     [None], 256, 0), (0, 1, 2)),
    ("flash_attn_fwd", (QF, KF, KF, 0.1, True, True), (0, 1, 2)),
    ("flash_attn_bwd", (QF, KF, KF, QF, QF, _t((1, 4, 8), F32), 0.1, True, 1),
     (0, 1, 2, 3, 4, 5)),
    ("paged_decode", (Q, POOL, POOL, _t((2, 1), I32), _t(2, I32), 1, 0.1),
     (0, 1, 2, 3, 4)),
    ("paged_rows", (Q, POOL, POOL, _t(99, I32), 1, 1, 1, False, 1, 0.1),
     (0, 1, 2, 3)),
    ("paged_append", (Q, KV, KV, POOL, POOL, _t(2, I32), TABLE, TABLE,
                      _t(2, I32), 1), (0, 1, 2, 3, 4, 5, 6, 7, 8)),
    ("rope", (QF, KF, _t((8, 32), F32), _t((8, 32), F32), _t((1, 8), I32),
              False), (0, 1, 2, 3, 4)),
    ("add_norm_fwd", (_t((2, 64)), _t((2, 64)), _t(64), 1e-5), (0, 1, 2)),
    ("norm_bwd", (_t((2, 64)), _t((2, 64)), _t(64), _t(2, F32), None, False,
                  _t((2, 64))), (0, 1, 2, 3, 6)),
]


@pytest.mark.parametrize("name,args,tensors", CALLS)
def test_other_devices_are_refused(name, args, tensors):
    call = getattr(get_ext(), name)
    for i in tensors:
        a = list(args)
        a[i] = [t.to("meta") for t in a[i]] if isinstance(a[i], list) \
            else a[i].to("meta")
        with pytest.raises(RuntimeError, match="different devices"):
            call(*a)


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
@pytest.mark.gpu
@torch.no_grad()
def test_the_current_device_does_not_matter():
    from deepspeed_amd.ops.linear import rows_linear
    lin = torch.nn.Linear(256, 64, device="cuda:1", dtype=BF16)
    x = torch.randn(2, 256, device="cuda:1").bfloat16()
    y, = rows_linear(x, (lin,))
    assert y.device == x.device
    assert (y - lin(x)).abs().max() < 0.05
