"""ZeRO on one rank: gradients are not copied on their way to the optimizer
(stages 1 and 2 step from the flat gradient buffers, stage 3 takes over whole
gradients). Against the mixed-precision reference loop and each other."""

import pytest
import torch

from .common import run_distributed
from .test_zero12 import _reference_mixed_precision_loop


class Net(torch.nn.Module):
    """Layers without bias (whole units), one used twice, one never."""

    def __init__(self, spare):
        super().__init__()
        torch.manual_seed(3)
        self.a = torch.nn.Linear(64, 64, bias=False)
        self.b = torch.nn.Linear(64, 64)
        self.out = torch.nn.Linear(64, 1, bias=False)
        if spare:
            self.spare = torch.nn.Linear(64, 64, bias=False)

    def forward(self, x, labels=None):
        x = torch.tanh(self.a(torch.tanh(self.b(torch.tanh(self.a(x))))))
        return torch.nn.functional.mse_loss(self.out(x).float(),
                                            labels.float())


def _data(n):
    g = torch.Generator().manual_seed(0)
    return [(torch.randn(4, 64, generator=g), torch.randn(4, 1, generator=g))
            for _ in range(n)]


def _masters(stage, gas, spare, steps):
    import deepspeed_amd
    engine, opt, _, _ = deepspeed_amd.initialize(model=Net(spare), config={
        "train_micro_batch_size_per_gpu": 4,
        "gradient_accumulation_steps": gas,
        "bf16": {"enabled": True}, "gradient_clipping": 0.5,
        "zero_optimization": {"stage": stage,
                              "stage3_param_persistence_threshold": 0},
        "optimizer": {"type": "AdamW", "params": {"lr": 1e-2}}})
    for x, y in _data(steps * gas):
        loss = engine(x.bfloat16(), labels=y)
        engine.backward(loss)
        engine.step()
    out = {}
    for part in opt.layout_manifest():
        flat = opt.param_groups[part["group_idx"]]["params"][0].data
        for name, off, n, shape in part["params"]:
            lo = part["master_offset"] + off
            out[name] = flat[lo:lo + n].view(shape).clone()
    return out


def _check(rank, world, gas):
    _, ref = _reference_mixed_precision_loop(
        Net(False), _data(3 * gas), 1e-2, 3, gas, torch.bfloat16, 0.5)
    ref = dict(ref.named_parameters())
    began = dict(Net(True).bfloat16().float().named_parameters())

    def close(a, b, name):
        # bf16 gradients added up in another order: a few turn the sign of
        # Adam's first updates, the rest of the way is the same
        way = (b - began[name]).detach().norm()
        assert (way == 0) == (name == "spare.weight"), name
        assert (a - b).detach().norm() <= 0.05 * way, name

    for stage in (1, 2, 3):
        got = _masters(stage, gas, False, 3)
        for n, p in ref.items():
            close(got[n], p, n)
    two, three = (_masters(s, gas, True, 3) for s in (2, 3))
    for n in two:
        close(two[n], three[n], n)


@pytest.mark.parametrize("gas", [1, 2])
def test_one_rank_matches_reference(gas):
    run_distributed(_check, 1, "gloo", (gas,))
