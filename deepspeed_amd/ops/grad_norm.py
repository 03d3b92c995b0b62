"""Global gradient norm over a list of tensors (csrc/grad_norm.hip)."""

import torch

from ._loader import get_ext


def sum_of_squares(tensors) -> torch.Tensor:
    """fp32 scalar tensor: the sum of the squares of all values. bf16 and fp32
    GPU tensors are summed in fp32 by one kernel; others (fp16, whose per-tensor
    norms overflow on purpose: that skips the step) tensor by tensor."""
    t0 = tensors[0]
    if (t0.is_cuda and get_ext() is not None
            and t0.dtype in (torch.bfloat16, torch.float32)
            and all(t.dtype is t0.dtype and t.device == t0.device
                    and t.is_contiguous() for t in tensors)):
        return get_ext().sum_of_squares(tensors)
    norms = torch._foreach_norm(tensors, 2.0)
    return torch.stack([n.float() for n in norms]).pow(2).sum()
