"""The HuggingFace forward's fused ops carry no derivative: tensors that need
one, in backward or in forward mode, are recognised and take the torch path."""
import torch
from torch.autograd import forward_ad

from fused_turboquant.hf.fused_cache import _needs_grad


def test_needs_grad_sees_both_modes():
    x = torch.zeros(2, 3)
    w = torch.zeros(2, 3, requires_grad=True)
    assert not _needs_grad(x, x)
    assert _needs_grad(x, w)
    with torch.no_grad():
        assert not _needs_grad(x, w)
    with forward_ad.dual_level():
        assert not _needs_grad(x)
        dual = forward_ad.make_dual(x, torch.ones_like(x))
        assert _needs_grad(x, dual)
        with torch.no_grad():
            assert _needs_grad(dual)
