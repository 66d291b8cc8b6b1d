"""Which backward passes run the gradient Functions' forwards directly: only those that nothing looks into."""
import pytest
import torch
from torch.autograd import forward_ad

from sparseforge_amd.linear import apply_in_backward


class _Twice(torch.autograd.Function):
    """Has neither a jvp nor a vmap rule, like the package's gradient Functions: apply refuses both."""

    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return x * 2

    @staticmethod
    def backward(ctx, g):
        return g * 2


def test_plain_pass_and_create_graph():
    x = torch.ones(3, requires_grad=True)
    with torch.no_grad():
        y = apply_in_backward(_Twice, x)
    assert not y.requires_grad and torch.equal(y, torch.full((3,), 2.0))
    y = apply_in_backward(_Twice, x)
    assert type(y.grad_fn).__name__ == "_TwiceBackward"


def test_forward_mode_is_refused_not_dropped():
    with torch.no_grad(), forward_ad.dual_level():
        x = forward_ad.make_dual(torch.ones(3), torch.ones(3))
        with pytest.raises(NotImplementedError):
            apply_in_backward(_Twice, x)


def test_vmap_is_refused():
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: apply_in_backward(_Twice, x))(torch.ones(2, 3))
