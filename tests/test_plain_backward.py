"""Which backward passes run the gradient Functions' forwards directly: only those that nothing looks into; and that
the package's gradient Functions can be run so."""
import ast
import inspect
import textwrap

import pytest
import torch
from torch.autograd import forward_ad

from sparseforge_amd import distill, linear, llama
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


GRADIENTS = [linear._MaskedLinearBackward, distill._KLGrad, llama._RMSNormGrad, llama._CausalSoftmaxGrad,
             llama._SwiGLUGrad]


def test_every_function_run_directly_is_listed():
    used = set()
    for module in (linear, distill, llama):
        for node in ast.walk(ast.parse(inspect.getsource(module))):
            if isinstance(node, ast.Call) and getattr(node.func, "id", "") == "apply_in_backward":
                used.add(node.args[0].id)
    assert used == {f.__name__ for f in GRADIENTS}


@pytest.mark.parametrize("fn", GRADIENTS, ids=lambda f: f.__name__)
def test_forward_asks_its_ctx_for_no_more_than_the_stand_in_has(fn):
    """forward() may set attributes and call what _Unrecorded has; needs_input_grad and the like would be missing."""
    tree = ast.parse(textwrap.dedent(inspect.getsource(fn.forward)))
    loads = {n.attr for n in ast.walk(tree) if isinstance(n, ast.Attribute) and isinstance(n.ctx, ast.Load)
             and isinstance(n.value, ast.Name) and n.value.id == "ctx"}
    assert loads <= {name for name in vars(linear._Unrecorded) if not name.startswith("__")}
