"""A plain backward pass (the gradient Functions run directly) gives the gradients of one that records them
(create_graph), bit for bit: the same kernels run on the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _linear(dev):
    from sparseforge_amd import _lib as L
    from sparseforge_amd import linear as lin

    x = torch.randn(96, 128, device=dev).to(torch.bfloat16)
    W, P, S = (torch.randn(*s, device=dev).to(torch.bfloat16) * 0.1 for s in ((64, 128), (16, 128), (64, 16)))
    b, M = torch.randn(64, device=dev).to(torch.bfloat16), torch.rand(64, 128, device=dev).to(torch.bfloat16)
    return (x, W, b, P, S), lambda x, W, b, P, S: lin.masked_linear(x, W, b, M, "soft", 1.0, L.HARD_NONE, 2, 1.0, P, S,
                                                                    decay=0.1)


def _kl(dev):
    from sparseforge_amd.distill import chunked_kl_loss

    s, t = (torch.randn(1, 9, 100, device=dev) for _ in range(2))
    return (s,), lambda s: chunked_kl_loss(s, t, 2.0)


def _norm(dev):
    from sparseforge_amd.llama import RMSNorm

    norm = RMSNorm(64, 1e-6, device=dev)
    x = torch.randn(5, 64, device=dev)
    return (x, norm.weight.detach() * 1.5), lambda x, w: torch.func.functional_call(norm, {"weight": w}, (x,))


def _softmax(dev):
    from sparseforge_amd.llama import causal_softmax

    x = torch.randn(3, 40, 40, device=dev).masked_fill(torch.ones(40, 40, dtype=torch.bool, device=dev).triu(1), -1e30)
    return (x,), causal_softmax


def _swiglu(dev):
    from sparseforge_amd.llama import swiglu

    return tuple(torch.randn(6, 32, device=dev).to(torch.bfloat16) for _ in range(2)), swiglu


@pytest.mark.parametrize("make", [_linear, _kl, _norm, _softmax, _swiglu])
def test_same_gradients(cuda_device, make):
    inputs, fn = make(cuda_device)
    grads = []
    for create_graph in (False, True):
        xs = [t.clone().requires_grad_(True) for t in inputs]
        y = fn(*xs)
        go = torch.randn(y.shape, generator=torch.Generator(device=cuda_device).manual_seed(1), device=cuda_device)
        grads.append(torch.autograd.grad(y, xs, go.to(y.dtype), create_graph=create_graph))
    for a, b in zip(*grads):
        assert b.requires_grad and not a.requires_grad
        assert torch.equal(a, b.detach())
