"""The fused attention's gradients under create_graph (llama._attention_grads_by_passes) where q, k and v share a tensor,
depend on each other or carry hooks, against autograd through the attention itself (CPU, float64 inputs; the softmax
is float32, so 1e-5)."""
import pytest
import torch

from sparseforge_amd import llama

B, S, H, D = 1, 7, 2, 8


class _LikeFused(torch.autograd.Function):
    """_FusedAttention with the device passes of its forward replaced by torch's ops."""

    @staticmethod
    def forward(ctx, q, k, v, cos, sin):
        ctx.save_for_backward(q, k, v, cos, sin)
        return llama._causal_attention_torch(q, k, v, cos, sin)

    @staticmethod
    def backward(ctx, go):
        q, k, v, cos, sin = ctx.saved_tensors
        return (*llama._attention_grads_by_passes(q, k, v, cos, sin, go, ctx.needs_input_grad[:3]), None, None)


def _inputs(kind, hooks):
    g = torch.Generator().manual_seed(5)
    x, y = (torch.randn(B, S, H, D, generator=g, dtype=torch.float64).requires_grad_(True) for _ in range(2))
    if kind == "one leaf":
        qkv = (x, x, x)
    elif kind == "q and k":
        qkv = (x, x, y)
    elif kind == "one non-leaf":
        z = x * 1.5
        qkv = (z, z, z)
    elif kind == "chain":
        k = x * 0.5 + y
        qkv = (x, k, 2 * k)
    else:
        qkv = (x * 1.0, y * 1.0, x + y)
    seen = []
    if hooks:
        qkv[0].register_hook(lambda t: seen.append(1) or t * 3)
    return x, y, qkv, seen


@pytest.mark.parametrize("hooks", [False, True])
@pytest.mark.parametrize("kind", ["one leaf", "q and k", "one non-leaf", "chain", "independent"])
def test_create_graph(monkeypatch, kind, hooks):
    monkeypatch.setattr(llama, "_causal_attention_device", llama._causal_attention_torch)
    cos, sin = llama.rotary_tables(S, D, 10000.0, "cpu")
    w = torch.randn(B, S, H * D, generator=torch.Generator().manual_seed(6), dtype=torch.float64)
    outs = []
    for fn in (_LikeFused.apply, llama._causal_attention_torch):
        x, y, qkv, seen = _inputs(kind, hooks)
        loss = (fn(*qkv, cos, sin) * w).sum()
        leaves = [x] if kind.startswith("one") else [x, y]
        first = torch.autograd.grad(loss, leaves, create_graph=True)
        calls = len(seen)
        second = torch.autograd.grad(sum((t * t).sum() for t in first), leaves)
        outs.append(([t.detach() for t in (*first, *second)], calls))
    (got, calls), (want, ref_calls) = outs
    assert calls == ref_calls == int(hooks)
    for a, b in zip(got, want):
        assert float((a - b).norm() / b.norm()) < 1e-5
