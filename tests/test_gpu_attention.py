"""The fused bf16 causal attention (llama.causal_attention for heads of 64 or 128) against float64.

Bar: the inputs are rotated in bf16 (both sides take the same rotated values), then p and ds round to bf16 once
each before their product and the outputs round once: every output is a sum whose terms are off by at most 2^-8
relative (2^-9 each for p or ds and for the stored result), so norm-wise 2^-8; 1e-2 leaves a factor of 2.5 for the
rotation's own roundings in dq and dk."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(q, k, v, cos, sin, go):
    from sparseforge_amd import llama

    B, S, H, D = q.shape
    c, s = cos.to(q.dtype), sin.to(q.dtype)
    rot = lambda t: llama._rotate(t.transpose(1, 2), c, s)  # noqa: E731
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    qd = rot(q).double()
    kd = rot(k).double()
    sc = qd @ kd.transpose(-1, -2) * D ** -0.5
    sc = sc.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    o = (sc.softmax(-1) @ v.transpose(1, 2).double()).transpose(1, 2).reshape(B, S, H * D)
    return o, torch.autograd.grad(o, (q, k, v), go.double())


@pytest.mark.parametrize("S", [1, 31, 64, 65, 128, 129, 200, 577, 1024])
@pytest.mark.parametrize("B,H,D", [(2, 4, 64), (1, 3, 64), (1, 8, 128), (2, 1, 128)])
def test_forward_and_gradients(cuda_device, S, B, H, D):
    from sparseforge_amd import llama

    g = torch.Generator(device=cuda_device).manual_seed(S + D)
    q, k, v = (torch.randn(B, S, H, D, generator=g, device=cuda_device).to(torch.bfloat16).requires_grad_(True)
               for _ in range(3))
    go = torch.randn(B, S, H * D, generator=g, device=cuda_device).to(torch.bfloat16)
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    assert llama._fused_attention_takes(q, k, v, cos, sin)
    o = llama.causal_attention(q, k, v, cos, sin)
    grads = torch.autograd.grad(o, (q, k, v), go)
    ro, rg = _ref(q, k, v, cos, sin, go)
    for got, want in zip((o, *grads), (ro, *rg)):
        got, want = got.detach(), want.detach()
        assert torch.isfinite(got).all()
        err = float((got.double() - want.double()).norm() / want.double().norm().clamp_min(1e-30))
        assert err < 1e-2 or float(want.double().norm()) < 1e-3, err


def test_large_scores_and_nan(cuda_device):
    """Rows whose scores are far apart (one key takes all), and a NaN that stays in its head's later rows."""
    from sparseforge_amd import llama

    S, D = 150, 64
    q, k, v = (torch.randn(1, S, 2, D, device=cuda_device) for _ in range(3))
    q, k, v = (t.to(torch.bfloat16) for t in (q * 60, k * 60, v))
    go = torch.randn(1, S, 2 * D, device=cuda_device).to(torch.bfloat16)
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    o = llama.causal_attention(q, k, v, cos, sin)
    ro, _ = _ref(q, k, v, cos, sin, go)
    assert torch.isfinite(o).all()
    assert float((o.double() - ro.detach()).norm() / ro.detach().norm()) < 1e-2
    v2 = v.clone()
    v2[0, 100, 1, 3] = float("nan")
    o2 = llama.causal_attention(q, k, v2, cos, sin).view(S, 2, D)
    assert torch.isfinite(o2[:, 0]).all() and torch.isfinite(o2[:64, 1]).all() and torch.isnan(o2[100:, 1, 3]).all()


def test_double_backward_takes_the_materialised_path(cuda_device):
    """With create_graph the gradients equal the materialised path's, and so do the second derivatives."""
    from sparseforge_amd import llama

    B, S, H, D = 1, 96, 2, 64
    g = torch.Generator(device=cuda_device).manual_seed(3)
    base = [torch.randn(B, S, H, D, generator=g, device=cuda_device).to(torch.bfloat16) for _ in range(3)]
    probes = [torch.randn(B, S, H, D, generator=g, device=cuda_device) for _ in range(3)]
    w = torch.randn(B, S, H * D, generator=g, device=cuda_device)
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    outs = []
    for fn in (llama.causal_attention, llama._causal_attention_device):
        x = [t.clone().requires_grad_(True) for t in base]
        loss = (fn(*x, cos, sin).float() * w).sum()  # linear in the output: the same upstream gradient
        grads = torch.autograd.grad(loss, x, create_graph=True)
        dot = sum((a.float() * p).sum() for a, p in zip(grads, probes))
        outs.append((*grads, *torch.autograd.grad(dot, x)))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_calls_outside_the_fused_path(cuda_device):
    """float32 and another head size run the materialised path, which refuses unaligned operands; the fused path takes
    rows up to the softmax passes' longest."""
    from sparseforge_amd import llama

    for D, dt in ((64, torch.float32), (32, torch.bfloat16), (96, torch.bfloat16)):
        q, k, v = (torch.randn(1, 40, 2, D, device=cuda_device).to(dt) for _ in range(3))
        cos, sin = llama.rotary_tables(40, D, 10000.0, cuda_device)
        assert not llama._fused_attention_takes(q, k, v, cos, sin)
        assert torch.equal(llama.causal_attention(q, k, v, cos, sin),
                           llama._causal_attention_device(q, k, v, cos, sin))
    cos, sin = llama.rotary_tables(40, 64, 10000.0, cuda_device)
    for which in range(3):  # one operand 2 bytes off a 16-byte boundary
        qkv = [torch.randn(1, 40, 2, 64, device=cuda_device).to(torch.bfloat16) for _ in range(3)]
        flat = torch.empty(40 * 2 * 64 + 1, dtype=torch.bfloat16, device=cuda_device)[1:]
        qkv[which] = flat.view(1, 40, 2, 64).copy_(qkv[which])
        assert not llama._fused_attention_takes(*qkv, cos, sin)
        with pytest.raises(ValueError, match="aligned"):
            llama.causal_attention(*qkv, cos, sin)
    for S in (4096, 4097):
        q = torch.empty(1, S, 1, 64, dtype=torch.bfloat16, device=cuda_device)
        t = torch.empty(S, 64, device=cuda_device)
        assert llama._fused_attention_takes(q, q, q, t, t) == (S <= llama.FUSED_MAX_S == 4096)


def test_unaligned_and_strided_gradient(cuda_device):
    """An upstream gradient 2 bytes off a boundary, or strided, gives the aligned one's gradients."""
    from sparseforge_amd import llama

    S, H, D = 70, 2, 64
    q, k, v = (torch.randn(1, S, H, D, device=cuda_device).to(torch.bfloat16).requires_grad_(True) for _ in range(3))
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    go = torch.randn(1, S, H * D, device=cuda_device).to(torch.bfloat16)
    want = torch.autograd.grad(llama.causal_attention(q, k, v, cos, sin), (q, k, v), go)
    off = torch.empty(go.numel() + 1, dtype=go.dtype, device=cuda_device)[1:].view_as(go).copy_(go)
    strided = go.transpose(1, 2).contiguous().transpose(1, 2)
    for g in (off, strided):
        got = torch.autograd.grad(llama.causal_attention(q, k, v, cos, sin), (q, k, v), g)
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("D", [64, 128])
def test_first_keys_at_minus_infinity(cuda_device, D):
    """Queries whose first tile of 64 keys (and 6 more) scores -inf in float32, the rest finite: those keys get
    probability 0 and nothing becomes NaN."""
    from sparseforge_amd import llama

    S = 200
    q, k, v, go = (torch.randn(1, S, 2, D, device=cuda_device) for _ in range(4))
    q[:, :70], q[:, 70:] = 1e-19, 1e18     # 1e18 * -1e21 * D overflows; 1e-19 * -1e21 * D does not
    k[:, :70] = -1e21
    k[:, 70:] *= 1e-18
    go[:, :70] = 0                         # those queries' dq is a cancelling sum of terms of 1e21
    q, k, v, go = (t.to(torch.bfloat16) for t in (q, k, v, go.reshape(1, S, 2 * D)))
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    cos, sin = torch.ones(S, D, device=cuda_device), torch.zeros(S, D, device=cuda_device)  # no rotation
    o = llama.causal_attention(q, k, v, cos, sin)
    grads = torch.autograd.grad(o, (q, k, v), go)
    ro, rg = _ref(q, k, v, cos, sin, go)
    for part in (slice(0, 70), slice(70, S)):  # gradients of the two parts differ by orders of magnitude
        for got, want in zip((o, *grads), (ro, *rg)):
            a, b = got.detach()[:, part].double(), want.detach()[:, part].double()
            assert torch.isfinite(a).all()
            assert float((a - b).norm()) <= 1e-2 * float(b.norm()) + 1e-30 * a.numel()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("size", [1.0, 30.0, 1e3, 1e6, 1e15])
def test_runaway_scores(cuda_device, D, size):
    """Scores up to 2^100 (one key takes all, or the first two share: they are equal) in all heads but the first, forward
    and backward.  dq, which cancels exactly where two equal keys share, only has to be finite."""
    from sparseforge_amd import llama

    S = 150
    g = torch.Generator(device=cuda_device).manual_seed(D)
    q, k, v, go = (torch.randn(1, S, 4, D, generator=g, device=cuda_device) for _ in range(4))
    k[:, :2] = 3 * k[:, :1]  # the first two keys take many rows
    q[:, :, 1:] *= size
    k[:, :, 1:] *= size
    q, k, v, go = (t.to(torch.bfloat16) for t in (q, k, v, go.reshape(1, S, 4 * D)))
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    cos, sin = torch.ones(S, D, device=cuda_device), torch.zeros(S, D, device=cuda_device)  # no rotation
    o = llama.causal_attention(q, k, v, cos, sin)
    grads = torch.autograd.grad(o, (q, k, v), go)
    ro, rg = _ref(q, k, v, cos, sin, go)
    assert torch.isfinite(grads[0]).all()
    for got, want in ((o, ro), (grads[1], rg[1]), (grads[2], rg[2])):
        got, want = (t.detach().double().view(S, 4, D) for t in (got, want))
        assert torch.isfinite(got).all()
        for h in range(4):
            assert float((got[:, h] - want[:, h]).norm() / want[:, h].norm()) < 1e-2


def test_output_changed_in_place(cuda_device):
    """The output may be changed in place before the backward, which then sees the change as an op of its own."""
    from sparseforge_amd import llama

    S, H, D = 70, 3, 64
    q, k, v = (torch.randn(1, S, H, D, device=cuda_device).to(torch.bfloat16).requires_grad_(True) for _ in range(3))
    go = torch.randn(1, S, H * D, device=cuda_device).to(torch.bfloat16)
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    want = torch.autograd.grad(llama.causal_attention(q, k, v, cos, sin), (q, k, v), go * 2)
    o = llama.causal_attention(q, k, v, cos, sin)
    o.mul_(2)
    for a, b in zip(torch.autograd.grad(o, (q, k, v), go), want):
        assert torch.equal(a, b)


def test_delta_from_the_unrounded_output(cuda_device):
    """delta = sum(go o) from the output before its rounding.  With values of 100 +- 1 the gradients are what is left of
    go v after delta, about 8; the output's rounding (0.14 rms at 100) would move delta by 0.14 sqrt(64) = 1.15, 14 %.
    The forward's own rounding of p moves o by 100 2^-9 / sqrt(3 n) over n keys, below 7e-3 at n >= 256; with ds's
    2^-9 that stays under 2e-2."""
    from sparseforge_amd import llama

    S, H, D = 512, 2, 64
    g = torch.Generator(device=cuda_device).manual_seed(2)
    q, k = (torch.randn(1, S, H, D, generator=g, device=cuda_device) * 0.05 for _ in range(2))
    v = 100.0 + torch.randn(1, S, H, D, generator=g, device=cuda_device)
    q, k, v = (t.to(torch.bfloat16).requires_grad_(True) for t in (q, k, v))
    go = torch.randn(1, S, H * D, generator=g, device=cuda_device).to(torch.bfloat16)
    go[:, :256] = 0
    cos, sin = torch.ones(S, D, device=cuda_device), torch.zeros(S, D, device=cuda_device)
    o = llama.causal_attention(q, k, v, cos, sin)
    dq, dk, _ = torch.autograd.grad(o, (q, k, v), go)
    _, rg = _ref(q, k, v, cos, sin, go)
    for a, b in ((dq, rg[0]), (dk, rg[1])):
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 2e-2


def test_graph_replays(cuda_device):
    """A captured forward and backward, replayed on inputs whose scores run away, then do not, and again: the word that
    selects the backward's body is written anew each time."""
    from sparseforge_amd import llama

    S, H, D = 130, 2, 64
    cos, sin = llama.rotary_tables(S, D, 10000.0, cuda_device)
    g = torch.Generator(device=cuda_device).manual_seed(9)
    mk = lambda f: [(torch.randn(1, S, H, D, generator=g, device=cuda_device) * f).to(torch.bfloat16) for _ in range(3)]  # noqa: E731
    q, k, v = (t.requires_grad_(True) for t in mk(1.0))
    go = torch.randn(1, S, H * D, generator=g, device=cuda_device).to(torch.bfloat16)

    def call():
        o = llama.causal_attention(q, k, v, cos, sin)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), go))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = call()
    for size in (1.0, 1e4, 2.0, 1e6):
        with torch.no_grad():
            for t, new in zip((q, k, v), mk(size)):
                t.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in outs]
        for a, b in zip(got, call()):
            assert torch.isfinite(a).all() and torch.equal(a, b)
