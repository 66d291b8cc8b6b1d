"""bf16 products at the shapes the 128 x 128 tiles take (sf_gemm picks them from the shape): edges of tiles, K tails, K
splits and fewer splits than planned, all three layouts, second K segment, every epilogue; against float64 products
of the same operands (conftest.gemm_err)."""
import pytest
import torch

from conftest import bias_slack, gemm_err, gemm_splits, gemm_workspace

pytestmark = pytest.mark.gpu


def _mk(g, dev, *shape):
    return torch.randn(*shape, generator=g, device=dev).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K", [
    (72, 72, 8), (128, 128, 64), (136, 72, 72), (256, 264, 1000), (1024, 2048, 2048), (520, 2056, 200),
    (1000, 704, 1952), (2048, 2048, 4096), (4096, 2048, 520), (2184, 2056, 8), (2184, 2056, 136),
])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_layouts(cuda_device, M, N, K, layout):
    from sparseforge_amd import linear as lin

    g = torch.Generator(device=cuda_device).manual_seed(M + N + K)
    A = _mk(g, cuda_device, *((K, M) if layout == "tn" else (M, K)))
    B = _mk(g, cuda_device, *((N, K) if layout == "nt" else (K, N)))
    a = A.double().t() if layout == "tn" else A.double()
    b = B.double().t() if layout == "nt" else B.double()
    ref = a @ b
    for cap in (None, 1, 2):
        with gemm_workspace(cap):
            assert gemm_err(getattr(lin, "mm_" + layout)(A, B), ref, torch.bfloat16) <= 1.0


@pytest.mark.parametrize("M,N,K,R", [(80, 96, 128, 8), (1000, 264, 520, 72), (200, 2048, 4096, 64), (1000, 704, 1952, 72),
                                     (5632, 2048, 1032, 64)])  # the last on 256 x 256 tiles
def test_segment_bias_mask_accumulate(cuda_device, M, N, K, R):
    from sparseforge_amd import linear as lin

    if (M, N) == (1000, 704):  # the split-K reduce of four columns a thread takes its epilogue from 2^19 outputs on
        assert gemm_splits(torch.bfloat16, M, N, K) > 1
    g = torch.Generator(device=cuda_device).manual_seed(M)
    A, B, z, S = (_mk(g, cuda_device, *s) for s in ((M, K), (N, K), (M, R), (N, R)))
    bias, C, W = _mk(g, cuda_device, N), _mk(g, cuda_device, M, N), _mk(g, cuda_device, M, N)
    E = torch.rand(M, N, generator=g, device=cuda_device).to(torch.bfloat16)
    prod = A.double() @ B.double().t() + z.double() @ S.double().t()
    kw = {"A2": z, "B2": S, "K2": R}
    slack = bias_slack(prod, torch.bfloat16)  # the epilogue works on the rounded product
    bf = torch.bfloat16
    assert gemm_err(lin.mm_nt(A, B, **kw), prod, bf) <= 1.0
    assert gemm_err(lin.mm_nt(A, B, out_dtype=torch.float32, **kw), prod, torch.float32) <= 1.0
    assert gemm_err(lin.mm_nt(A, B, bias=bias, **kw), prod + bias.double(), bf, slack) <= 1.0
    assert gemm_err(lin.mm_nt(A, B, emask=E, **kw), prod * E.double(), bf, slack) <= 1.0
    got = lin.mm_nt(A, B, out=C.clone(), accumulate=True, **kw)
    assert gemm_err(got, prod + C.double(), bf, slack) <= 1.0
    got = lin.mm_nt(A, B, emask=E, dw=W, decay=0.25, **kw)
    assert gemm_err(got, prod + 0.25 * W.double() * (E < 0.5), bf, 2 * slack) <= 1.0
