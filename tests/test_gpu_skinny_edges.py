"""Skinny bf16 products at the edges of their plan: short sides of 8 to 64, long sides below and above a tile, K below
one stage per wave, K tails, K split over workgroups; all three layouts, against float64 (conftest.gemm_err)."""
import pytest
import torch

from conftest import bias_slack, gemm_err, gemm_workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("short", [8, 32, 40, 64])
@pytest.mark.parametrize("long,K", [(8, 8), (72, 200), (264, 1000), (1024, 8192), (96, 16384), (12296, 520)])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("rows_short", [False, True])
def test_edges(cuda_device, short, long, K, layout, rows_short):
    from sparseforge_amd import linear as lin

    M, N = (short, long) if rows_short else (long, short)
    g = torch.Generator(device=cuda_device).manual_seed(M * 3 + N + K)
    mk = lambda *s: torch.randn(*s, generator=g, device=cuda_device).to(torch.bfloat16)  # noqa: E731
    A = mk(*((K, M) if layout == "tn" else (M, K)))
    B = mk(*((N, K) if layout == "nt" else (K, N)))
    a = A.double().t() if layout == "tn" else A.double()
    b = B.double().t() if layout == "nt" else B.double()
    ref = a @ b
    f = getattr(lin, "mm_" + layout)
    assert gemm_err(f(A, B), ref, torch.bfloat16) <= 1.0
    with gemm_workspace(1):
        assert gemm_err(f(A, B, out_dtype=torch.float32), ref, torch.float32) <= 1.0
    bias = mk(N)
    assert gemm_err(f(A, B, bias=bias), ref + bias.double(), torch.bfloat16, bias_slack(ref, torch.bfloat16)) <= 1.0
