"""The f32 products (sf_gemm on dense f32 operands) at the edges of their tiles and K splits, all three layouts, with
the second K segment and every epilogue, against float64 (conftest.gemm_err: 1e-5 of the output scale; a float32 sum
of K terms is off by about sqrt(K) 2^-24 of the terms' scale, K at most 8168 here)."""
import pytest
import torch

from conftest import gemm_err, gemm_splits, gemm_workspace

pytestmark = pytest.mark.gpu


def _mk(g, dev, *shape):
    return torch.randn(*shape, generator=g, device=dev)


@pytest.mark.parametrize("M,N,K", [
    (4, 4, 4), (32, 32, 36), (33, 16, 768), (16, 768, 8168), (3072, 16, 1000), (100, 132, 68),
    (129, 65, 260), (1021, 768, 3072), (768, 3072, 1021), (260, 2052, 33 * 4), (8168, 20, 768),
])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_layouts(cuda_device, M, N, K, layout):
    from sparseforge_amd import linear as lin

    if layout == "nt" and K % 4 or layout != "nt" and N % 4 or layout == "tn" and M % 4 or layout == "nn" and K % 4:
        pytest.skip("rows of whole 16-byte vectors only")
    g = torch.Generator(device=cuda_device).manual_seed(M + N + K)
    A = _mk(g, cuda_device, *((K, M) if layout == "tn" else (M, K)))
    B = _mk(g, cuda_device, *((N, K) if layout == "nt" else (K, N)))
    got = getattr(lin, "mm_" + layout)(A, B)
    a = A.double().t() if layout == "tn" else A.double()
    b = B.double().t() if layout == "nt" else B.double()
    assert gemm_err(got, a @ b, torch.float32) <= 1.0


@pytest.mark.parametrize("M,N,K,R", [(64, 96, 128, 4), (1000, 260, 516, 20), (48, 32, 8192, 64), (1000, 704, 1952, 20)])
def test_segment_bias_mask_accumulate(cuda_device, M, N, K, R):
    from sparseforge_amd import linear as lin

    if (M, N) == (1000, 704):  # the split-K reduce of four columns a thread takes its epilogue from 2^19 outputs on
        assert gemm_splits(torch.float32, M, N, K) > 1
    g = torch.Generator(device=cuda_device).manual_seed(M)
    A, B = _mk(g, cuda_device, M, K), _mk(g, cuda_device, N, K)
    z, S, bias = _mk(g, cuda_device, M, R), _mk(g, cuda_device, N, R), _mk(g, cuda_device, N)
    E, C, W = torch.rand(M, N, generator=g, device=cuda_device), _mk(g, cuda_device, M, N), _mk(g, cuda_device, M, N)
    prod = A.double() @ B.double().t() + z.double() @ S.double().t()
    kw = {"A2": z, "B2": S, "K2": R}
    assert gemm_err(lin.mm_nt(A, B, bias=bias, **kw), prod + bias.double(), torch.float32) <= 1.0
    assert gemm_err(lin.mm_nt(A, B, emask=E, **kw), prod * E.double(), torch.float32) <= 1.0
    got = lin.mm_nt(A, B, emask=E, dw=W, decay=0.25, **kw)
    assert gemm_err(got, prod + 0.25 * W.double() * (E < 0.5), torch.float32) <= 1.0
    got = lin.mm_nt(A, B, out=C.clone(), accumulate=True, **kw)
    assert gemm_err(got, prod + C.double(), torch.float32) <= 1.0
    for cap in (1, 2):  # fewer splits than planned: the workspace a caller gives
        with gemm_workspace(cap):
            assert gemm_err(lin.mm_nt(A, B, **kw), prod, torch.float32) <= 1.0


@pytest.mark.parametrize("layout,M,N,K,pieces", [
    ("nn", 8168, 768, 3072, 3), ("nt", 3312, 312, 632, 2), ("nn", 204, 3956, 804, 3), ("tn", 1024, 4096, 4096, 4),
    ("nt", 1384, 1308, 1896, 7), ("nt", 2692, 560, 516, 2)])
def test_error_of_the_sums(cuda_device, layout, M, N, K, pieces):
    """K is summed in pieces (runs or splits), so that the rounding of a chain of adds stays that of its length: each of
    n adds (two k each) of a random walk rounds by up to 2^-24 of a partial sum that has grown to sqrt(j / n) of the
    result, 2^-24 sqrt(n / 6) in all (rms); 15 % for the sums of the pieces."""
    from sparseforge_amd import linear as lin

    g = torch.Generator(device=cuda_device).manual_seed(K)
    A = _mk(g, cuda_device, *((K, M) if layout == "tn" else (M, K)))
    B = _mk(g, cuda_device, *((N, K) if layout == "nt" else (K, N)))
    a = A.double().t() if layout == "tn" else A.double()
    b = B.double().t() if layout == "nt" else B.double()
    ref = a.contiguous() @ b.contiguous()
    err = float((getattr(lin, "mm_" + layout)(A, B).double() - ref).norm() / ref.norm())
    assert err < 1.15 * 2.0 ** -24 * (K / pieces / 2 / 6) ** 0.5 + 2.0 ** -25, err
    z, S = _mk(g, cuda_device, M, 20), _mk(g, cuda_device, N, 20)
    if layout == "nt":  # a second segment after the last run
        got = lin.mm_nt(A, B, A2=z, B2=S, K2=20)
        assert gemm_err(got, ref + z.double() @ S.double().t(), torch.float32) <= 1.0
