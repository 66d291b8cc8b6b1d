"""The packed 2:4 product at the edges of its kernels: the 32 x 32 and 64 x 64 K-split tiles, the 128 x 128 tile and
the 256 x 256 tile are picked from the shape; each is checked against float64 products of the same bf16 operands
(conftest.gemm_err), with bias, low-rank term and both output types."""
import pytest
import torch

from conftest import bias_slack, gemm_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,out_f,in_f", [
    (1, 32, 64), (3, 96, 128), (31, 4096, 512), (33, 2048, 576),          # 32 x 32, fewer stages than waves
    (65, 4096, 4096), (300, 4064, 1088), (512, 2080, 2112),               # 64 x 64, a half row tile
    (129, 11008, 1024), (700, 4096, 1984), (1537, 2016, 832),             # 128 x 128, ragged both ways
    (2048, 8192, 256),                                                    # 256 x 256
])
@pytest.mark.parametrize("rank,bias", [(0, False), (8, True), (72, True)])
def test_small_tiles(cuda_device, tokens, out_f, in_f, rank, bias):
    from sparseforge_amd import finalize as F
    from sparseforge_amd import linear as lin

    g = torch.Generator(device=cuda_device).manual_seed(tokens + out_f)
    W = (torch.randn(out_f, in_f, generator=g, device=cuda_device) * 0.05).to(torch.bfloat16)
    keep = torch.rand(out_f, in_f // 4, 4, generator=g, device=cuda_device).topk(2, -1).indices
    M = torch.zeros(out_f, in_f // 4, 4, device=cuda_device).scatter_(-1, keep, 1.0).view(out_f, in_f)
    x = torch.randn(tokens, in_f, generator=g, device=cuda_device).to(torch.bfloat16)
    b = torch.randn(out_f, generator=g, device=cuda_device).to(torch.bfloat16) if bias else None
    p = F.pack_2to4(W, M.to(torch.bfloat16))
    prod = x.double() @ (W.double() * M).t()
    if rank:
        z = torch.randn(tokens, rank, generator=g, device=cuda_device).to(torch.bfloat16)
        S = (torch.randn(out_f, rank, generator=g, device=cuda_device) * 0.05).to(torch.bfloat16)
        prod = prod + z.double() @ S.double().t()
        y = lin.gemm_2to4(x, p.vals, p.idx, out_f, z=z, S=S, bias=b)
    else:
        y = F.gemm_2to4(x, p, b)
        y32 = F.gemm_2to4(x, p, b, out_dtype=torch.float32)
        assert gemm_err(y32, prod + (b.double() if bias else 0), torch.float32) <= 1.0
    ref = prod + (b.double() if bias else 0)
    extra = bias_slack(prod, torch.bfloat16) if bias else None
    assert gemm_err(y, ref, torch.bfloat16, extra) <= 1.0
