"""The KL kernels on vocabularies that are no multiple of a vector: rows then start at every offset from a 16-byte
boundary, with elements before the first whole slice and after the last.  f32 against the float64 oracle with the bars
of test_gpu_distill.py (loss 2e-6, gradient 1e-5 of its largest), bf16 gradients within 2^-7 relative plus 1e-3 of it;
rows below and above the count that takes 1024 threads a row; a view off a 16-byte boundary."""
import numpy as np
import pytest
import torch

from oracle import distill as od

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3, 256, 257])
@pytest.mark.parametrize("vocab", [1, 5, 8, 9, 15, 33, 2051, 8190])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])
def test_ragged_vocabulary(cuda_device, rows, vocab, dtype, shift):
    from sparseforge_amd.distill import chunked_kl_loss

    g = torch.Generator().manual_seed(rows * vocab)
    s = (torch.randn(rows, vocab, generator=g) * 4).to(dtype)
    t = (torch.randn(rows, vocab, generator=g) * 4).to(dtype)
    s[-1, -1] = 200.0  # beyond the clamp
    flat = torch.empty(rows * vocab + shift, dtype=dtype, device=cuda_device)
    sd = flat[shift:].view(rows, vocab)
    sd.copy_(s)
    sd = sd.detach().requires_grad_(True)
    kl = chunked_kl_loss(sd, t.to(cuda_device))
    ref = od.kl_loss(s.float().numpy(), t.float().numpy(), 2.0)
    tol = 2e-6 if dtype == torch.float32 else 2.0 ** -7
    np.testing.assert_allclose(kl.float().item(), ref, rtol=tol, atol=1e-6)
    (kl * 3.0).backward()
    want = od.kl_grad(s.float().numpy(), t.float().numpy(), 2.0, g=3.0)
    got = sd.grad.float().cpu().numpy()
    big = np.abs(want).max()
    if dtype == torch.float32:
        np.testing.assert_allclose(got, want, rtol=0, atol=1e-5 * big + 1e-12)
    else:
        np.testing.assert_allclose(got, want, rtol=2.0 ** -7, atol=1e-3 * big + 1e-12)
    assert got[-1, -1] == 0.0


@pytest.mark.parametrize("rows,vocab,dtype", [(3, 49157, torch.bfloat16), (65, 49152, torch.bfloat16),
                                              (65, 24581, torch.float32), (3, 24576, torch.float32)])
@pytest.mark.parametrize("shift", [0, 1])
def test_few_wide_rows(cuda_device, rows, vocab, dtype, shift):
    """The forward's 1024 threads a row: few rows of 96 KiB and more."""
    test_ragged_vocabulary(cuda_device, rows, vocab, dtype, shift)
