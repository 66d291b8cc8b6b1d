"""sf_column_sum (the bias gradient) against float64 sums.

Bar: a float32 running sum of n terms is off by at most n 2^-24 times the sum of their magnitudes in the
worst case; here each thread adds at most rows / 128 terms before the fixed-order folds, so
rows 2^-24 sum|a| bounds every element, plus half an ulp of the output's dtype."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [
    (1, 8), (16, 264), (127, 36), (128, 2048), (513, 1536), (2049, 3072), (8168, 3072), (2050, 12288),
    (777, 6), (1031, 33),        # rows of no whole 16-byte chunk: the element loads
    (0, 64),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_column_sum(cuda_device, rows, cols, dtype):
    from sparseforge_amd import linear as lin

    g = torch.Generator().manual_seed(rows + cols)
    a = torch.randn(rows, cols, generator=g).to(dtype)
    got = lin.column_sum(a.to(cuda_device), dtype).double().cpu()
    ref, mag = a.double().sum(0), a.double().abs().sum(0)
    bound = max(rows, 1) * 2.0 ** -24 * mag + (ref.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    assert bool(((got - ref).abs() <= bound).all())


def test_column_sum_unaligned_rows(cuda_device):
    """A matrix that starts off a 16-byte boundary takes the element loads."""
    from sparseforge_amd import linear as lin

    a = torch.randn(300 * 64 + 1, device=cuda_device)[1:].view(300, 64)
    assert a.data_ptr() % 16
    got = lin.column_sum(a, torch.float32).double()
    assert float((got - a.double().sum(0)).abs().max()) <= 300 * 2.0 ** -24 * float(a.double().abs().sum(0).max())
