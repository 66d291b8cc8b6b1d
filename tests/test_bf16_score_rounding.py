"""The bf16 importance scores |W| / sqrt(H + eps) need no correctly rounded f32 root or quotient.

The mask kernels round the root and the quotient of bf16 operands to bf16 straight from the hardware's
approximate f32 results.  Here every significand goes through the claim, with errors larger than the
hardware's: an f32 root off by up to 2 units in the last place, and a quotient off by up to 4, round to the
bf16 that the exact value rounds to."""
import numpy as np


def _bf16(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32)


def _exact_bf16(x):
    """float64 values rounded to 8 significant bits, ties to even."""
    m, e = np.frexp(x)
    return np.ldexp(np.rint(m * 256.0), e - 8).astype(np.float32)


def test_root_of_every_bf16():
    sig = np.arange(128, 256, dtype=np.float64) / 128
    for exp in (-2, -1, 0, 1):  # both parities of the exponent
        x = sig * 2.0 ** exp
        root = np.sqrt(x)
        want = _exact_bf16(root)
        near = root.astype(np.float32)
        for ulps in (-2, -1, 0, 1, 2):
            got = _bf16((near.view(np.int32) + ulps).view(np.float32))
            assert np.array_equal(got, want), (exp, ulps)


def test_quotient_of_every_bf16_pair():
    sig = np.arange(128, 256, dtype=np.float64) / 128
    q = sig[:, None] / sig[None, :]
    want = _exact_bf16(q)
    near = q.astype(np.float32)
    for ulps in range(-4, 5):
        got = _bf16((near.view(np.int32) + ulps).view(np.float32))
        assert np.array_equal(got, want), ulps
