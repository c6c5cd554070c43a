"""The quantiser's quotients, on the CPU: x / s for a bf16 value x and its block's scale
s = amax / 448 by one fused residual step (csrc/moe_quant_block.h), for every pair of
significands, against the correctly rounded division. The steps scale exactly with the
exponents, so one exponent of the maximum covers them all."""
import numpy as np
import pytest

F = np.float32
SIGNIFICANDS = (1 + np.arange(128) / 128.0).astype(F)


def _fma(a, b, c):
    # a * b is exact in 64 bits, and so is its sum with c in the extended type here
    return ((a.astype(np.float64) * b.astype(np.float64)).astype(np.longdouble) + c.astype(np.longdouble)).astype(F)


def _step(x, y, s):
    q = x * y
    return _fma(_fma(-s, q, x), y, q)


@pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="needs an extended float for the exact sum")
@pytest.mark.parametrize("ulps", [-3, 0, 3])
def test_quotients_are_correctly_rounded(ulps):
    """With y up to 3 ulps from 1 / s (the hardware's reciprocal is within 1)."""
    for m in SIGNIFICANDS * F(2.0 ** 5):
        s = F(m / F(448))
        y = (np.array([F(1) / s]).view(np.int32) + ulps).astype(np.int32).view(F)[0]
        x = np.concatenate([SIGNIFICANDS * F(2.0 ** (5 - d)) for d in range(24)])
        x = x[x <= m]
        got = _step(x, np.full_like(x, y), np.full_like(x, s))
        np.testing.assert_array_equal(got, x / s)


def test_scales_are_correctly_rounded():
    m = np.concatenate([SIGNIFICANDS, [F(1e-12)]]).astype(F)
    got = _step(m, np.full_like(m, F(1) / F(448)), np.full_like(m, 448))
    np.testing.assert_array_equal(got, m / F(448))
