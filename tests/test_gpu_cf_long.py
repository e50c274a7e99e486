"""Continued fractions of runs longer than the coefficients that are staged at
a time (1024 steps), around the multiples of that, in a context and in many
fractions of a batch's form, against the bottom-up fraction in numpy (both
backward stable at these points: |Im z| >= 0.3 keeps every denominator away from
zero; 1e-10 relative, as for the shorter ones)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [1, 65, 256])
@pytest.mark.parametrize("nlanc", [1026, 1500, 2047, 2048, 2049, 2050, 3073])
def test_long_fractions(nz, nlanc):
    import edlib_amd as ea
    rng = np.random.default_rng(nlanc)
    a, b = rng.normal(size=nlanc), np.concatenate([[0.0], rng.uniform(0.5, 2.0, nlanc)])
    z = 1j * (0.3 + 0.4 * np.arange(nz)) + 0.1
    ref = 1.0 / (z - a[-1])
    for i in range(nlanc - 2, -1, -1):
        ref = 1.0 / (z - a[i] - b[i + 1] ** 2 * ref)
    ctx = ea.Context(0)
    got = ctx.cf_eval(z, 0.7, nlanc, 1, 0.5, a, b)
    neg = ctx.cf_eval(-z, 0.7, nlanc, -1, 0.5, a, b)  # isign -1: the same up to the sign
    ctx.close()
    assert np.abs(got - 0.35 * ref).max() <= 1e-10 * np.abs(ref).max()
    assert np.abs(neg + 0.35 * ref).max() <= 1e-10 * np.abs(ref).max()
