"""Single-sector Lanczos runs at the edges of the two-launch step: one state,
a handful of states (the recurrence stops by itself), odd lengths (the update
works on pairs of elements), lengths around the update's block and grid
limits, both H*v variants.

Tolerance: the coefficients follow the oracle's recurrence with sums in
another order; over 8 steps from a normalised random vector the difference
stays within 1e-10 of the spectrum's scale (as in the other Lanczos tests)."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, random_hubbard_params, siam_params

pytestmark = pytest.mark.gpu

# (model kind, sites, sector): 1, 5, 10, 225, 1225 = 35^2, 8,820, 731,808 states
CASES = [("hubbard", 5, (0, 0)), ("hubbard", 5, (0, 1)), ("hubbard", 5, (5, 3)), ("siam", 6, (2, 4)),
         ("hubbard", 7, (3, 4)), ("siam", 9, (4, 2)), ("siam", 12, (7, 6))]


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("kind,ns,sec", CASES)
def test_lanczos_steps_match_oracle(kind, ns, sec, variant):
    import edlib_amd as ea
    rng = np.random.default_rng(ns)
    p = random_hubbard_params(ns, rng) if kind == "hubbard" else siam_params(ns, 1, rng)
    ctx = ea.Context(0)
    ctx.set_model(product_model(kind, p))
    n = ctx.set_sector(*sec)
    ctx.hv_variant = variant
    srs = eo.SRS(oracle_model(kind, p), *sec)
    v = rng.uniform(-1, 1, n)
    v /= np.linalg.norm(v)
    for nl in (1, 2, 8):
        nlanc, a, b = ctx.lanczos(v, nl)
        no, ao, bo = srs.lanczos(v, nl)
        assert nlanc == no
        scale = max(1.0, np.abs(ao).max(), np.abs(bo).max())
        assert np.abs(a[:nlanc] - ao[:nlanc]).max() <= 1e-10 * scale
        assert np.abs(b[:nlanc] - bo[:nlanc]).max() <= 1e-10 * scale
        assert not a[nlanc:].any() and not b[nlanc + 1:].any()
    ctx.close()


@pytest.mark.parametrize("nz", [1, 63, 64, 257])
@pytest.mark.parametrize("nlanc", [1, 2, 3, 60, 1024, 1025])
def test_fractions_match_plain_recursion(nz, nlanc):
    """cf_eval around its block size and the longest staged run, against the
    bottom-up fraction in numpy (both are backward stable at these points:
    |Im z| >= 0.3 keeps every denominator away from zero; 1e-10 relative)."""
    import edlib_amd as ea
    rng = np.random.default_rng(nlanc)
    a, b = rng.normal(size=nlanc), np.concatenate([[0.0], rng.uniform(0.5, 2.0, nlanc)])
    z = 1j * (0.3 + 0.4 * np.arange(nz)) + 0.1
    ref = 1.0 / (z - a[-1])
    for i in range(nlanc - 2, -1, -1):
        ref = 1.0 / (z - a[i] - b[i + 1] ** 2 * ref)
    ctx = ea.Context(0)
    got = ctx.cf_eval(z, 0.7, nlanc, 1, 0.5, a, b)
    ctx.close()
    assert np.abs(got - 0.35 * ref).max() <= 1e-10 * np.abs(ref).max()
