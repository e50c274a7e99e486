"""Lanczos steps on rows that do not fit LDS (24,310 elements): the single pass
then has no barrier of its own between the step's scales, which every
work-group sums through LDS, and the sum of <v, w> through the same LDS.

Tolerance: over 8 steps from a normalised random vector the coefficients stay
within 1e-10 of the spectrum's scale of the oracle's (another order of sums, as
in the other Lanczos tests); two runs give the same bits."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, ring_hopping

pytestmark = pytest.mark.gpu


def test_lanczos_on_rows_longer_than_lds():
    import edlib_amd as ea
    p = dict(Ns=17, t=ring_hopping(17), U=np.full(17, 4.0), xmu=np.full(17, 2.0))
    ctx = ea.Context(0)
    ctx.set_model(product_model("hubbard", p))
    n = ctx.set_sector(1, 8)  # 17 x 24310
    ctx.hv_variant = 0
    srs = eo.SRS(oracle_model("hubbard", p), 1, 8)
    v = np.random.default_rng(2).uniform(-1, 1, n)
    v /= np.linalg.norm(v)
    no, ao, bo = srs.lanczos(v, 8)
    runs = [ctx.lanczos(v, 8) for _ in range(3)]
    for nl, a, b in runs:
        assert nl == no
        scale = max(1.0, np.abs(ao).max(), np.abs(bo).max())
        assert np.abs(a - ao).max() <= 1e-10 * scale and np.abs(b - bo).max() <= 1e-10 * scale
        assert np.array_equal(a, runs[0][1]) and np.array_equal(b, runs[0][2])
    ctx.close()
