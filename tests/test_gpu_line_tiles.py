"""Row tiles of the line passes with slots that hold no row (more runs of
several rows than single rows to fill them up; tests/test_row_tiles_host.py
walks them), with infinities and NaN in the vector: an empty slot follows no
impurity term, so what is in its neighbours must not reach any element that
the operator does not couple to them.

Elements that are finite in the oracle's result are finite here and agree to
1e-13 of the largest (sums of at most ~100 products in FP64 in another order,
as for the other line-pass tests); the others are not finite here either."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, siam_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,nup,ndn", [(9, 4, 5), (11, 6, 5)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_empty_slots_take_nothing_from_their_neighbours(ns, nup, ndn, bad):
    import edlib_amd as ea
    p = siam_params(ns, 3, np.random.default_rng(ns), mu=1.3, h0_offdiag=0.2)
    ctx = ea.Context(0)
    ctx.set_model(product_model("siam", p))
    n = ctx.set_sector(nup, ndn)
    ctx.hv_variant = 1
    srs = eo.SRS(oracle_model("siam", p), nup, ndn)
    rng = np.random.default_rng(3)
    v = rng.uniform(-1, 1, n)
    finite = srs.av(v)
    tol = 1e-13 * max(1.0, np.abs(finite).max())
    assert np.abs(ctx.av(v) - finite).max() <= tol
    for at in rng.integers(0, n, 8):
        x = v.copy()
        x[at] = bad
        with np.errstate(invalid="ignore"):
            ref = srs.av(x)
        got = ctx.av(x)
        ok = np.isfinite(ref)
        assert not ok.all() and np.array_equal(np.isfinite(got), ok)
        assert np.abs(got[ok] - ref[ok]).max() <= tol
    ctx.close()
