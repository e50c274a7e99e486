"""Lanczos steps of sectors with many rows, whose scales and shares of <v, w>
are summed once in launches of their own: rows around the lines (2000 with a
million states, 3000 shares, 6000 rows), both H*v variants, and runs that stop
by themselves at the first and the second step.

Tolerance: over 8 steps from a normalised random vector the coefficients stay
within 1e-10 of the spectrum's scale of the oracle's (another order of sums, as
in the other Lanczos tests)."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, ring_hopping, siam_params

pytestmark = pytest.mark.gpu


def _ring(ns):
    return "hubbard", dict(Ns=ns, t=ring_hopping(ns), U=np.full(ns, 4.0), xmu=np.full(ns, 2.0))


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("model,sec", [
    (_ring(14), (5, 3)),     # 2002 x 364: fewer than a million states
    (_ring(14), (5, 4)),     # 2002 x 1001: scales once, shares as they are
    (_ring(14), (6, 2)),     # 3003 x 91: shares folded
    (_ring(14), (7, 4)),     # 3432 x 1001: both
    (_ring(15), (6, 1)),     # 5005 x 15
    (_ring(15), (7, 1)),     # 6435 x 15: both, short rows
    (_ring(16), (8, 1)),     # 12870 x 16, tiles
    (("siam", siam_params(15, 1, np.random.default_rng(1))), (7, 2)),
])
def test_steps_match_oracle(model, sec, variant):
    import edlib_amd as ea
    kind, p = model
    ctx = ea.Context(0)
    ctx.set_model(product_model(kind, p))
    n = ctx.set_sector(*sec)
    ctx.hv_variant = variant
    srs = eo.SRS(oracle_model(kind, p), *sec)
    v = np.random.default_rng(3).uniform(-1, 1, n)
    v /= np.linalg.norm(v)
    for nl in (1, 2, 8):
        nlanc, a, b = ctx.lanczos(v, nl)
        no, ao, bo = srs.lanczos(v, nl)
        assert nlanc == no
        scale = max(1.0, np.abs(ao).max(), np.abs(bo).max())
        assert np.abs(a - ao).max() <= 1e-10 * scale and np.abs(b - bo).max() <= 1e-10 * scale
    r0, r1 = ctx.lanczos(v, 8), ctx.lanczos(v, 8)
    assert np.array_equal(r0[1], r1[1]) and np.array_equal(r0[2], r1[2])
    ctx.close()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("states", [1, 2])
def test_runs_stop_by_themselves(states, variant):
    """Without hopping a state is an eigenvector, two of different energy span
    an invariant subspace: the exact recurrence ends after one or two steps."""
    import edlib_amd as ea
    rng = np.random.default_rng(8)
    p = dict(Ns=15, t=np.zeros((15, 15)), U=rng.uniform(1, 5, 15), xmu=rng.uniform(0, 2, 15))
    ctx = ea.Context(0)
    ctx.set_model(product_model("hubbard", p))
    n = ctx.set_sector(7, 1)
    ctx.hv_variant = variant
    at = [n // 3, n // 2 + 1][:states]
    e = [ctx.av(np.eye(1, n, k)[0])[k] for k in at]
    v = np.zeros(n)
    v[at] = states ** -0.5
    nl, a, b = ctx.lanczos(v, 8)
    assert nl == states and not a[states:].any() and not b[states + 1:].any()
    assert abs(a[0] - np.mean(e)) <= 1e-12 * max(1.0, np.abs(e).max())
    if states == 2:
        assert abs(e[0] - e[1]) > 1e-3
        assert abs(b[1] - abs(e[0] - e[1]) / 2) <= 1e-12 * np.abs(e).max()
    ctx.close()
