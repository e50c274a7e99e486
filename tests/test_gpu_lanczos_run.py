"""Lanczos runs that one work-group takes whole (csrc/lanczos_run.hip) and the
first sectors that it leaves to the stepwise form: one state, one row, one
column, rows and columns that do not divide the work-group evenly, the longest
rows of either entry count, every cross term, impurity terms, a start vector
in an invariant subspace (the recurrence stops by itself), and sectors just
past the limits (line length, states, hops).

Tolerance: the coefficients follow the oracle's recurrence with sums in
another order; over 8 steps from a normalised random vector the difference
stays within 1e-10 of the spectrum's scale (as in the other Lanczos tests)."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import (kanamori_tensor, oracle_model, product_model, random_hubbard_params, ring_hopping,
                          siam_params)

pytestmark = pytest.mark.gpu


def _ring(ns):
    return "hubbard", dict(Ns=ns, t=ring_hopping(ns), U=np.full(ns, 4.0), xmu=np.full(ns, 2.0))


def _siam(ns, ml, seed):
    p = siam_params(ns, ml, np.random.default_rng(seed), mu=1.3, h0_offdiag=0.2 if ml > 1 else 0.0)
    if ml not in (1, 3):
        p["U"] = kanamori_tensor(ml, 4.0, 0.7)
    return "siam", p


def _dense(ns, seed):
    return "hubbard", random_hubbard_params(ns, np.random.default_rng(seed))


CASES = {
    "one state": (_ring(6), (6, 0)),
    "one row": (_ring(9), (0, 4)),
    "one column": (_ring(9), (4, 9)),
    "ring 8": (_ring(8), (5, 4)),                     # 56 x 70, at most 8 hops
    "ring 8, largest": (_ring(8), (4, 4)),            # 70 x 70
    "wide": (_ring(12), (1, 4)),                      # 12 x 495: two rows at a time
    "tall": (_ring(12), (4, 1)),
    "too long a line": (_ring(13), (1, 5)),           # 13 x 1287: stepwise
    "too many states": (_ring(9), (4, 4)),            # 126 x 126: stepwise
    "sixteen hops": (_dense(8, 3), (4, 4)),           # 16 hops a row, general cross term
    "more hops": (_dense(9, 4), (4, 2)),              # 20 hops: stepwise
    "Anderson": (_siam(8, 1, 5), (3, 5)),
    "two orbitals": (_siam(8, 2, 6), (4, 3)),
    "three orbitals": (_siam(8, 3, 7), (4, 4)),
    "four orbitals": (_siam(7, 4, 8), (3, 4)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_run_matches_oracle(name):
    import edlib_amd as ea
    (kind, p), (nup, ndn) = CASES[name]
    ctx = ea.Context(0)
    ctx.set_model(product_model(kind, p))
    n = ctx.set_sector(nup, ndn)
    srs = eo.SRS(oracle_model(kind, p), nup, ndn)
    rng = np.random.default_rng(9)
    v = rng.uniform(-1, 1, n)
    v /= np.linalg.norm(v)
    starts = [v]
    if n > 1:  # a state of two eigenvector-like components: stops early or runs on, as the oracle does
        e = np.zeros(n)
        e[n // 2] = 1.0
        starts.append(e)
    for x in starts:
        for nl in (1, 2, 8):
            nlanc, a, b = ctx.lanczos(x, nl)
            no, ao, bo = srs.lanczos(x, nl)
            assert nlanc == no
            scale = max(1.0, np.abs(ao).max(), np.abs(bo).max())
            assert np.abs(a[:nlanc] - ao[:nlanc]).max() <= 1e-10 * scale
            assert np.abs(b[:nlanc] - bo[:nlanc]).max() <= 1e-10 * scale
            assert not a[nlanc:].any() and not b[nlanc + 1:].any()
    # the same bits again
    r0, r1 = ctx.lanczos(v, 8), ctx.lanczos(v, 8)
    assert r0[0] == r1[0] and np.array_equal(r0[1], r1[1]) and np.array_equal(r0[2], r1[2])
    ctx.close()
