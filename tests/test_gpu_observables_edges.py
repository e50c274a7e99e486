"""Static observables at the edges of their kernels: fewer and more columns
than a round of a block (1024), one row and one column, row tiles of 128 with
a remainder, 16 and 17 sites (16 or 32 bit slots).

The sums run over at most n positive terms of a normalised vector, so they
agree with numpy's to n eps < 1e-10 (n <= 1e5)."""
import numpy as np
import pytest

from edlib_amd.workloads import torus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,nup,ndn", [(6, 0, 3), (6, 3, 6), (9, 4, 4), (10, 5, 1), (13, 1, 6), (13, 6, 1),
                                        (16, 2, 3), (16, 3, 1), (17, 2, 2), (17, 1, 3)])
def test_observables_match_numpy(ns, nup, ndn):
    import edlib_amd as ea
    from itertools import combinations
    ctx = ea.Context(0)
    ctx.set_model(ea.HubbardModel(ns, torus(1, ns), np.full(ns, 4.0), np.full(ns, 2.0)))
    n = ctx.set_sector(nup, ndn)
    v = np.random.default_rng(ns).uniform(-1, 1, n)
    v /= np.linalg.norm(v)
    got = ctx.static_observables(v, ns)
    ctx.close()

    def occ(k):  # site s at bit ns - 1 - s, combinations of positions in order
        b = [sum(1 << q for q in c) for c in combinations(range(ns), k)]
        return np.array([[(x >> (ns - 1 - i)) & 1 for x in b] for i in range(ns)], dtype=float)

    ou, od = occ(nup), occ(ndn)
    w = (v ** 2).reshape(ou.shape[1], od.shape[1])
    nu, nd = ou @ w.sum(1), od @ w.sum(0)
    uu, dd = (ou * w.sum(1)) @ ou.T, (od * w.sum(0)) @ od.T
    ud = ou @ w @ od.T
    ref = {"N": nu + nd, "N_up": nu, "N_dn": nd, "M": nu - nd, "D_occ": np.diag(ud),
           "M_i M_j": (uu - ud - ud.T + dd).reshape(-1), "N_eff": np.array([1.0 / (v ** 4).sum()])}
    for k, r in ref.items():
        assert np.abs(np.asarray(got[k]).reshape(-1) - r).max() <= 1e-10 * max(1.0, np.abs(r).max())
