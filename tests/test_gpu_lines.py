"""The two line passes of H*v (csrc/hv_lines.hip) at the edges of their tiles:
rows and columns that are not a multiple of four, lines longer than one round
of a work-group (1024 states) and than four at a time (4096), one-line and
two-line sectors, and the impurity terms in whole-run tiles (two and three
orbitals) and from memory (four orbitals, and a tensor whose terms meet).

Tolerance: an element is a sum of at most ~100 products in FP64, in an order of
its own, so the two sides differ by at most about 100 eps of the sum of its
absolute terms; 1e-13 of the largest element covers that with room for the
difference between the two."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import (kanamori_tensor, oracle_model, product_model, random_hubbard_params, ring_hopping,
                          siam_params, torus_hopping)

pytestmark = pytest.mark.gpu


def _hubbard(t, U):
    n = t.shape[0]
    return "hubbard", dict(Ns=n, t=t, U=np.full(n, U), xmu=np.full(n, U / 2))


def _siam(Ns, ml, seed, tensor=None):
    p = siam_params(Ns, ml, np.random.default_rng(seed), mu=1.3, h0_offdiag=0.2 if ml > 1 else 0.0)
    if ml not in (1, 3):
        p["U"] = kanamori_tensor(ml, 4.0, 0.7)
    if tensor is not None:
        p["U"] = tensor
    return "siam", p


def _general_tensor(ml, seed):
    """Symmetric under exchange of the two electrons, otherwise without structure."""
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(ml, ml, ml, ml))
    u = u + np.transpose(u, (1, 0, 3, 2))
    u = u + np.transpose(u, (2, 3, 0, 1))
    return np.broadcast_to(0.1 * u, (2, 2) + u.shape).copy()


CASES = {
    "ring9": (_hubbard(ring_hopping(9), 4.0), (5, 4)),
    "one row": (_hubbard(torus_hopping(2, 5, 1.0, -0.3), 3.0), (0, 5)),
    "one column": (_hubbard(torus_hopping(2, 5, 1.0, -0.3), 3.0), (5, 10)),
    "two rounds": (_hubbard(torus_hopping(1, 13), 3.0), (1, 6)),  # 13 x 1716
    "two rounds, columns": (("hubbard", random_hubbard_params(13, np.random.default_rng(2))), (6, 2)),  # 1716 x 78
    "two lines": (_siam(15, 1, 3), (2, 6)),  # 105 x 5005
    "two lines, columns": (_siam(15, 1, 4), (6, 2)),
    "two lines, three orbitals": (_siam(15, 3, 5), (2, 6)),
    "two orbitals": (_siam(8, 2, 6), (4, 3)),
    "three orbitals": (_siam(9, 3, 7), (4, 5)),
    "three orbitals, few electrons": (_siam(9, 3, 8), (1, 2)),
    "four orbitals": (_siam(8, 4, 9), (4, 4)),
    "general tensor": (_siam(8, 3, 10, _general_tensor(3, 11)), (4, 4)),
    "general cross term": (("hubbard", random_hubbard_params(9, np.random.default_rng(12))), (4, 5)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_line_passes_match_oracle(name):
    import edlib_amd as ea
    (kind, p), (nup, ndn) = CASES[name]
    ctx = ea.Context(0)
    ctx.set_model(product_model(kind, p))
    n = ctx.set_sector(nup, ndn)
    ctx.hv_variant = 1
    srs = eo.SRS(oracle_model(kind, p), nup, ndn)
    rng = np.random.default_rng(1)
    v, w0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    ref = srs.av(v)
    tol = 1e-13 * max(1.0, np.abs(ref).max())
    assert np.abs(ctx.av(v) - ref).max() <= tol
    # accumulated input in place (w = H v + w)
    assert np.abs(ctx.av(v, w0, clear=False) - (ref + w0)).max() <= tol
    # accumulated input in another buffer, and the shares of <v, w>
    v /= np.linalg.norm(v)
    nl, a, b = ctx.lanczos(v, 6)
    nlo, ao, bo = srs.lanczos(v, 6)
    assert nl == nlo
    assert np.abs(a[:nl] - ao[:nl]).max() <= 1e-10 and np.abs(b[:nl] - bo[:nl]).max() <= 1e-10
    ctx.close()


@pytest.mark.parametrize("case", ["kanamori", "anderson"])
def test_line_pass_operands_are_bit_identical_alone_and_grouped(case):
    """Runs on two sectors of different line lengths (256 states and more of
    either spin), alone and together: the launch's work-group size and LDS are
    then another sector's."""
    from edlib_amd.batch import Batch
    kind, p = _siam(12, 3, 21) if case == "kanamori" else _siam(12, 1, 22)
    m = product_model(kind, p)
    rng = np.random.default_rng(5)
    nl = 8
    secs = [(6, 6), (4, 5), (7, 4), (6, 6)]
    got = []
    for groups in ([[0], [1], [2], [3]], [[0, 1, 2, 3]]):
        rng = np.random.default_rng(5)
        vs = []
        res = {}
        b = Batch(0)
        sid = {s: b.add_sector(m, *s) for s in sorted(set(secs))}
        for s in secs:
            v = rng.uniform(-1, 1, sid[s][1])
            vs.append(v / np.linalg.norm(v))
        for g in groups:
            jobs = {q: b.submit_lanczos(sid[secs[q]][0], vs[q], nl) for q in g}
            b.run()
            for q, j in jobs.items():
                res[q] = b.lanczos_result(j, nl)
        b.close()
        got.append(res)
    for q in range(len(secs)):
        assert got[0][q][0] == got[1][q][0]
        assert np.array_equal(got[0][q][1], got[1][q][1]) and np.array_equal(got[0][q][2], got[1][q][2])
