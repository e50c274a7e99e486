"""Batched Lanczos operands on the line passes (csrc/hv_lines.hip), which sectors
of 2.5 million states and more take where the line passes beat the single pass
(with 32-bit entries from 28 hops a state on): a 13-site sector of the
three-orbital impurity (row tiles with slots that hold no row) and a 14-site
torus with t and t' (no impurity terms), alone and up to five together, one of
them with a start vector that ends its run at the first step.

A single context makes the same choice by the same rule from that size on, and
says which variant it took; tests/test_batch_routes.py counts the batch's
launches.

Tolerances: alone and grouped bit for bit; against the single-sector run and
the oracle 1e-10 of the spectrum's scale over 8 steps (another order of sums, as
in the other Lanczos tests)."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, siam_params, torus_hopping

pytestmark = pytest.mark.gpu
NL = 8


def _spin_vector(model, ns, nel):
    """An eigenvector of one spin's hopping and levels without interaction."""
    import ctypes

    from edlib_amd import _lib
    L = _lib.lib()
    rows, nnz = ctypes.c_int64(), ctypes.c_int64()
    _lib.check(L.edh_sector_csr(model.handle, nel, 0, 0, ctypes.byref(rows), ctypes.byref(nnz), None, None, None))
    rp, col, val = np.zeros(rows.value + 1, np.int32), np.zeros(nnz.value, np.int32), np.zeros(nnz.value)
    ip = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))
    dp = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    _lib.check(L.edh_sector_csr(model.handle, nel, 0, 0, ctypes.byref(rows), ctypes.byref(nnz), ip(rp), ip(col), dp(val)))
    d = np.zeros(rows.value)
    _lib.check(L.edh_sector_diagonal(model.handle, nel, 0, dp(d)))
    h = np.diag(d)
    for r in range(rows.value):
        h[r, col[rp[r]:rp[r + 1]]] += val[rp[r]:rp[r + 1]]
    return np.linalg.eigh(h)[1][:, 0]


def _on_lines(m, sec):
    """Checks the route and returns the context."""
    import edlib_amd as ea
    ctx = ea.Context(0)
    ctx.set_model(m)
    n = ctx.set_sector(*sec)
    dup, ddn = ctx.sector_info()[:2]
    assert n >= 2500000 and max(dup, ddn) <= 4096 and ctx.hv_variant == 1
    return ctx, n


def _runs(b, sid, vs, groups):
    res = {}
    for g in groups:
        jobs = {q: b.submit_lanczos(sid, vs[q], NL) for q in g}
        b.run()
        for q, j in jobs.items():
            res[q] = b.lanczos_result(j, NL)
    return res


@pytest.mark.parametrize("case", ["kanamori", "torus", "free"])
def test_grouped_operands(case):
    from edlib_amd.batch import Batch
    if case == "kanamori":
        kind, sec, p = "siam", (7, 6), siam_params(13, 3, np.random.default_rng(21), mu=1.3, h0_offdiag=0.2)
    else:  # free: without interaction products of one spin's eigenvectors are eigenvectors
        u = 0.0 if case == "free" else 4.0
        kind, sec, p = "hubbard", (5, 5), dict(Ns=14, t=torus_hopping(2, 7, 1.0, -0.3), U=np.full(14, u),
                                               xmu=np.full(14, 0.7))
    m = product_model(kind, p)
    ctx, n = _on_lines(m, sec)
    rng = np.random.default_rng(5)
    vs = [rng.uniform(-1, 1, n) for _ in range(5)]
    vs = [v / np.linalg.norm(v) for v in vs]
    if case == "free":
        x = _spin_vector(m, 14, 5)
        vs[1] = np.kron(x, x)
    b = Batch(0)
    sid = b.add_sector(m, *sec)[0]
    alone = _runs(b, sid, vs, [[q] for q in range(5)])
    for groups in ([[0, 1, 2, 3, 4]], [[3, 1], [0, 2, 4]]):
        got = _runs(b, sid, vs, groups)
        for q in range(5):
            assert got[q][0] == alone[q][0]
            assert np.array_equal(got[q][1], alone[q][1]) and np.array_equal(got[q][2], alone[q][2])
    b.close()
    for q in range(5):
        nl, a, be = alone[q]
        assert nl == (1 if case == "free" and q == 1 else NL)
        n1, a1, b1 = ctx.lanczos(vs[q], NL)
        scale = max(1.0, np.abs(a1).max())
        assert n1 == nl and np.abs(a - a1).max() <= 1e-10 * scale and np.abs(be - b1)[:nl].max() <= 1e-10 * scale
    ctx.close()
    srs = eo.SRS(oracle_model(kind, p), *sec)
    no, ao, bo = srs.lanczos(vs[0], NL)
    scale = max(1.0, np.abs(ao).max())
    assert no == NL and np.abs(alone[0][1] - ao).max() <= 1e-10 * scale
    assert np.abs(alone[0][2] - bo).max() <= 1e-10 * scale
