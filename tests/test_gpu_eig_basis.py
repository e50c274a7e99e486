"""The single-sector eigensolver's orthogonalisation at the edges of its
column groups (12 columns in registers): bases of 11, 12, 13, 24, 25 and 47
vectors, odd sector sizes, and a sector whose Krylov space is exhausted inside
one cycle (atomic limit), where the norm by difference is replaced by the
exact form.

Tolerance: eigenvalues to 1e-10 of the largest (the solver's own target),
residuals and orthogonality to 1e-8, the square root of that."""
import numpy as np
import pytest

from tests.models import product_model, siam_params

pytestmark = pytest.mark.gpu


def _check(ctx, ev, vecs, n):
    scale = max(1.0, np.abs(ev).max())
    for k in range(len(ev)):
        r = ctx.av(np.ascontiguousarray(vecs[:, k])) - ev[k] * vecs[:, k]
        assert np.linalg.norm(r) <= 1e-8 * scale
    g = vecs.T @ vecs
    assert np.abs(g - np.eye(len(ev))).max() <= 1e-8


@pytest.mark.parametrize("nev,ncv", [(1, 4), (4, 11), (4, 12), (4, 13), (6, 24), (6, 25), (8, 47)])
def test_lowest_pairs_match_dense(nev, ncv):
    import edlib_amd as ea
    p = siam_params(7, 1, np.random.default_rng(3))
    m = product_model("siam", p)
    ctx = ea.Context(0)
    ctx.set_model(m)
    n = ctx.set_sector(3, 2)  # 35 x 21 = 735 states
    H = np.zeros((n, n))
    e = np.zeros(n)
    for i in range(n):
        e[:] = 0.0
        e[i] = 1.0
        H[:, i] = ctx.av(e)
    ref = np.linalg.eigvalsh(0.5 * (H + H.T))[:nev]
    ev, vecs, _ = ctx.eigsh(nev, ncv)
    assert len(ev) == nev
    assert np.abs(ev - ref).max() <= 1e-10 * np.abs(ref).max()
    _check(ctx, ev, vecs, n)
    ctx.close()


def test_exhausted_krylov_space():
    """Six independent sites at half filling: the sector's 400 states have four
    distinct energies, so the fifth basis vector is rounding noise."""
    import edlib_amd as ea
    U = 4.0
    ctx = ea.Context(0)
    ctx.set_model(ea.HubbardModel(6, np.zeros((6, 6)), np.full(6, U), np.full(6, U / 2)))
    n = ctx.set_sector(3, 3)
    ev, vecs, _ = ctx.eigsh(4)
    assert len(ev) >= 1 and np.all(np.isfinite(ev))
    levels = -6 * U / 2 + U * np.arange(4)
    assert abs(ev[0] - levels[0]) <= 1e-10 * abs(levels[0])
    assert all(np.abs(levels - x).min() <= 1e-8 for x in ev)
    _check(ctx, ev, vecs, n)
    ctx.close()
