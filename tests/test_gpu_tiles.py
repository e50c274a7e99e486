"""The tile pass of H*v (csrc/hv_tiles.hip), which takes the up-spin hopping
where lines do not fit LDS: tiles of 128 rows x 64 columns with a last tile
and a last slab that are not full, an odd number of columns (no 16-byte
access), one column, fewer rows than a tile, and several slabs per XCD.

Tolerance as for the line passes: a sum of at most ~100 FP64 products in
another order differs by at most about 100 eps of its absolute terms, 1e-13 of
the largest element."""
import numpy as np
import pytest

from oracle import edoracle as eo
from tests.models import oracle_model, product_model, random_hubbard_params, ring_hopping, siam_params, torus_hopping

pytestmark = pytest.mark.gpu


def _uniform(t, U):
    n = t.shape[0]
    return "hubbard", dict(Ns=n, t=t, U=np.full(n, U), xmu=np.full(n, U / 2))


CASES = {
    "12870 x 16": (_uniform(torus_hopping(4, 4), 4.0), (8, 1)),
    "24310 x 17": (_uniform(ring_hopping(17), 4.0), (8, 1)),
    "12870 x 1": (("hubbard", random_hubbard_params(16, np.random.default_rng(1))), (8, 0)),
    "16 x 12870": (("hubbard", random_hubbard_params(16, np.random.default_rng(2))), (1, 8)),
    "11440 x 120, impurity": (("siam", siam_params(16, 3, np.random.default_rng(3), mu=1.3, h0_offdiag=0.2)), (7, 2)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_tile_pass_matches_oracle(name):
    import edlib_amd as ea
    (kind, p), (nup, ndn) = CASES[name]
    ctx = ea.Context(0)
    ctx.set_model(product_model(kind, p))
    n = ctx.set_sector(nup, ndn)
    ctx.hv_variant = 1
    srs = eo.SRS(oracle_model(kind, p), nup, ndn)
    rng = np.random.default_rng(4)
    v, w0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    ref = srs.av(v)
    tol = 1e-13 * max(1.0, np.abs(ref).max())
    assert np.abs(ctx.av(v) - ref).max() <= tol
    assert np.abs(ctx.av(v, w0, clear=False) - (ref + w0)).max() <= tol
    # accumulated input in another buffer, and the shares of <v, w>
    v /= np.linalg.norm(v)
    nl, a, b = ctx.lanczos(v, 6)
    nlo, ao, bo = srs.lanczos(v, 6)
    assert nl == nlo
    assert np.abs(a[:nl] - ao[:nl]).max() <= 1e-10 and np.abs(b[:nl] - bo[:nl]).max() <= 1e-10
    ctx.close()
