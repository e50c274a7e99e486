"""Green's-function start vectors of a batch (one launch for all runs of a
submission, chunks of 4096 elements) against the single-sector operator on the
same eigenvector: one orbital and a pair, both spins, create and annihilate,
target sectors shorter and longer than a chunk.

The gathered elements are the eigenvector's up to a sign (a sum of two for a
pair), so the squared norms agree to n eps; the first Lanczos coefficients to
1e-10 of the spectrum's scale."""
import numpy as np
import pytest

from tests.models import product_model, siam_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,sec", [(6, (2, 3)), (8, (4, 4)), (9, (4, 5))])
def test_start_vectors_match_single_sector_operator(ns, sec):
    import edlib_amd as ea
    from edlib_amd.batch import Batch
    m = product_model("siam", siam_params(ns, 3, np.random.default_rng(ns)))
    b = Batch(0)
    sids = {}
    for d in ((0, 0), (1, 0), (-1, 0), (0, 1), (0, -1)):
        s = (sec[0] + d[0], sec[1] + d[1])
        sids[s] = b.add_sector(m, *s)[0]
    jid = b.submit_eig(sids[sec], 2, 7)
    b.run()
    ev, vecs = b.eig_result(jid, vectors=True)
    reqs, meta = [], []
    for k in range(2):
        for spin in (0, 1):
            for ann in (0, 1):
                dst = list(sec)
                dst[spin] += -1 if ann else 1
                for orb2 in (-1, 2):
                    reqs.append((jid, k, spin * ns, ann, sids[tuple(dst)], orb2 + spin * ns if orb2 >= 0 else -1))
                    meta.append((k, spin, ann, tuple(dst), orb2))
    nl = 4
    ids = b.submit_gf(reqs, nl)
    b.run()
    n2 = b.lanczos_norm2(ids)
    ctx = ea.Context(0)
    ctx.set_model(m)
    for jid2, x2, (k, spin, ann, dst, orb2) in zip(ids, n2, meta):
        v = np.ascontiguousarray(vecs[:, k])
        _, x = ctx.adag(sec, spin * ns, bool(ann), v)
        if orb2 >= 0:
            _, y = ctx.adag(sec, orb2 + spin * ns, bool(ann), v)
            x = x + y
        assert abs(x2 - x @ x) <= 1e-11
        ctx.set_sector(*dst)
        _, a, be = ctx.lanczos(x / np.linalg.norm(x), nl)
        _, ab, bb = b.lanczos_result(jid2, nl)
        scale = max(1.0, np.abs(a).max())
        assert np.abs(a - ab).max() <= 1e-10 * scale and np.abs(be - bb).max() <= 1e-10 * scale
    ctx.close()
    b.close()
