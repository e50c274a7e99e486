"""Launches of a single-sector Lanczos run, on the host with a stand-in for the
device: one for a small sector, two a step for an ordinary one, the scales and
the shares of <v, w> in a launch each where the sector has many rows."""
from tests import fake_device


def test_launches_of_a_run(tmp_path):
    fake_device.run(tmp_path, """
    for ns, sec, variant, per_step in ((12, (6, 6), 0, 2), (14, (5, 3), 0, 2), (14, (5, 4), 0, 3), (14, (6, 2), 0, 3),
                                       (14, (7, 4), 0, 4), (15, (7, 1), 0, 4), (15, (7, 1), 1, 3), (16, (8, 1), 1, 4),
                                       (8, (4, 4), 0, 0)):
        ctx = ea.Context(0)
        ctx.set_model(hubbard(ns))
        n = ctx.set_sector(*sec)
        ctx.hv_variant = variant
        before = counts()["launches"]
        ctx.lanczos(np.full(n, n ** -0.5), 10)
        got = counts()["launches"] - before
        assert got == (10 * per_step or 1), (ns, sec, variant, got)
        ctx.close()
    """)
