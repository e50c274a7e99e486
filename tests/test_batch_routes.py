"""Which H*v a batch's Lanczos operands take, by the launches of a steady sweep of
three runs on one sector, on the host with a stand-in for the device: the line
passes are two kernels for all three, the multi-operand rows kernel is one, the
rows kernel one each, the grouped kernel one; the update's kernels are the same
ones for all."""
from tests import fake_device


def test_launches_of_a_sweep(tmp_path):
    fake_device.run(tmp_path, """
    def siam(ns, ml):
        return product_model("siam", siam_params(ns, ml, np.random.default_rng(1), mu=1.3))

    def torus(tp=0.0):
        return hubbard(14, torus_hopping(2, 7, 1.0, tp))

    def sweep(m, sec):
        b = Batch(0)
        b.set_graphs(False)
        sid, n = b.add_sector(m, *sec)
        for _ in range(3):
            b.submit_lanczos(sid, np.full(n, n ** -0.5), 50)
        b.step(3)
        before = counts()["launches"]
        b.step(1)
        got = counts()["launches"] - before
        b.close()
        return got

    grouped = sweep(hubbard(8), (4, 4))
    for m, sec, hv in ((siam(13, 1), (6, 6), 1), (siam(14, 1), (5, 5), 1), (siam(13, 3), (7, 6), 2),
                       (product_model("hubbard", random_hubbard_params(13, np.random.default_rng(1))), (6, 6), 2),
                       (torus(), (5, 6), 2), (torus(), (6, 5), 3), (torus(-0.3), (5, 5), 2)):
        assert sweep(m, sec) - grouped + 1 == hv, (sec, hv, sweep(m, sec), grouped)
    """)
