"""Which H*v variant a sector takes for w = H v and for w = H v + w in place
(two kernels where it takes the two passes), on the host with a stand-in for
the device.  The sectors are ones where the other variant, or the same variant
for both forms, was measured slower on an MI355X (single pass : two passes,
us), and ones on the two passes' side of each line."""
from tests import fake_device


def test_choice(tmp_path):
    fake_device.run(tmp_path, """
    def siam(ns, ml):
        return product_model("siam", siam_params(ns, ml, np.random.default_rng(1), mu=1.3))

    def torus(a, b, tp=0.0):
        return hubbard(a * b, torus_hopping(a, b, 1.0, tp))

    def dimers(ns, k):  # k neighbours, two hopping values
        t = np.zeros((ns, ns))
        for i in range(ns):
            for r in range(1, k + 1):
                t[i, (i + r) % ns] = t[(i + r) % ns, i] = 0.6 if r % 2 == 0 else 1.0
        return hubbard(ns, t)

    dis = lambda ns: product_model("hubbard", random_hubbard_params(ns, np.random.default_rng(1)))
    for m, sec, plain, in_place in (
        (torus(3, 4, -0.3), (6, 4), 0, 0),    # 17.1 : 18.9, in place 17.8 : 23.1
        (torus(3, 4, -0.3), (6, 6), 1, 1),    # 29.5 : 23.4, 31.0 : 28.8
        (torus(3, 4), (6, 6), 0, 0),          # 18.2 : 19.7
        (siam(12, 3), (6, 6), 1, 1),          # 27.7 : 22.5, 28.8 : 27.6
        (dis(12), (6, 4), 0, 0),              # 18.7 : 19.5, 19.5 : 23.7
        (dis(13), (4, 4), 1, 1),              # 26.8 : 20.4, 27.6 : 23.8
        (siam(13, 1), (6, 6), 1, 0),          # 45.5 : 41.7, 49.4 : 54.3
        (siam(14, 1), (5, 6), 1, 0),          # 91.6 : 79.6 on three streams, in place 98 : 111
        (siam(14, 1), (6, 5), 0, 0),          # 74.7 : 76.7 on three streams
        (torus(2, 7), (8, 5), 0, 0),          # 74.6 : 82.1 on three streams
        (torus(2, 7), (5, 6), 1, 0),          # 89.0 : 83.9 on three streams
        (siam(14, 1), (7, 7), 1, 1),          # 175 : 121, 188 : 169
        (siam(14, 3), (7, 7), 1, 1),          # 378 : 194, 394 : 241
        (torus(2, 7), (5, 5), 0, 0),          # 54.3 : 54.4, 59.3 : 70.5
        (torus(2, 7), (7, 7), 1, 0),          # 177 : 156, 191 : 201
        (siam(15, 3), (7, 7), 1, 0),          # 1443 : 1248, 1509 : 1554
        (torus(4, 4), (6, 6), 0, 0),          # 1224 : 1374, 1317 : 1645
        (torus(4, 4), (7, 6), 1, 1),          # 1847 : 1648, 1975 : 1819
        (siam(16, 1), (5, 8), 0, 0),          # 896 : 958, 975 : 1039
        (siam(16, 1), (8, 5), 1, 1),          # 1219 : 909, 1274 : 1014
        (dimers(16, 2), (7, 6), 0, 0),        # 1892 : 2048
    ):
        ctx = ea.Context(0)
        ctx.set_model(m)
        n = ctx.set_sector(*sec)
        assert ctx.hv_variant == plain, (sec, n)
        for want, clear in ((plain, True), (in_place, False)):
            v = ctypes.c_void_p(256)
            before = counts()["launches"]
            rc = ea._lib.lib().edh_av(ctx.handle, v, ctypes.c_void_p(512), n, int(clear), ea.EDH_MEM_DEVICE)
            assert rc == 0
            assert counts()["launches"] - before == 1 + want, (sec, n, clear)
        # a fixed variant holds for both forms
        for var in (0, 1):
            ctx.hv_variant = var
            for clear in (1, 0):
                before = counts()["launches"]
                ea._lib.lib().edh_av(ctx.handle, v, ctypes.c_void_p(512), n, clear, ea.EDH_MEM_DEVICE)
                assert counts()["launches"] - before == 1 + var
        ctx.close()
    """)
