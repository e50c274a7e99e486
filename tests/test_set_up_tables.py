"""Setting a sector uploads only the tables of the H*v variant that it takes;
the two passes' tables follow when that variant is asked for, once.  On the
host, with a stand-in for the device."""
from tests import fake_device


def test_two_pass_tables_come_with_their_variant(tmp_path):
    out = fake_device.run(tmp_path, """
    kan = product_model("siam", siam_params(9, 3, np.random.default_rng(1), mu=1.3))
    kan12 = product_model("siam", siam_params(12, 3, np.random.default_rng(1), mu=1.3))
    # (model, sector, variant of its own): lines, lines with impurity terms,
    # tiles (a spin of 12,870 states), and a sector that takes the line passes
    for m, sec, own in ((hubbard(8), (4, 4), 0), (kan, (4, 4), 0), (hubbard(16), (8, 1), 0), (kan12, (6, 6), 1)):
        ctx = ea.Context(0)
        ctx.set_model(m)
        a = counts()
        ctx.set_sector(*sec)
        b = counts()
        assert ctx.hv_variant == own
        assert b["allocs"] - a["allocs"] == 1
        ctx.hv_variant = 0
        assert counts() == b
        ctx.hv_variant = 1
        c = counts()
        assert c["allocs"] - b["allocs"] == (0 if own else 1) and ctx.hv_variant == 1
        for v in (0, 1, -1, 1):
            ctx.hv_variant = v
        assert counts()["allocs"] == c["allocs"]
        # with its tables there the variant launches its two kernels
        n = ctx.sector_info()[0] * ctx.sector_info()[1]
        before = counts()["launches"]
        ctx.av(np.ones(n))
        assert counts()["launches"] == before + 2
        # the next sector starts without them
        ctx.set_sector(1, 1)
        d = counts()["allocs"]
        ctx.hv_variant = 1
        assert counts()["allocs"] == d + 1
        ctx.close()
        print(counts()["live"])
    """)
    live = [int(x) for x in out.split()]
    assert live == [live[0]] * len(live)  # nothing stays with the device


def test_variant_fixed_by_the_environment(tmp_path):
    fake_device.run(tmp_path, """
    import os
    ctx = ea.Context(0)
    ctx.set_model(hubbard(8))
    libc = ctypes.CDLL(None)
    libc.setenv(b"EDH_HV_VARIANT", b"1", 1)
    ctx.set_sector(4, 4)
    assert ctx.hv_variant == 1
    before = counts()["launches"]
    ctx.av(np.ones(4900))
    assert counts()["launches"] == before + 2
    libc.unsetenv(b"EDH_HV_VARIANT")
    ctx.set_sector(4, 4)
    assert ctx.hv_variant == 0
    libc.setenv(b"EDH_HV_VARIANT", b"1", 1)  # between the sector and the choice
    ctx.hv_variant = -1
    before = counts()["launches"]
    ctx.av(np.ones(4900))
    assert counts()["launches"] == before + 2
    """)
