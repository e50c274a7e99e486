"""A context's first calls allocate no pinned host memory (about a millisecond
each): it is taken when the context is created and goes to the next context
afterwards.  On the host, with a stand-in for the device."""
from tests import fake_device


def test_first_calls_allocate_no_pinned_memory(tmp_path):
    fake_device.run(tmp_path, """
    def calls(ctx):
        ctx.set_model(hubbard(8))
        n = ctx.set_sector(4, 4)
        before = counts()["host_allocs"]
        v = np.full(n, n ** -0.5)
        ctx.cf_eval(1j * np.arange(1, 2001), 1.0, 40, 1, 1.0, np.zeros(40), np.ones(41))
        ctx.static_observables(v, 8)
        ctx.lanczos(v, 500)
        try:
            ctx.eigsh(8, 47)  # (no kernels run: the projected matrix is garbage)
        except ea.EdhError:
            pass
        return counts()["host_allocs"] - before

    a = ea.Context(0)
    assert counts()["host_allocs"] == 1
    assert calls(a) == 0
    b = ea.Context(0)  # while the first one lives: a buffer of its own
    assert counts()["host_allocs"] == 2
    b.close()
    a.close()
    for _ in range(100):  # kept for the next ones
        c = ea.Context(0)
        assert counts()["host_allocs"] == 2
        c.close()
    # a mesh beyond the usual sizes still works, and its memory is given back
    c = ea.Context(0)
    live = counts()["live"]
    c.cf_eval(1j * np.arange(1, 100001), 1.0, 4, 1, 1.0, np.zeros(4), np.ones(5))
    assert counts()["host_allocs"] == 3
    c.close()
    assert counts()["live"] <= live
    """)
