"""A context's calls allocate no pinned host memory (up to a millisecond each):
they borrow it from a store that the process's first context fills, and contexts
hold none, however many there are.  On the host, with a stand-in for the
device."""
from tests import fake_device


def test_calls_allocate_no_pinned_memory(tmp_path):
    fake_device.run(tmp_path, """
    def calls(ctx, eig=False):
        ctx.set_model(hubbard(8))
        n = ctx.set_sector(4, 4)
        before = counts()["host_allocs"]
        v = np.full(n, n ** -0.5)
        ctx.cf_eval(1j * np.arange(1, 2001), 1.0, 40, 1, 1.0, np.zeros(40), np.ones(41))
        ctx.static_observables(v, 8)
        ctx.lanczos(v, 500)
        try:
            if eig:
                ctx.eigsh(8, 47, maxitr=2)  # (no kernels run: the projected matrix is garbage)
        except ea.EdhError:
            pass
        return counts()["host_allocs"] - before

    a = ea.Context(0)
    assert counts()["host_allocs"] == 1
    assert calls(a, True) == 0
    many = [ea.Context(0) for _ in range(5)]  # while the first one lives
    assert sum(calls(c) for c in many) == 0 and counts()["host_allocs"] == 1
    for c in many:
        c.close()
    # a mesh beyond the usual sizes: its buffer is kept, one too large to keep is given back
    z = lambda n: 1j * np.arange(1, n + 1)
    for n, allocs, kept in ((100000, 1, 1), (100000, 0, 0), (3000000, 1, 0)):
        x = z(n)
        c = ea.Context(0)
        b4 = counts()
        c.cf_eval(x, 1.0, 4, 1, 1.0, np.zeros(4), np.ones(5))
        c.close()
        assert counts()["host_allocs"] - b4["host_allocs"] == allocs
        assert counts()["live"] - b4["live"] == kept, (n, counts()["live"] - b4["live"])
    """)


def test_concurrent_calls_borrow_a_buffer_each(tmp_path):
    """Calls on eight threads, each with a context, hold at most a buffer per
    thread, and every one comes back."""
    fake_device.run(tmp_path, """
    import threading
    def work():
        ctx = ea.Context(0)
        for _ in range(200):
            ctx.cf_eval(np.full(500, 1j), 1.0, 3, 1, 1.0, np.zeros(3), np.ones(4))
        ctx.close()
    th = [threading.Thread(target=work) for _ in range(8)]
    [t.start() for t in th]
    [t.join() for t in th]
    n = counts()["host_allocs"]
    assert 1 <= n <= 8
    many = [threading.Thread(target=work) for _ in range(8)]
    [t.start() for t in many]
    [t.join() for t in many]
    assert counts()["host_allocs"] <= 8 and counts()["live"] == counts()["host_allocs"]
    """)
