"""A submission to the batch that fails part-way (any of its allocations)
leaves no process behind, no memory in use, and an engine that goes on: on the
host, with a stand-in for the device (tests/fake_device.py)."""
import pytest

from tests import fake_device

SETUP = """
    b = Batch(0)
    m = hubbard(6)
    sid = {s: b.add_sector(m, *s)[0] for s in ((2, 1), (3, 1), (1, 1), (2, 2), (3, 3))}
    eig = b.submit_eig(sid[2, 1], 2, 120)  # the whole sector: solved on the host
    reqs = [(eig, 0, 0, 0, sid[3, 1]), (eig, 0, 0, 1, sid[1, 1]), (eig, 1, 7, 0, sid[2, 2]), (eig, 1, 0, 0, sid[3, 1], 2)]
"""


@pytest.mark.parametrize("what", ["b.submit_gf(reqs, 10)", "b.submit_eig(sid[3, 3], 2, 8)",
                                  "b.submit_lanczos(sid[3, 3], np.ones(400), 10)"])
def test_failed_submission_leaves_nothing(tmp_path, what):
    out = fake_device.run(tmp_path, SETUP + """
    used, failed = b.memory(), 0
    for n in range(1, 100):
        fake.fake_fail_alloc(n)
        try:
            %s
        except ea.EdhError as e:
            failed += 1
            assert b.memory() == used, (n, b.memory(), used)
            before = counts()["launches"]
            fake.fake_fail_alloc(0)
            assert b.step(1) == 0, n  # no process is there ...
            assert counts()["launches"] == before  # ... and nothing is launched
            continue
        break
    fake.fake_fail_alloc(0)
    assert b.step(1) > 0  # the submission that went through
    print(failed)
    """ % what)
    assert int(out) >= 1


def test_next_submission_does_not_report_the_error_again(tmp_path):
    """The runtime keeps an error until it is asked for; a failed submission
    must not show up in the check of another request's launch."""
    fake_device.run(tmp_path, SETUP + """
    for submit in (lambda: b.submit_gf(reqs, 10), lambda: b.submit_eig(sid[3, 3], 2, 8),
                   lambda: b.submit_lanczos(sid[3, 3], np.ones(400), 10), lambda: b.add_sector(m, 4, 4)):
        fake.fake_fail_alloc(1)
        try:
            submit()
            raise SystemExit("the submission did not fail")
        except ea.EdhError:
            pass
        fake.fake_fail_alloc(0)
        b.submit_gf(reqs, 10)
    """)
