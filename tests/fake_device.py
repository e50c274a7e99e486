"""Runs a script against the library on a host stand-in for the HIP runtime
(tests/host/fake_hip.cpp), in a process of its own: `fake` is the stand-in,
counts() its tallies as a dict."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, %r)
import numpy as np
import edlib_amd as ea
from edlib_amd.batch import Batch
from tests.models import product_model, random_hubbard_params, ring_hopping, siam_params, torus_hopping

def counts():
    a = (ctypes.c_long * 6)()
    fake.fake_counts(a)
    return dict(zip(("allocs", "alloc_bytes", "host_allocs", "launches", "copies", "live"), a))

def hubbard(ns, t=None):
    return ea.HubbardModel(ns, ring_hopping(ns) if t is None else t, np.full(ns, 4.0), np.full(ns, 2.0))
"""


def run(tmp_path, script):
    so = str(tmp_path / "fake_hip.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", "host", "fake_hip.cpp")])
    code = PRELUDE % ROOT + textwrap.dedent(script)
    r = subprocess.run([sys.executable, "-c", code, so], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
