"""A process's first use of a kernel loads the code object it is in, whole: the
autotuner of a large grid, which times the paired x pass among its shapes, must not
load the small grids' y passes with it (some 7 ms, in a call that takes 1 afterwards).

In a process of its own: the first tune() of a 1024^2 solver, whose upload has loaded
the large grids' passes, against the second.  Measured 2.0 / 1.0 ms; 9.3 / 1.0 with
both in one code object.  Bar: 5 times."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import time
import numpy as np
import tara_amd as T
n = 1024
w = np.asfortranarray(np.random.default_rng(0).standard_normal((n // 2 + 1, n)) + 0j)
for rep in range(3):
    s = T.CshSolver(n, n, 1e-3, 1e-4, T.SCHEME_RK4)
    s.upload(w)
    s.sync()
    t = time.perf_counter()
    s.tune()
    print("tune", time.perf_counter() - t, flush=True)
    s.close()
"""


def test_first_tune_loads_little():
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    t = [float(x.split()[1]) for x in r.stdout.splitlines() if x.startswith("tune")]
    print("tune ms:", [round(1e3 * x, 2) for x in t])
    assert t[0] < 5 * min(t[1:])
