"""Small grids whose last workgroup of columns is partly empty (Nh is odd): its
unused threads must read nothing that another workgroup writes during the pass.
Every number of columns a workgroup, with one, two and four groups a column, in a
single run and in batches: the state after several in-place steps agrees with the
oracle, and is the same bit for bit when the run is repeated.

Bar: a few steps 1e-12 (as the other grids' tests)."""
import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [T.SCHEME_AB2, T.SCHEME_RK4])
@pytest.mark.parametrize("nx,ny", [(64, 16), (128, 32), (64, 64), (256, 128), (128, 256)])
def test_steps_repeat(nx, ny, scheme):
    print(f"last column {nx}x{ny}", flush=True)
    w, nu, dt = _noise(nx, ny, nx + 3 * ny), 1e-3, 1e-5
    got = []
    for _ in range(4):
        s = T.CshSolver(nx, ny, nu, dt, scheme)
        s.upload(w)
        for k in (1, 1, 4):  # each call's last pass runs one group a column
            s.advance(k)
        got.append(s.download())
        s.close()
    assert rel_l2(got[0], _steps(w, nx, nu, dt, 6, scheme, False)) < 1e-12
    for g in got[1:]:
        assert np.array_equal(g, got[0])


@pytest.mark.parametrize("n,runs", [(64, 8), (64, 100), (128, 40)])
def test_batches_repeat(n, runs):
    print(f"last column {runs} x {n}", flush=True)
    dt, w = 1e-5, _noise(n, n, n)
    want = _steps(w, n, 1e-3, dt, 4, T.SCHEME_RK4, False)
    e = T.Ensemble([n] * runs, [1e-3] * runs, dt, T.SCHEME_RK4)
    for r in range(runs):
        e.upload(r, w)
    e.advance(4)
    e.sync()
    first = e.download(0)
    assert rel_l2(first, want) < 1e-12
    for r in range(1, runs):
        assert np.array_equal(e.download(r), first), r
    e.close()
