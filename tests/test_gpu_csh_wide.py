"""Transforms of several wavefronts (lengths 1024 to 4096) in the large grids'
passes: x and y direction, columns side by side and interleaved, one and two rows
a workgroup, both equations, and the x pass's shapes, against the oracle.

Bars: one right-hand side 1e-13, two steps 1e-12 (as the other grids' tests)."""
import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _rhs, _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("screened", [False, True])
@pytest.mark.parametrize("nx,ny", [(2048, 1024), (1024, 2048), (4096, 512), (128, 4096), (4096, 1024)])
def test_rhs_vs_oracle(nx, ny, screened):
    print(f"wide {nx}x{ny} screened {screened}", flush=True)
    w, nu = _noise(nx, ny, nx + 2 * ny), 1e-3
    nh = nx // 2 + 1
    f = T.derive2css(nx, ny, nh, 1.5, nu, w, 3.0) if screened else T.derive2csh(nx, ny, nh, nu, w)
    assert rel_l2(f, _rhs(w, nx, nu, screened)) < 1e-13


@pytest.mark.parametrize("nx,ny", [(1024, 1024), (2048, 512), (4096, 512)])
def test_x_shapes_vs_oracle(nx, ny):
    w, nu, dt = _noise(nx, ny, 11), 1e-3, 1e-5
    want = _steps(w, nx, nu, dt, 2, T.SCHEME_AB2, False)
    s = T.CshSolver(nx, ny, nu, dt, T.SCHEME_AB2)
    for k in range(T.lib().tara_csh_num_xshapes()):
        try:
            s.set_xshape(k)
        except T.TaraError:
            continue
        print(f"wide {nx}x{ny} x shape {k}", flush=True)
        s.upload(w)
        s.advance(2)
        assert rel_l2(s.download(), want) < 1e-12, k
    s.close()
