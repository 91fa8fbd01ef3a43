"""3D grids whose live kx tiles reach past Nh, where a step transforms padding
columns of the buffer that host copies are packed in: steps between downloads and
uploads give the bits of steps alone, and agree with the oracle.

Bar: 1e-12 relative L2 per field (as the other 3D tests)."""
import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_mhd_live import PI2, _oracle, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,scale,steps", [
    (16, 256, 256, (1.0, 1.0, 1.0), 2),   # Nh = 9 in 16, all kx alive in the 2 pi box
    (32, 16, 64, (3.0, 4.0, 9.0), 4),
    (16, 16, 16, (3.0, 4.0, 9.0), 4),
])
def test_steps_between_host_copies(nx, ny, nz, scale, steps):
    print(f"mhd padding {nx}x{ny}x{nz} box x {scale}", flush=True)
    box = [PI2 * a for a in scale]
    mu, eta, dt = 2e-3, 1e-3, 1e-5
    prm = T.MhdParams(*box, mu, eta, 10.0, dt)
    st = _state(nx, ny, nz, nx)
    ref = _oracle(st, nx, box, mu, eta, dt, steps)
    alone = T.MhdSolver(nx, ny, nz, prm)
    alone.upload(st)
    for _ in range(steps):  # the same calls: a call's later steps round differently
        alone.advance(1)
    want = alone.download()
    alone.close()
    s = T.MhdSolver(nx, ny, nz, prm)
    s.upload(_state(nx, ny, nz, 7))
    s.advance(1)
    s.download()
    s.upload(st)
    for _ in range(steps):
        s.advance(1)
        got = s.download()  # packs the state over the fluxes' padding
    s.close()
    for k in range(8):
        assert rel_l2(want[k], ref[k]) < 1e-12, k
        assert np.array_equal(got[k], want[k]), k


def test_many_steps_after_a_host_copy():
    """Leftovers in the padding, transformed in place, would pass the largest double
    after some 500 steps."""
    n = 16
    prm = T.MhdParams(3 * PI2, 4 * PI2, 9 * PI2, 2e-3, 1e-3, 10.0, 1e-6)
    s = T.MhdSolver(n, n, n, prm)
    s.upload(_state(n, n, n, 1))
    s.advance(1)
    s.download()
    s.advance(999)
    got = s.download()
    s.close()
    t = T.MhdSolver(n, n, n, prm)
    t.upload(_state(n, n, n, 1))
    t.advance(1)
    t.advance(999)
    for a, b in zip(got, t.download()):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
    t.close()
