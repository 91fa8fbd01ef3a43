"""The 3D stepper carries only the modes the dealiasing leaves alive through its
forward passes, and within one advance call only their part of the inverse
passes: checked against the oracle on states with every mode present, over
boxes that leave all, some (ragged tiles), or hardly any modes alive, on unequal
sides, for several steps in one call and split over calls.

Bar: 1e-12 relative L2 per field (different FFT factorisations, a few steps)."""
import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2

pytestmark = pytest.mark.gpu

PI2 = 2 * np.pi


def _state(nx, ny, nz, seed):
    """Real-space white noise around a uniform state: no mode is zero."""
    rng = np.random.default_rng(seed)
    mean = (1.0, 0.0, 0.0, 0.0, 2.0, 0.3, -0.2, 0.1)
    return [O.r2c(np.asfortranarray(m + 0.02 * rng.standard_normal((nx, ny, nz)))) for m in mean]


def _oracle(st, nx, box, mu, eta, dt, steps):
    hist = [np.zeros_like(a, order="F") for a in st]
    for _ in range(steps):
        f = O.derive3com(st, nx, *box, mu, eta, 10.0)
        st = O.ab3com(st, hist, f, nx, dt)
        hist = f
    return st


@pytest.mark.parametrize("nx,ny,nz,scale", [
    (16, 16, 16, (1.0, 1.0, 1.0)),      # 2 pi box
    (64, 32, 16, (1.0, 1.0, 1.0)),      # every ky, kz of one side alive, kx cut
    (32, 64, 32, (1.0, 2.0, 0.5)),      # an ellipsoid of modes
    (32, 16, 64, (3.0, 4.0, 9.0)),      # every mode alive
    (32, 32, 16, (0.2, 0.15, 0.3)),     # a handful of modes alive
    (32, 16, 16, (0.01, 0.01, 0.01)),   # only k = 0 alive
    (16, 128, 32, (0.7, 1.0, 1.3)),
])
def test_live_modes_vs_oracle(nx, ny, nz, scale):
    print(f"mhd live modes {nx}x{ny}x{nz} box x {scale}", flush=True)
    box = [PI2 * a for a in scale]
    mu, eta, dt, steps = 2e-3, 1e-3, 1e-5, 4
    st = _state(nx, ny, nz, nx + ny)
    prm = T.MhdParams(*box, mu, eta, 10.0, dt)
    f = T.derive3com(nx, ny, nz, nx // 2 + 1, prm, st)
    want = O.derive3com(st, nx, *box, mu, eta, 10.0)
    for k in range(8):
        assert np.linalg.norm(f[k] - want[k]) <= 1e-12 * max(np.linalg.norm(want[k]), 1.0), k
    ref = _oracle(st, nx, box, mu, eta, dt, steps)
    for split in ((steps,), (1, steps - 1), (1,) * steps):
        s = T.MhdSolver(nx, ny, nz, prm)
        s.upload(_state(nx, ny, nz, 99))  # replaced below: nothing of it may remain
        s.advance(1)
        s.upload(st)
        for k in split:
            s.advance(k)
        got = s.download()
        s.close()
        for k in range(8):
            assert rel_l2(got[k], ref[k]) < 1e-12, (split, k)
