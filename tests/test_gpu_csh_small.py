"""The 2D passes of grids too small to fill the chip: every transform length they
have, several columns and rows per workgroup, a last workgroup that is partly
empty (Nh is odd), both equations, both schemes, batches, and grids on either
side of the rule that chooses them, against the oracle's right-hand side.

Bars: one right-hand side 1e-13, a few steps 1e-12 (as the large grids' tests)."""
import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2

pytestmark = pytest.mark.gpu

# Ny = 16 .. 1024 with 1..8 columns a workgroup; 256 x 1024 is the last grid of
# Ny = 1024 that runs here, 512 x 1024 the first that does not
GRIDS = [(64, 16), (128, 32), (64, 64), (64, 128), (256, 256), (1024, 128), (128, 512), (256, 1024), (512, 1024),
         (2048, 64), (4096, 16)]


def _noise(nx, ny, seed):
    """Spectrum of a random real field, plus entries no real field has (kx = 0
    and Nyquist columns that are not Hermitian)."""
    rng = np.random.default_rng(seed)
    w = O.r2c(np.asfortranarray(rng.standard_normal((nx, ny))))
    w[0, :] += 0.1j * rng.standard_normal(ny) * np.sqrt(nx * ny)
    w[nx // 2, :] += 0.1j * rng.standard_normal(ny) * np.sqrt(nx * ny)
    return np.asfortranarray(w)


def _rhs(w, nx, nu, screened):
    return O.derive2css(w, nx, 1.5, nu, 3.0) if screened else O.derive2csh(w, nx, nu)


def _steps(w, nx, nu, dt, n, scheme, screened):
    old = np.zeros_like(w)
    for _ in range(n):
        if scheme == T.SCHEME_AB2:
            f = _rhs(w, nx, nu, screened)
            w = w + (1.5 * f - 0.5 * old) * dt
            old = f
        else:
            k1 = _rhs(w, nx, nu, screened)
            k2 = _rhs(w + 0.5 * dt * k1, nx, nu, screened)
            k3 = _rhs(w + 0.5 * dt * k2, nx, nu, screened)
            k4 = _rhs(w + dt * k3, nx, nu, screened)
            w = w + dt / 6.0 * (k1 + 2 * k2 + 2 * k3 + k4)
    return w


@pytest.mark.parametrize("screened", [False, True])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_rhs_and_steps_vs_oracle(nx, ny, screened):
    print(f"small grid {nx}x{ny} screened {screened}", flush=True)
    w, nu, dt = _noise(nx, ny, nx + ny), 1e-3, 1e-5
    nh = nx // 2 + 1
    f = T.derive2css(nx, ny, nh, 1.5, nu, w, 3.0) if screened else T.derive2csh(nx, ny, nh, nu, w)
    assert rel_l2(f, _rhs(w, nx, nu, screened)) < 1e-13
    for scheme in (T.SCHEME_AB2, T.SCHEME_RK4):
        want = _steps(w, nx, nu, dt, 3, scheme, screened)
        for split in ((3,), (1, 2)):
            s = T.CshSolver(nx, ny, nu, dt, scheme, screened=screened, alpha=1.5, lam=3.0)
            s.upload(w)
            for k in split:
                s.advance(k)
            got = s.download()
            s.close()
            assert rel_l2(got, want) < 1e-12, (scheme, split)


@pytest.mark.parametrize("sizes", [[64] * 5, [128, 64, 128], [64, 256, 1024]])
def test_small_batches_vs_oracle(sizes):
    print(f"small batch {sizes}", flush=True)
    nus, dt = [1e-3 * (r + 1) for r in range(len(sizes))], 1e-5
    for graph in (True, False):
        e = T.Ensemble(sizes, nus, dt, T.SCHEME_RK4)
        e.use_graph(graph)
        ws = [_noise(n, n, 7 * r) for r, n in enumerate(sizes)]
        for r, w in enumerate(ws):
            e.upload(r, w)
        e.advance(1)
        e.advance(2)
        e.sync()
        for r, n in enumerate(sizes):
            assert rel_l2(e.download(r), _steps(ws[r], n, nus[r], dt, 3, T.SCHEME_RK4, False)) < 1e-12, r
        e.close()
