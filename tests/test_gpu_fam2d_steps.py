"""The 2D compressible steppers over every transform length they have (rows and
columns packed several to a workgroup on the shortest), unequal sides, steps in
one call and split over calls (the inverse transforms of a new state come from
the step before it, except a call's first), a new state on a used handle, and
one right-hand side: against the oracle.

Bar: 1e-12 relative L2 (as single right-hand sides: a few steps of small dt)."""
import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2

pytestmark = pytest.mark.gpu

PI = np.pi
BOX = dict(pi=PI, lx=2 * PI, ly=3 * PI)
COH = dict(mux=2e-4, muy=3e-4, cs=3.77)
COM = dict(mu=1e-3, eta=1e-4, cs=2.0, kf=1.0, a=0.3)
GRIDS = [(16, 16), (16, 256), (256, 16), (32, 64), (128, 32), (64, 128), (256, 256)]


def _state(nx, ny, nf, seed):
    rng = np.random.default_rng(seed)
    mean = (1.0, 0.0, 0.0, 2.0, 0.2, -0.1)
    return [O.r2c(np.asfortranarray(mean[f] + 0.02 * rng.standard_normal((nx, ny)))) for f in range(nf)]


@pytest.mark.parametrize("family", ["coh", "com"])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_rhs_and_steps_vs_oracle(family, nx, ny):
    print(f"{family} {nx}x{ny}", flush=True)
    dt, n = 1e-5, 4
    if family == "coh":
        prm, nf = T.CohParams(BOX["pi"], BOX["lx"], BOX["ly"], COH["mux"], COH["muy"], COH["cs"], dt), 3
        rhs = lambda s: O.derive2coh(s, nx, **BOX, **COH)  # noqa: E731
        one = lambda s: T.derive2coh(nx, ny, nx // 2 + 1, prm, s)  # noqa: E731
    else:
        prm, nf = T.ComParams(BOX["pi"], BOX["lx"], BOX["ly"], COM["mu"], COM["eta"], COM["cs"], COM["kf"], COM["a"],
                              dt), 6
        rhs = lambda s: O.derive2com(s, nx, **BOX, **COM)  # noqa: E731
        one = lambda s: T.derive2com(nx, ny, nx // 2 + 1, prm, s)  # noqa: E731
    st = _state(nx, ny, nf, nx + 2 * ny)
    for k, (a, b) in enumerate(zip(one(st), rhs(st))):
        assert rel_l2(a, b) < 1e-12, k
    ref, hist = st, [np.zeros_like(a) for a in st]
    for _ in range(n):
        f = rhs(ref)
        ref = [w + (1.5 * a - 0.5 * b) * dt for w, a, b in zip(ref, f, hist)]
        hist = f
    s = T.F2Solver(nx, ny, prm)
    for split in ((n,), (1, n - 1), (1,) * n, (3, 0, 1)):
        s.upload(st)
        for k in split:
            s.advance(k)
        for k, (a, b) in enumerate(zip(s.download(), ref)):
            assert rel_l2(a, b) < 1e-12, (split, k)
    s.close()
