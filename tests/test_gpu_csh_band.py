"""States that are zero outside the dealiasing circle take passes that carry the
circle only, run by run: such states and states one mode away from it, both
schemes and equations, fused and separate y passes, both kinds of x pass, runs of
both kinds in one batch, and a solver that is given one kind after the other,
against the oracle's right-hand side.

Bars: a few steps 1e-12 (as the other grids' tests); outside the circle a limited
state stays exactly zero; a state set anew runs as in a new solver, bit for bit."""
import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _steps

pytestmark = pytest.mark.gpu


def _outside(nx, ny):
    """Modes that lose their nonlinear term: |k| not below (Nx+Ny)/2/3."""
    i = np.arange(nx // 2 + 1)[:, None].astype(float)
    j = np.arange(ny)
    ky = np.where(j <= ny // 2, j, j - ny)[None, :].astype(float)
    return np.sqrt(i * i + ky * ky) >= ((nx + ny) / 2.0) / 3.0


def _state(nx, ny, kind, seed):
    """kind: "in" (circle only), "edge" (and one mode next to it), "all"."""
    w = _noise(nx, ny, seed)
    if kind != "all":
        out = _outside(nx, ny)
        w[out] = 0.0
        if kind == "edge":
            i, j = np.argwhere(out[:, : ny // 2])[0]
            w[i, j] = 1.0 + 2.0j
    return np.asfortranarray(w)


# 512 x 1024 paired x pass; 2048 x 512 one y transform a workgroup, no fusion;
# 4096 x 256 the large x pass
@pytest.mark.parametrize("kind", ["in", "edge"])
@pytest.mark.parametrize("nx,ny,screened", [(512, 1024, False), (1024, 1024, True), (2048, 512, False),
                                            (4096, 256, False), (64, 4096, False)])
def test_steps_vs_oracle(nx, ny, screened, kind):
    print(f"support {nx}x{ny} screened {screened} {kind}", flush=True)
    w, nu, dt = _state(nx, ny, kind, nx + ny), 1e-3, 1e-5
    for scheme in (T.SCHEME_AB2, T.SCHEME_RK4):
        want = _steps(w, nx, nu, dt, 3, scheme, screened)
        s = T.CshSolver(nx, ny, nu, dt, scheme, screened=screened, alpha=1.5, lam=3.0)
        first = []
        for start in (w, _state(nx, ny, "all", 3), w):  # the other kind of state in between
            s.upload(start)
            s.advance(1)
            s.advance(2)
            first.append(s.download())
        s.close()
        assert rel_l2(first[0], want) < 1e-12, scheme
        assert np.array_equal(first[0], first[2]), scheme
        if kind == "in":
            assert not first[0][_outside(nx, ny)].any()
        else:
            assert first[0][_outside(nx, ny)].any()


@pytest.mark.parametrize("n,runs", [(512, 9), (1024, 3)])
def test_batch_of_both_kinds_vs_oracle(n, runs):
    print(f"support batch {runs} x {n}", flush=True)
    nus, dt = [1e-3 * (r + 1) for r in range(runs)], 1e-5
    kinds = [("in", "all", "edge")[r % 3] for r in range(runs)]
    ws = [_state(n, n, k, 5 * r) for r, k in enumerate(kinds)]
    want = [_steps(ws[r], n, nus[r], dt, 2, T.SCHEME_RK4, False) for r in range(3)]
    for graph in (True, False):
        e = T.Ensemble([n] * runs, nus, dt, T.SCHEME_RK4)
        e.use_graph(graph)
        for r in range(runs):
            e.upload(r, ws[(r + 1) % runs])
        e.advance(1)
        for r in range(runs):
            e.upload(r, ws[r])
        e.advance(1)
        e.advance(1)
        e.sync()
        for r in range(3):
            assert rel_l2(e.download(r), want[r]) < 1e-12, kinds[r]
        e.close()
