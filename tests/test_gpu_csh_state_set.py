"""What setting a run's state does besides the copy, in one launch: history, non-finite
flag, and whether the state is zero outside the dealiasing circle.  States of changing
kinds set one after another with nothing waited for in between, the largest and
smallest grids that look, and that looking costs no more than not looking."""
import time

import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_band import _outside, _state
from test_gpu_csh_small import _steps

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_states_set_back_to_back():
    """ic_random (outside the circle at 2^-1000 or zero), set_omega (rounding noise
    outside) and uploads of both kinds, a run at a time and all over again."""
    n, runs, dt, nu = 256, 47, 1e-5, 1e-3
    ws = {k: _state(n, n, k, 3) for k in ("in", "edge", "all")}
    x = torch.from_numpy(np.random.default_rng(0).standard_normal((n, n)).astype(np.float32)).cuda()
    e = T.Ensemble([n] * runs, [nu] * runs, dt, T.SCHEME_AB2)
    for r in range(runs):
        e.upload(r, ws["all"])
    e.advance(3)  # leaves a history everywhere
    for kind in ("all", "in", "edge", "in"):
        for r in range(runs):
            e.ic_random(r, 5)
            e.set_omega(r, x)
            e.upload(r, ws[kind])
        e.advance(2)
        e.sync()
        want = _steps(ws[kind], n, nu, dt, 2, T.SCHEME_AB2, False)  # history zero again
        for r in (0, 1, runs - 1):
            got = e.download(r)
            assert rel_l2(got, want) < 1e-12, (kind, r)
            assert got[_outside(n, n)].any() == (kind != "in"), (kind, r)
    e.close()


def test_non_finite_flag_cleared():
    n, runs = 128, 200
    e = T.Ensemble([n] * runs, [1e-3] * runs, 1e-5, T.SCHEME_AB2)
    bad = _state(n, n, "in", 1)
    bad[1, 1] = np.nan
    for r in range(runs):
        e.upload(r, bad if r in (0, 77, runs - 1) else _state(n, n, "in", 2))
    e.advance(1)
    assert [r for r, f in enumerate(e.nonfinite()) if f] == [0, 77, runs - 1]
    e.upload(77, _state(n, n, "in", 2))
    assert [r for r, f in enumerate(e.nonfinite()) if f] == [0, runs - 1]
    e.close()


def _set_time(sizes):
    e = T.Ensemble(sizes, [1e-3] * len(sizes), 1e-5, T.SCHEME_AB2)
    x = torch.ones((sizes[0], sizes[0]), dtype=torch.float32, device="cuda")
    best = 1e9
    for k in range(40):
        t = time.perf_counter()
        e.set_omega(0, x)
        e.sync()
        if k > 5:
            best = min(best, time.perf_counter() - t)
    e.close()
    return best


def test_looking_costs_little():
    """One run more moves the batch to the passes that use the flag (46 / 47 runs of
    256^2).  With a launch each for the flag and the scan the call took 72 against 50 us;
    bar 1.25 times."""
    without, with_ = _set_time([256] * 46), _set_time([256] * 47)
    print(f"set_omega: not looking {1e6 * without:.1f} us, looking {1e6 * with_:.1f} us")
    assert with_ < 1.25 * without
