"""The narrowest grids of the fused 2D passes, Nx = 32 (16 half-length points, eight
rows a workgroup): every y length from one column tile to 4096, both equations and
schemes, the call on device arrays, and batches of 32^2 on the small grids' y passes
(two and four groups a column) and on the large grids', against the oracle.

Bars: one right-hand side 1e-13, a few steps 1e-12 (as the other grids' tests)."""
import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _rhs, _steps

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")  # before the library opens the device

NX = 32


@pytest.mark.parametrize("screened", [False, True])
@pytest.mark.parametrize("ny", [16, 32, 128, 1024, 2048, 4096])
def test_rhs_and_steps_vs_oracle(ny, screened):
    print(f"grid {NX}x{ny} screened {screened}", flush=True)
    w, nu, dt = _noise(NX, ny, ny), 1e-3, 1e-5
    nh = NX // 2 + 1
    f = T.derive2css(NX, ny, nh, 1.5, nu, w, 3.0) if screened else T.derive2csh(NX, ny, nh, nu, w)
    assert rel_l2(f, _rhs(w, NX, nu, screened)) < 1e-13
    for scheme in (T.SCHEME_AB2, T.SCHEME_RK4):
        s = T.CshSolver(NX, ny, nu, dt, scheme, screened=screened, alpha=1.5, lam=3.0)
        s.tune()  # finds the one shape there is
        s.upload(w)
        s.advance(1)
        s.advance(2)
        got = s.download()
        s.close()
        assert rel_l2(got, _steps(w, NX, nu, dt, 3, scheme, screened)) < 1e-12, scheme


@pytest.mark.parametrize("ny", [16, 32, 512])
def test_device_arrays(ny):
    print(f"device arrays {NX}x{ny}", flush=True)
    w = _noise(NX, ny, 3 * ny)
    d = torch.from_numpy(np.ascontiguousarray(w.T)).cuda()
    out = torch.full_like(d, float("nan"))
    T.derive2csh_noalloc(NX, ny, NX // 2 + 1, 1e-3, d.data_ptr(), out.data_ptr(),
                         torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rel_l2(out.cpu().numpy().T, _rhs(w, NX, 1e-3, False)) < 1e-13


@pytest.mark.parametrize("runs", [3, 2500, 2900])
def test_batches_vs_oracle(runs):
    """2500 runs: two groups a column; 2900: past the small grids' rule."""
    print(f"batch {runs} x {NX}", flush=True)
    dt, kinds = 1e-5, [_noise(NX, NX, k) for k in range(3)]
    nus = [1e-3 * (1 + r % 3) for r in range(runs)]
    want = [_steps(kinds[k], NX, 1e-3 * (1 + k), dt, 3, T.SCHEME_RK4, False) for k in range(3)]
    e = T.Ensemble([NX] * runs, nus, dt, T.SCHEME_RK4)
    for r in range(runs):
        e.upload(r, kinds[r % 3])
    e.advance(1)
    e.advance(2)
    e.sync()
    nodes, kernels = e.graph_nodes()
    assert kernels == (12 if runs == 2900 else 8)  # three kernels a stage, or two
    for r in {0, 1, 2, runs // 2, runs - 1}:
        assert rel_l2(e.download(r), want[r % 3]) < 1e-12, r
    e.close()
