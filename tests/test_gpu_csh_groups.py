"""The small grids' y passes with two thread groups a column (batches and grids
between those of four groups and the large grids' passes): every length they have,
a last workgroup that is partly empty, both equations and schemes, against the
oracle.

Bar: a few steps 1e-12 (as the other grids' tests)."""
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _steps

pytestmark = pytest.mark.gpu


# wavefronts of two groups: 1650, 2080, 3096, 2570; a batch with the other kinds
@pytest.mark.parametrize("scheme", [T.SCHEME_AB2, T.SCHEME_RK4])
@pytest.mark.parametrize("sizes", [[64] * 200, [128] * 64, [256] * 24, [512] * 5, [512] * 9 + [128] * 3 + [64] * 300])
def test_batches_vs_oracle(sizes, scheme):
    print(f"two groups {len(sizes)} runs of {sizes[0]}", flush=True)
    nus, dt = [1e-3 * (1 + r % 7) for r in range(len(sizes))], 1e-5
    e = T.Ensemble(sizes, nus, dt, scheme)
    look = sorted({0, len(sizes) // 2, len(sizes) - 1})
    ws = {r: _noise(sizes[r], sizes[r], 7 * r) for r in look}
    for r, n in enumerate(sizes):
        if r in ws:
            e.upload(r, ws[r])
        else:
            e.ic_random(r, r + 1, 4.0)
    e.advance(1)
    e.advance(2)
    e.sync()
    for r in look:
        assert rel_l2(e.download(r), _steps(ws[r], sizes[r], nus[r], dt, 3, scheme, False)) < 1e-12, r
    e.close()


@pytest.mark.parametrize("screened", [False, True])
@pytest.mark.parametrize("nx,ny", [(2048, 512), (1024, 512), (2048, 256)])
def test_grids_vs_oracle(nx, ny, screened):
    w, nu, dt = _noise(nx, ny, nx - ny), 1e-3, 1e-5
    for scheme in (T.SCHEME_AB2, T.SCHEME_RK4):
        s = T.CshSolver(nx, ny, nu, dt, scheme, screened=screened, alpha=1.5, lam=3.0)
        s.upload(w)
        s.advance(1)
        s.advance(1)
        got = s.download()
        s.close()
        assert rel_l2(got, _steps(w, nx, nu, dt, 2, scheme, screened)) < 1e-12, scheme
