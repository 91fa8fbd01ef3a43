"""Host boundary of the padded layouts: what is uploaded comes back bit for bit
through the device-side row packing, at the narrowest rows (Nh = 9 in 16), the
widest, and planes of unequal sides; and the transforms' host copies at widths
whose padding differs."""
import numpy as np
import pytest

import tara_amd as T

pytestmark = pytest.mark.gpu

L = 2 * np.pi


def _fields(shape, n, seed):
    rng = np.random.default_rng(seed)
    return [np.asfortranarray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) for _ in range(n)]


@pytest.mark.parametrize("nx,ny,nz", [(16, 16, 16), (64, 32, 16), (256, 16, 32), (32, 256, 64)])
def test_mhd_upload_download_bits(nx, ny, nz):
    print(f"mhd rows {nx}x{ny}x{nz}", flush=True)
    s = T.MhdSolver(nx, ny, nz, T.MhdParams(L, L, L, 1e-3, 1e-3, 10.0, 1e-4))
    for seed in (1, 2):  # twice: the second state replaces every row of the first
        st = _fields((nx // 2 + 1, ny, nz), 8, seed)
        s.upload(st)
        for a, b in zip(st, s.download()):
            assert np.array_equal(a, b)
    s.close()


@pytest.mark.parametrize("family", ["coh", "com"])
@pytest.mark.parametrize("nx,ny", [(16, 16), (16, 256), (256, 16), (128, 64)])
def test_f2_upload_download_bits(family, nx, ny):
    print(f"{family} rows {nx}x{ny}", flush=True)
    p = (T.CohParams(np.pi, L, L, 1e-3, 1e-3, 3.0, 1e-4) if family == "coh"
         else T.ComParams(np.pi, L, L, 1e-3, 1e-4, 2.0, 0.0, 0.0, 1e-4))
    s = T.F2Solver(nx, ny, p)
    st = _fields((nx // 2 + 1, ny), s.nf, nx + ny)
    s.upload(st)
    for a, b in zip(st, s.download()):
        assert np.array_equal(a, b)
    s.close()


@pytest.mark.parametrize("shape", [(14, 3), (16, 8), (30, 7, 5), (32, 16, 8), (6, 1)])
def test_host_transforms_any_row_width(shape):
    print(f"transform rows {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    a = np.asfortranarray(rng.standard_normal(shape))
    want = np.fft.rfftn(a.T).T
    got = T.fft_r2c(a)
    assert np.linalg.norm(got - want) < 1e-13 * np.linalg.norm(want)
    back = T.fft_c2r(want, shape[0]) / a.size
    assert np.linalg.norm(back - a) < 1e-13 * np.linalg.norm(a)
