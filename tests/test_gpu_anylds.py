"""Mixed-radix transforms in LDS: lengths at the edges of what they take (2048),
each radix and primes, batches that leave the last workgroup partly empty, one
and many sequences per workgroup, and calls of different sizes one after another
and from several threads through the kept work space.

Bar: 1e-14 relative L2 against numpy.  A prime of length n sums n products in
order, whose rounding grows as sqrt(n/2) ulp at most: 32 x 1.1e-16 at 2048, and
two axes add in quadrature."""
import threading

import numpy as np
import pytest

import oracle as O
import tara_amd as T
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2047, 3), (2049, 3), (2048, 5), (2017, 2), (3, 2047), (5, 2050), (9, 300), (50, 49),
                                   (35, 2500), (1458, 17), (11, 13), (6, 1), (2, 7)])
def test_transforms_vs_numpy(shape):
    print(f"any length {shape}", flush=True)
    rng = np.random.default_rng(shape[0] + 7 * shape[1])
    a = np.asfortranarray(rng.standard_normal(shape))
    want = np.asfortranarray(np.fft.rfftn(a.T).T)
    assert rel_l2(T.fft_r2c(a), want) < 1e-14
    assert rel_l2(T.fft_c2r(want, shape[0]) / a.size, a) < 1e-14


def _w(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return O.r2c(np.asfortranarray(rng.standard_normal((nx, ny))))


def test_rhs_sizes_in_turn_and_from_threads():
    """The kept work space holds another size's data when a call starts."""
    sizes = [(30, 18), (96, 80), (9, 21), (64, 48), (30, 18), (250, 100)]
    ws = [_w(nx, ny, nx) for nx, ny in sizes]
    want = [O.derive2csh(w, nx, 1e-3) for w, (nx, _) in zip(ws, sizes)]

    def call(k, out):
        nx, ny = sizes[k]
        out[k] = T.derive2csh(nx, ny, nx // 2 + 1, 1e-3, ws[k])

    print("sizes in turn", flush=True)
    got = {}
    for k in range(len(sizes)):
        call(k, got)
    print("sizes from threads", flush=True)
    got2 = {}
    th = [threading.Thread(target=call, args=(k, got2)) for k in range(len(sizes))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(len(sizes)):
        assert rel_l2(got[k], want[k]) < 1e-12, sizes[k]
        assert np.array_equal(got[k], got2[k]), sizes[k]
