"""Any-length transforms with a large prime factor: the rule that sends few
sequences of a prime above 1000 over the whole chip, both sides of it, workgroups
of a thread per output up to their largest, and that a prime just below the longest
length that runs in LDS costs no more than one just above it.

Bar: 1e-14 relative L2 against numpy (a prime of length n sums n products in order,
whose rounding grows as sqrt(n/2) ulp at most: 32 x 1.1e-16 at 2048)."""
import time

import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (67, 9), (113, 600), (251, 1), (1021, 1), (2042, 3), (2036, 4),
    (1009, 84), (1009, 85),       # rows past and at 1009 / 12; columns of 84 and 85
    (16, 1013), (256, 1013),      # 16 columns of a large prime, 136
    (2039, 169), (2039, 170),
])
def test_large_primes_vs_numpy(shape):
    print(f"large prime {shape}", flush=True)
    rng = np.random.default_rng(shape[0] + 11 * shape[1])
    a = np.asfortranarray(rng.standard_normal(shape))
    want = np.asfortranarray(np.fft.rfftn(a.T).T)
    assert rel_l2(T.fft_r2c(a), want) < 1e-14
    assert rel_l2(T.fft_c2r(want, shape[0]) / a.size, a) < 1e-14


def _time(f):
    f()
    best = 1e9
    for _ in range(10):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("rows", [1, 16])
def test_prime_below_lds_limit_costs_no_more_than_above(rows):
    """2039 and 2053 do the same work; one workgroup a sequence took 4.3 times as long."""
    print(f"prime cost at {rows} rows", flush=True)
    rng = np.random.default_rng(rows)
    below, above = (np.asfortranarray(rng.standard_normal((n, rows))) for n in (2039, 2053))
    wb, wa = T.fft_r2c(below), T.fft_r2c(above)
    assert _time(lambda: T.fft_r2c(below)) < 1.5 * _time(lambda: T.fft_r2c(above))
    assert _time(lambda: T.fft_c2r(wb, 2039)) < 1.5 * _time(lambda: T.fft_c2r(wa, 2053))
