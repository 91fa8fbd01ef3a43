"""Advance calls of one and a few steps on ensembles whose y passes are fused: a call's
first and last step (launched at first, captured from their second use on), steps set
anew in between, fused and unfused buckets side by side, captured and not, both schemes:
all the same bits, and the oracle's values.

Bar: a few steps 1e-12 (as the other ensemble tests)."""
import time

import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_small import _noise, _steps

pytestmark = pytest.mark.gpu

SIZES = [128] * 8 + [64] + [256] * 3 + [1024]


@pytest.mark.parametrize("scheme", [T.SCHEME_AB2, T.SCHEME_RK4])
@pytest.mark.parametrize("sizes", [SIZES, [512] * 12 + [64]])  # 12 runs of 512^2 are not fused
def test_calls_of_every_length(sizes, scheme):
    print(f"short calls {len(sizes)} runs scheme {scheme}", flush=True)
    dt, nu = 1e-5, 1e-3
    ws = {n: _noise(n, n, n) for n in set(sizes)}
    calls = [1, 1, 1, 2, 2, 3, 5, 1]
    look = {n: sizes.index(n) for n in set(sizes)}
    first = {}
    for graph, capture_first in ((True, False), (True, True), (False, False)):
        e = T.Ensemble(sizes, [nu] * len(sizes), dt, scheme)
        e.use_graph(graph)
        if capture_first:
            e.advance(0)
        for rep in range(2):  # set anew: nothing of the first run's end may remain
            for r, n in enumerate(sizes):
                e.upload(r, ws[n])
            for k in calls:
                e.advance(k)
            e.sync()
            for n, r in look.items():
                got = e.download(r)
                if n not in first:
                    first[n] = got
                    if n <= 256:
                        assert rel_l2(got, _steps(ws[n], n, nu, dt, sum(calls), scheme, False)) < 1e-12, n
                assert np.array_equal(got, first[n]), (graph, capture_first, rep, n)
        e.close()


def test_single_steps_cost_no_more_than_together():
    """40 runs of 256^2, AB2: a call of one step runs the inverse y pass once more and
    the last step's fused one not at all: 75 us against 73 in a long call.  Ending every
    call with the next one's inverse pass and beginning it with another, outside the
    graph, took 116.  Bar: 1.3 times."""
    e = T.Ensemble([256] * 40, [1e-3] * 40, 1e-7, T.SCHEME_AB2)
    for r in range(40):
        e.ic_random(r, r)

    def per_step(n):
        best = 1e9
        for _ in range(8):
            t = time.perf_counter()
            for _ in range(40 // n):
                e.advance(n)
            e.sync()
            best = min(best, (time.perf_counter() - t) / 40)
        return best

    long, single = per_step(40), per_step(1)
    print(f"per step: long call {1e6 * long:.1f} us, single steps {1e6 * single:.1f} us")
    assert single < 1.3 * long
    e.close()
