"""Batches that fill the chip, whose y passes are those of the large grids (three
kernels a stage, Ny below 1024): every length they have, runs that are zero outside
the dealiasing circle, next to it and everywhere side by side, both schemes, captured
and not, and runs whose kind changes when they are set anew, against the oracle.  The
kernels of the captured step say which passes a batch takes.

Bars: a few steps 1e-12 (as the other grids' tests); outside the circle a limited
state stays exactly zero."""
import numpy as np
import pytest

import tara_amd as T
from conftest import rel_l2
from test_gpu_csh_band import _outside, _state
from test_gpu_csh_small import _steps

pytestmark = pytest.mark.gpu

KINDS = ("in", "edge", "all")


# the smallest batch of each size past two groups a column (wavefronts: 6168, 6063,
# 6013, 6006), the largest below it
@pytest.mark.parametrize("scheme", [T.SCHEME_AB2, T.SCHEME_RK4])
@pytest.mark.parametrize("n,runs,large", [(512, 12, True), (256, 47, True), (128, 185, True), (64, 728, True),
                                          (512, 11, False), (256, 46, False)])
def test_kinds_side_by_side(n, runs, large, scheme):
    print(f"batch {runs} x {n} scheme {scheme}", flush=True)
    dt, steps = 1e-5, 3
    nus = [1e-3 * (1 + r % 4) for r in range(runs)]
    ws = [_state(n, n, k, 5 + 3 * q) for q, k in enumerate(KINDS)]
    look = [0, 1, 2, runs // 2, runs - 2, runs - 1]
    want = {(q, nu): _steps(ws[q], n, nu, dt, steps, scheme, False)
            for q, nu in {(r % 3, nus[r]) for r in look}}
    out = _outside(n, n)
    for graph in (True, False):
        e = T.Ensemble([n] * runs, nus, dt, scheme)
        e.use_graph(graph)
        for r in range(runs):  # another kind first
            e.upload(r, ws[(r + 1) % 3])
        e.advance(1)
        for r in range(runs):
            e.upload(r, ws[r % 3])
        e.advance(1)
        e.advance(steps - 1)
        e.sync()
        if graph:
            stages = 4 if scheme == T.SCHEME_RK4 else 1
            assert e.graph_nodes()[1] == stages * (3 if large else 2)
        for r in look:
            got = e.download(r)
            assert rel_l2(got, want[r % 3, nus[r]]) < 1e-12, (graph, r)
            if r % 3 == 0:
                assert not got[out].any(), (graph, r)
        e.close()


def test_mixed_sizes_in_one_ensemble():
    """Buckets on both sides of the rule in one captured step."""
    sizes = [512] * 12 + [128] * 5 + [64] * 728 + [256] * 3
    print(f"mixed {len(sizes)} runs", flush=True)
    dt, nu = 1e-5, 1e-3
    ws = {n: [_state(n, n, k, n + q) for q, k in enumerate(KINDS)] for n in (64, 128, 256, 512)}
    e = T.Ensemble(sizes, [nu] * len(sizes), dt, T.SCHEME_RK4)
    for r, n in enumerate(sizes):
        e.upload(r, ws[n][r % 3])
    e.tune(2)
    e.advance(2)
    e.sync()
    assert e.graph_nodes()[1] == 2 * 12 + 2 * 8
    for r in (0, 1, 2, 11, 12, 13, 16, 17, 300, 744, 745, 746, 747):
        n = sizes[r]
        assert rel_l2(e.download(r), _steps(ws[n][r % 3], n, nu, dt, 2, T.SCHEME_RK4, False)) < 1e-12, r
    e.close()
