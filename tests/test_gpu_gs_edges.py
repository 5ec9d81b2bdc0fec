"""The Gauss-Seidel units' edge waves (fs2d_sweeps.hip) against the oracle, bit for bit.

A wave takes a loop by the edges that its sweep meets: rows 1 or n, column 1 with
the ring of the sweep before, column n, both columns, none.  Sizes: grids inside
one unit (both columns, both rows in a wave), of one unit and a row more or less,
and of a few units; sweep counts past 64 and 128, where row 1 comes to lie in
lane 0 and column 1 in a unit's first column; stale rings that differ from every
cell, and cells with zeros and subnormal values, whose quotients are redone.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle

pytestmark = pytest.mark.gpu

SIZES = [(1, 3), (2, 9), (5, 70), (62, 20), (63, 66), (64, 131), (65, 20), (127, 9), (130, 131), (200, 70)]


def values(R, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((3, R, R), dtype=np.float32) * np.float32(0.02)
    at = rng.integers(0, 60, x.shape)
    x[at == 0] = 0.0
    x[at == 1] *= np.float32(1e-36)
    x[at == 2] *= np.float32(1e-42)
    x[:, 0, :] += 1.0
    x[:, :, -1] -= 2.0
    return [np.ascontiguousarray(f) for f in x]


@pytest.mark.parametrize("n, K", SIZES)
@pytest.mark.parametrize("cols, block, lag", [(64, 8, 4), (64, 8, 8), (128, 8, 4), (64, 4, 1), (128, 4, 8), (64, 2, 4)])
def test_edges(n, K, cols, block, lag, oracle_lib):
    R, O = n + 2, oracle_lib
    st = values(R, 1000 * n + K)
    want = [x.copy() for x in st]
    for f in range(3):
        O.diffuse(want[f], f, 1e-3, 0.05, K, oracle.GS_LEX)
    want.append(O.project(want[1], want[2], K, oracle.GS_LEX, want_p=True))
    with fs2d_amd.Solver(R, diffuse_iterations=K, pressure_iterations=K, gs_tile_cols=cols, gs_block=block,
                         gs_lag=lag) as s:
        s.upload(*st)
        for f in range(3):
            s.diffuse(f, 1e-3, 0.05, K)
        s.project(K)
        got = [*s.download(), s.pressure()]
        s.upload(*st)
        s.set_sources(None, None, None)
        s.step_n(2, 1e-3, 1e-3, 0.05)  # all solves of a step, pipelined
        got += s.download()
    more, z = [x.copy() for x in st], np.zeros((R, R), np.float32)
    for _ in range(2):
        O.solve(more[0], z, 1e-3, more[1], more[2], z, z, 1e-3, 0.05, K, K, oracle.GS_LEX)
    for k, (a, b) in enumerate(zip(got, want + more)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"array {k}: {int(np.sum(a != b))} differ"
