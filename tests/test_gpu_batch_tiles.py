"""Batched Jacobi launches on block tiles against the oracle, bit for bit.

Sizes at the edges of a tile's 32, 48 or 96 rows and 64 columns; sweep counts that
split evenly into launches of at most 8 and counts that do not, the smallest
among them (2: two launches of one sweep); divisors with and without a known
quotient beside each other in one batch; batches below and from 500 000 and
8 000 000 cells of three fields, where the tile's height changes.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle

pytestmark = pytest.mark.gpu

SMALL = [(3, 2, 1e-4), (32, 17, 0.0), (33, 9, 1e-5), (48, 8, 1e-4), (49, 20, 1e-6), (64, 3, 0.0), (65, 40, 1e-5),
         (96, 7, 1e-4), (97, 16, 7.24575e-3), (67, 8, 7.24575e-3)]


def special_values(R, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((3, R, R), dtype=np.float32) * np.float32(0.02)
    at = rng.integers(0, 40, x.shape)
    x[at == 0] = 0.0
    x[at == 1] *= np.float32(1e-36)
    x[at == 2] *= np.float32(1e-42)
    return [np.ascontiguousarray(f) for f in x]


@pytest.mark.parametrize("large,rows", [((), 16), (((385, 20, 1e-5),), 32), (((129, 33, 7.24575e-3), (412, 10, 0.0)), 32),
                                        (((130, 33, 7.24575e-3), (1650, 9, 1e-6)), 80)])
@pytest.mark.parametrize("block_per_cu", [0, 1])
def test_batched_tiles(large, rows, block_per_cu, oracle_lib):
    sims = [(R, K, 0.05, rate, 0.5 * rate) for R, K, rate in (*SMALL, *large)]
    with fs2d_amd.Batch(sims) as b:
        b.set_occupancy(block_per_cu, 8)
        starts = [special_values(s[0], 1000 * s[0] + s[1]) for s in sims]
        for k, st in enumerate(starts):
            b.upload(k, *st)
            b.set_sources(k)
        b.step_n(2)
        got = [b.download(k) for k in range(len(sims))]
        assert b.info()["tile_rows"] == rows
    for k, (R, K, dt, diff, visc) in enumerate(sims):
        want, z = [x.copy() for x in starts[k]], np.zeros((R, R), np.float32)
        for _ in range(2):
            oracle_lib.solve(want[0], z, diff, want[1], want[2], z, z, visc, dt, K, K, oracle.JACOBI)
        for f in range(3):
            a, w = got[k][f], want[f]
            assert np.all((a.view(np.uint32) == w.view(np.uint32)) | (np.isnan(a) & np.isnan(w))), \
                f"R={R} K={K} field {f}: {int(np.sum(a != w))} differ"
