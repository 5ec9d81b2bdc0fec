"""Batched Jacobi launches of one and two sweeps, which take strips of 16 rows and 62 or
60 columns a wave after a solve's first launch, against the oracle, bit for bit: sizes
at the strips' edges, the fewest sweeps, divisors of every kind, -0 and subnormal cells;
and the height of the tiles of many equal grids.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle
from test_gpu_batch_tiles import special_values

pytestmark = pytest.mark.gpu

SIMS = [(3, 4, 1e-4), (4, 2, 0.0), (17, 8, 1e-5), (18, 6, 1e-4), (19, 4, 0.0), (34, 2, 1e-6), (35, 12, 1e-5),
        (61, 8, 7.24575e-3), (62, 4, 0.0), (63, 6, 1e-4), (64, 20, 1e-5), (65, 4, 7.24575e-3), (66, 8, 0.0), (122, 4, 1e-4),
        (126, 6, 1e-5), (127, 8, 0.0), (130, 2, 1e-4), (200, 4, 1e-5)]


def compare(got, st, R, K, dt, diff, visc, steps, O):
    want, z = [x.copy() for x in st], np.zeros((R, R), np.float32)
    for _ in range(steps):
        O.solve(want[0], z, diff, want[1], want[2], z, z, visc, dt, K, K, oracle.JACOBI)
    for f in range(3):
        a, w = got[f], want[f]
        assert np.all((a.view(np.uint32) == w.view(np.uint32)) | (np.isnan(a) & np.isnan(w))), \
            f"R={R} K={K} field {f}: {int(np.sum(a != w))} differ"


@pytest.mark.parametrize("block", [1, 2])
@pytest.mark.parametrize("per_cu", [0, 1])  # an entry a wave, and waves that walk many
def test_strips(block, per_cu, oracle_lib):
    sims = [(R, K * block // 2, 0.05, rate, 0.5 * rate) for R, K, rate in SIMS if K * block // 2 >= 2 * block]
    starts = [special_values(s[0], 1000 * s[0] + s[1]) for s in sims]
    for st in starts:
        st[1][::3, ::2] = -0.0
    with fs2d_amd.Batch(sims * 4, jacobi_block=block) as b:
        b.set_occupancy(per_cu, 8)
        for k, st in enumerate(starts):
            b.upload(k, *st)
            b.set_sources(k)
        b.step_n(2)
        for k, (R, K, dt, diff, visc) in enumerate(sims):
            compare(b.download(k), starts[k], R, K, dt, diff, visc, 2, oracle_lib)


@pytest.mark.parametrize("R, count, rows", [(98, 300, 32), (130, 180, 80)])
def test_height_of_many_equal_grids(R, count, rows, oracle_lib):
    """9 and 8 million cells of three fields: regions of 48 rows (32 written after 8 sweeps) and of 96."""
    st = special_values(R, R)
    with fs2d_amd.Batch([(R, 16, 0.05, 1e-5, 1e-6)] * count) as b:
        for k in (0, count // 2, count - 1):
            b.upload(k, *st)
        b.step_n(1)
        assert b.info()["tile_rows"] == rows
        for k in (0, count // 2, count - 1):
            compare(b.download(k), st, R, 16, 0.05, 1e-5, 1e-6, 1, oracle_lib)
