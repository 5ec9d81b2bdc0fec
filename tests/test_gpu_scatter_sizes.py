"""The density scatter at the sizes where its launches change, against the oracle, bit
for bit: bands of the window path (4 rows, remainders, radii 1 to 4), and the sorted
path's chunks (1 to 16 rounds of 256 items, the last chunk partial) and scan tiles
(16384 counts, the last partial), with sources that pile up on few targets.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [3, 5, 6, 7, 10, 18, 63, 66, 92, 93, 94, 130, 131, 258, 363, 364, 366, 515, 726])
@pytest.mark.parametrize("reach", [0.9, 1.9, 2.9, 3.9, 10.0, -3.0])
def test_scatter(R, reach, oracle_lib):
    rng = np.random.default_rng(7 * R + int(10 * abs(reach)))
    rho = rng.standard_normal((R, R), dtype=np.float32)
    u, v = (rng.uniform(-1, 1, (R, R)).astype(np.float32) for _ in range(2))
    if reach < 0:  # every source of a row moves onto a few cells
        i, j = np.indices((R, R))
        dt, k = np.float32(0.1), np.float32(R) * np.float32(0.1)
        u = ((R // 2 + i % 3 - j) / k).astype(np.float32)
        v = (rng.uniform(-1, 1, (R, R)) / k).astype(np.float32)
    else:
        dt = np.float32(reach / R)
    with fs2d_amd.Solver(R) as s:
        s.upload(rho, u, v)
        s.advect_density(float(dt))
        got = s.download()[0]
    want = rho.copy()
    oracle_lib.advect(want, u, v, 0, float(dt), True)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{int(np.sum(got != want))} differ"
