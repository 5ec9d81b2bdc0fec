"""The density scatter's window path at the sizes where its bands are neither the
shortest nor the longest, radii 1 to 4, against the oracle, bit for bit: the band
follows from the waves per SIMD, and the last one may be a remainder of one row.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [4, 770, 771, 899, 1026, 1031, 1282, 1533, 2050])
@pytest.mark.parametrize("reach", [0.9, 1.9, 2.9, 3.9])
def test_bands(R, reach, oracle_lib):
    rng = np.random.default_rng(7 * R + int(10 * reach))
    rho = rng.standard_normal((R, R), dtype=np.float32)
    u, v = (rng.uniform(-1, 1, (R, R)).astype(np.float32) for _ in range(2))
    dt = float(np.float32(reach / R))
    with fs2d_amd.Solver(R) as s:
        s.upload(rho, u, v)
        s.advect_density(dt)
        got = s.download()[0]
    want = rho.copy()
    oracle_lib.advect(want, u, v, 0, dt, True)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{int(np.sum(got != want))} differ"
