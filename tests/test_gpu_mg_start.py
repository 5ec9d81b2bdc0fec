"""A multigrid-seeded projection starts from zero, whatever the pressure field holds:
after a pressure of NaN it gives what a new handle gives, on grids whose whole cycle is
one launch, on grids with levels above that, and where no level coarsens."""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from conftest import bits_equal
from fs2d_amd import pressure_net as PN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 64, 128, 129, 130, 256, 258])
@pytest.mark.parametrize("sweeps", [0, 3])
def test_from_zero_whatever_was_there(n, sweeps):
    rng = np.random.default_rng(n)
    R = n + 2
    u, v = (rng.standard_normal((2, R, R)) * 0.01).astype(np.float32)
    z = np.zeros((R, R), np.float32)
    got = []
    for spoiled in (False, True):
        with fs2d_amd.Solver(R, pressure_iterations=4, order=fs2d_amd.JACOBI, jacobi_block=2) as s:
            if spoiled:
                s.upload(z, np.full_like(z, np.nan), np.full_like(z, np.nan))
                s.project(4)
                assert np.isnan(s.pressure()).any()
            s.upload(z, u, v)
            run, rel, _, _ = PN.seeded_projection(s, None, 3, 0.0 if sweeps else 0.5, sweeps, check=1, fallback=False)
            got.append([*s.download()[1:], s.pressure(), run, rel])
    for a, b in zip(got[0][:3], got[1][:3]):
        assert bits_equal(a, b)
    assert got[0][3:] == got[1][3:]
