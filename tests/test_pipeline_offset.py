"""The levels by which a Gauss-Seidel step's first pressure solve trails its diffuses, at
diffuse sweep counts of one more than a multiple of the tile's 64 rows: there the last
velocity row that a pressure unit's divergence reads is the first of the next tile."""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from schedule_models import gs_pipeline_min_offset


@pytest.mark.parametrize("Kd", [1, 2, 64, 65, 66, 129])
@pytest.mark.parametrize("R, Kp, TW, M", [(66, 1, 64, 4), (130, 20, 64, 8), (200, 20, 128, 8), (213, 2, 64, 8),
                                          (176, 5, 128, 4), (128, 9, 64, 2)])
def test_offset_is_the_brute_force_minimum(R, Kd, Kp, TW, M):
    assert fs2d_amd.gs_pipeline_offset(R, Kd, Kp, TW, M) == gs_pipeline_min_offset(R, Kd, Kp, TW, M)


@pytest.mark.gpu
@pytest.mark.parametrize("R, kd, kp", [(66, 1, 3), (341, 1, 2), (473, 1, 9), (600, 1, 20), (341, 65, 4), (300, 129, 2)])
@pytest.mark.parametrize("options", [{}, {"gs_block": 4, "gs_lag": 1}, {"gs_block": 8, "gs_lag": 8, "gs_tile_cols": 128}])
def test_steps_at_those_counts(R, kd, kp, options, oracle_lib):
    import oracle
    from fs2d_amd import workloads as W

    st, z = W.random_state(R, seed=R, vel_scale=0.3)[:3], np.zeros((R, R), np.float32)
    want = [x.copy() for x in st]
    with fs2d_amd.Solver(R, diffuse_iterations=kd, pressure_iterations=kp, **options) as s:
        s.upload(*st)
        s.set_sources(None, None, None)
        for _ in range(3):
            s.step_n(1, 1e-4, 1e-5, 0.02)
            oracle_lib.solve(want[0], z, 1e-4, want[1], want[2], z, z, 1e-5, 0.02, kd, kp, oracle.GS_LEX)
            for k, (a, b) in enumerate(zip(s.download(), want)):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"field {k}: {int(np.sum(a != b))} differ"
