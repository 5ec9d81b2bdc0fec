"""The launches of a step, counted by hand where the configuration fixes them, and that
asking for them changes nothing."""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from fs2d_amd import workloads as W

pytestmark = pytest.mark.gpu

GS, JAC = fs2d_amd.GS_LEX, fs2d_amd.JACOBI


def scatter(targets, local, gates):
    """Window, keys, bounds and merge, a batch's gate; each sort pass of 9 bits scatters, all but the
    first count, and with more than 32 chunks (`local` false) each scans."""
    passes = -(-targets.bit_length() // 9)
    return 4 + gates + passes + (passes - 1) + (0 if local else passes)


@pytest.mark.parametrize("R, kd, kp, block", [(202, 20, 20, 8), (202, 3, 0, 2), (514, 8, 9, 4)])
def test_jacobi_launches(R, kd, kp, block):
    st = W.random_state(R, seed=R, vel_scale=0.05)[:3]
    with fs2d_amd.Solver(R, diffuse_iterations=kd, pressure_iterations=kp, order=JAC, jacobi_block=block) as s, \
            fs2d_amd.Solver(R, diffuse_iterations=kd, pressure_iterations=kp, order=JAC, jacobi_block=block) as other:
        for t in (s, other):
            t.upload(*st)
            t.set_sources(None, None, None)
        with pytest.raises(fs2d_amd.Fs2dError, match="first step"):
            s.step_launches()
        for k in range(5):
            s.step_n(1, 1e-5, 1e-6, 0.01)
            other.step_n(1, 1e-5, 1e-6, 0.01)
            # diffuses together, with the sources; scatter; gather; pressure solves with the divergence and
            # the gradient (0 sweeps: divergence and gradient a pass each), the last with a fold
            p = -(-kp // block) if kp else 2
            assert s.step_launches() == -(-kd // block) + scatter((R - 1) ** 2, (R - 2) ** 2 <= 32 * 256 * 16, 0) + 1 + 2 * p + 1
        for a, b in zip(s.download(), other.download()):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("R, options", [(130, {}), (130, {"gs_block": 1}), (300, {"gs_block": 8, "gs_lag": 4})])
def test_gauss_seidel_launches(R, options):
    st = W.random_state(R, seed=R, vel_scale=0.05)[:3]
    with fs2d_amd.Solver(R, diffuse_iterations=8, pressure_iterations=8, **options) as s, \
            fs2d_amd.Solver(R, diffuse_iterations=8, pressure_iterations=8, launch_mode=1, **options) as other:
        for t in (s, other):
            t.upload(*st)
            t.set_sources(None, None, None)
        for _ in range(3):
            s.step_n(1, 1e-5, 1e-6, 0.01)
            other.step_n(1, 1e-5, 1e-6, 0.01)
            n = s.step_launches()
            assert n == s.step_launches() == other.step_launches()
            p = s.gs_policy(1)["levels"]
            sc = scatter((R - 1) ** 2, True, 0)
            if options.get("gs_block") == 1:  # one-sweep tiles: each diffuse and its source alone
                assert n == 3 + 3 * s.gs_policy(0)["levels"] + sc + 2 * (2 + p) + 1 + 1
            else:  # sources, zero pressure, joint levels; the second projection's divergence zeroes it
                assert n == 2 + s.gs_policy(2)["levels"] + sc + 1 + 1 + (1 + p + 2)
        for a, b in zip(s.download(), other.download()):
            assert np.array_equal(a, b)


def test_batch_launches():
    sims = [(66, 20, 0.05, 1e-5, 1e-6), (130, 40, 0.05, 1e-5, 1e-6), (10, 3, 0.05, 0.0, 0.0)]
    with fs2d_amd.Batch(sims) as b, fs2d_amd.Batch(sims) as other:
        for t in (b, other):
            for k, s in enumerate(sims):
                t.upload(k, *W.batch_state(s[0], seed=1, sim_index=k))
            t.step_n(1)
        targets = sum((s[0] - 1) ** 2 for s in sims)
        got = b.step_launches()
        # 5 launches of the longest solve, three solves; two gradients, one fold; scatter with its gate; gather
        assert got == {"launches": 15 + 3 + scatter(targets, True, 1) + 1, "fewest_sweeps": 1, "most_sweeps": 8}
        for _ in range(3):
            b.step_n(1)
            other.step_n(1)
            assert b.step_launches() == got
        for k in range(len(sims)):
            for x, y in zip(b.download(k), other.download(k)):
                assert np.array_equal(x, y)
