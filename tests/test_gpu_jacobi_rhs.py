"""Jacobi solves whose first launch forms the right-hand sides (the source terms, the
divergence) and whose last one subtracts the gradient, against the oracle, bit for bit: one launch a solve (the result is in the
scratch field, the gradient a pass of its own) and several, sizes at the tiles' edges
and at both sides of where the gradient's place changes, source rings that must not be
read, and no sweeps at all (the separate passes).
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle

pytestmark = pytest.mark.gpu


SIZES = [3, 4, 32, 33, 48, 63, 64, 65, 97, 128, 129, 410, 1640]
SWEEPS = [(1, 1), (8, 3), (9, 17), (0, 5), (5, 0)]


@pytest.mark.parametrize("R,kd,kp", [(R, *k) for R in SIZES for k in SWEEPS] + [(3162, 1, 9), (3163, 1, 9)])
def test_step(R, kd, kp, oracle_lib):
    rng = np.random.default_rng(1000 * R + 10 * kd + kp)
    x = rng.standard_normal((6, R, R), dtype=np.float32) * np.float32(0.02)
    x[rng.integers(0, 30, x.shape) == 0] = 0.0
    x[rng.integers(0, 30, x.shape) == 0] *= np.float32(-1e-42)
    st, src = [np.ascontiguousarray(f) for f in x[:3]], [np.ascontiguousarray(f) for f in x[3:]]
    want, zeroed = [f.copy() for f in st], [f.copy() for f in src]
    for f, g in zip(src, zeroed):
        for h, v in ((f, np.nan), (g, 0.0)):
            h[0] = h[-1] = h[:, 0] = h[:, -1] = v
    steps = 2 if R < 1000 else 1
    with fs2d_amd.Solver(R, diffuse_iterations=kd, pressure_iterations=kp, order=fs2d_amd.JACOBI, jacobi_block=8) as s:
        s.upload(*st)
        s.set_sources(*src)
        s.step_n(steps, 1e-5, 1e-5, 0.05)
        got = s.download()
    for _ in range(steps):
        oracle_lib.solve(want[0], zeroed[0], 1e-5, want[1], want[2], zeroed[1], zeroed[2], 1e-5, 0.05, kd, kp,
                         oracle.JACOBI)
    for f, (a, w) in enumerate(zip(got, want)):
        assert np.all((a.view(np.uint32) == w.view(np.uint32)) | (np.isnan(a) & np.isnan(w))), \
            f"R={R} K={kd},{kp} field {f}: {int(np.sum(a != w))} differ"
