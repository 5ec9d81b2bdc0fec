"""The multigrid seed's kernels against the same V-cycles in float64.

Sides at the edges of what the kernels split: 128 (the largest that runs whole
in one block), 130 and 272 (the first levels above it; 65 and 17 x 17 coarsest
grids, 4096 and 289 sweeps), 116 (29 x 29), 112 and 224 (multiples of the
56-column tile), 258 (an odd side past the block, swept as launches), and
grids that no level coarsens.  Rounding: the smoothers damp every mode but the
mean, so float32's 6e-8 a sweep stays near 1e-6 of the field; 1e-3 is asked
for, and a lost halo, edge or level is over 1e-2.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from fs2d_amd import pressure_net as PN

pytestmark = pytest.mark.gpu


def residual(p, b):
    q = np.pad(p, 1, mode="edge")
    return b - (4 * p - q[:-2, 1:-1] - q[2:, 1:-1] - q[1:-1, :-2] - q[1:-1, 2:])


def v_cycle(p, b):
    n = p.shape[0]

    def smooth(p, count):
        for _ in range(count):
            p = p + 0.2 * residual(p, b)
        return p

    if n % 2 or n // 2 < 4:
        return smooth(p, min(4096, max(64, n * n)))
    p = smooth(p, 2)
    r = residual(p, b)
    c = v_cycle(np.zeros((n // 2, n // 2)), r[::2, ::2] + r[::2, 1::2] + r[1::2, ::2] + r[1::2, 1::2])
    q = np.pad(c, 1, mode="edge")
    i = np.arange(1, n + 1)
    near, far = (i + 1) // 2, np.where(i % 2 == 1, (i + 1) // 2 - 1, (i + 1) // 2 + 1)
    rows = 0.75 * q[near] + 0.25 * q[far]
    return smooth(p + 0.75 * rows[:, near] + 0.25 * rows[:, far], 2)


@pytest.mark.parametrize("n,tol", [(1, 1e-3), (7, 1e-2), (8, 1e-2), (20, 1e-2), (112, 1e-2), (116, 1e-2), (128, 1e-2),
                                   (130, 2e-1), (224, 1e-2), (258, 5e-1), (272, 1e-2), (480, 5e-2)])
def test_v_cycles_match_float64(n, tol):
    rng = np.random.default_rng(n)
    R = n + 2
    u, v = (rng.standard_normal((2, R, R)) * 0.01).astype(np.float32)
    with fs2d_amd.Solver(R, diffuse_iterations=4, pressure_iterations=4, order=fs2d_amd.JACOBI) as s:
        s.upload(np.zeros((R, R), np.float32), u, v)
        sweeps, rel, _, _ = PN.seeded_projection(s, None, 3, tol, 0, check=1, fallback=False)
        p = s.pressure().astype(np.float64)
    coarse = n % 2 == 0 and n // 2 >= 4
    cycles = sweeps // (4 if coarse else min(4096, max(64, n * n)))
    d = PN.divergence(u, v)
    want = np.zeros((n, n))
    for _ in range(cycles):
        want = v_cycle(want, d)
    got = p[1:-1, 1:-1]
    assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
    assert np.array_equal(p[0, 1:-1], p[1, 1:-1]) and np.array_equal(p[1:-1, -1], p[1:-1, -2])  # its ring
    r = np.linalg.norm(residual(got, d)) / np.linalg.norm(d)
    assert abs(r - rel) <= 1e-3 * r + 1e-5
