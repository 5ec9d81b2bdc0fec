"""The Jacobi block tiles (fs2d_jacobi.hip) against the oracle, bit for bit.

A launch takes tiles of 32, 48 or 96 rows by the cells it relaxes (below 500 000,
below 8 000 000, from there on; three fields count three times), 64 columns
wide.  Sizes: one tile, one tile and a row or column more, the last and first
size of each tile height, and the sweep counts that end on either slot.  Values:
random with zeros, subnormal and tiny ones (below the quotient's range) and
infinities.  A result that is not a number has no bits of its own to compare.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle

pytestmark = pytest.mark.gpu

def values(R, seed, special):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((3, R, R), dtype=np.float32) * np.float32(0.02)
    if special:
        at = rng.integers(0, 40, x.shape)
        x[at == 0] = 0.0
        x[at == 1] *= np.float32(1e-36)
        x[at == 2] *= np.float32(1e-42)
        x[0, R // 2, R // 3] = np.inf
    return [np.ascontiguousarray(f) for f in x]


def same(a, b):
    return bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))))


def check(R, m, special, rate, steps, O):
    st = values(R, 100 * R + m, special)
    K, kp, z = 2 * m + 1, m, np.zeros((R, R), np.float32)
    want = [x.copy() for x in st]
    for f in range(3):
        O.diffuse(want[f], f, rate, 0.05, K, oracle.JACOBI)
    want.append(O.project(want[1], want[2], kp, oracle.JACOBI, want_p=True))
    with fs2d_amd.Solver(R, diffuse_iterations=m + 1, pressure_iterations=kp, order=fs2d_amd.JACOBI,
                         jacobi_block=m) as s:
        s.upload(*st)
        for f in range(3):  # one field a launch
            s.diffuse(f, rate, 0.05, K)
        s.project(kp)
        got = [*s.download(), s.pressure()]
        s.upload(*st)
        s.set_sources(None, None, None)
        s.step_n(steps, rate, rate, 0.05)  # three fields a launch
        got += s.download()
    more = [x.copy() for x in st]
    for _ in range(steps):
        O.solve(more[0], z, rate, more[1], more[2], z, z, rate, 0.05, m + 1, kp, oracle.JACOBI)
    for k, (a, b) in enumerate(zip(got, want + more)):
        assert same(a, b), f"R={R} m={m} array {k}: {int(np.sum(a != b))} differ"


@pytest.mark.parametrize("R", [3, 31, 32, 33, 48, 49, 63, 64, 65, 96, 97, 127, 128, 129, 130])
@pytest.mark.parametrize("m", [1, 2, 5, 8])
def test_small_grids(R, m, oracle_lib):
    check(R, m, R % 2 == 0, 1e-4, 2, oracle_lib)


@pytest.mark.parametrize("R,m", [(408, 8), (409, 7), (707, 4), (708, 8), (1632, 8), (1633, 8), (1633, 3), (2828, 8),
                                 (2829, 8), (2829, 5)])
def test_tile_heights(R, m, oracle_lib):
    check(R, m, True, 1e-6, 1, oracle_lib)


@pytest.mark.parametrize("rate", [0.0, 7.24575e-3])  # a = 0 (divisor 1), and a divisor whose quotient is not checked
@pytest.mark.parametrize("special", [False, True])
def test_divisors(rate, special, oracle_lib):
    check(67, 8, special, rate, 2, oracle_lib)
