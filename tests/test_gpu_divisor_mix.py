"""Steps whose fields have divisors of different kinds, against the oracle, bit for bit.

A divisor of a diffuse solve is 1 + 4 a.  It is exact by a pair of reciprocals (a
checked divisor, or a power of two, 1 where the rate is 0) or takes the corrected
quotient, and fields that share a launch take the kernel of the least of them.  The
corrected quotient turns a dividend of -0 into +0 and loses bits below 2^-100, so both
go to the IEEE division there, whatever the other divisors of the launch are.

-0 survives a step's later stages only where every value that meets it is negative or
-0, and where the pressure is exactly 0: velocities here are -|x| with many -0 where no
pressure is solved, and -0 but for two cells at each edge where one is (the sweeps'
pressure falls by 4 a cell along the rows, so it is 0 in the middle of 256 x 256).
Sources are -0 (+0 would turn -0 into +0).
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
import oracle

pytestmark = pytest.mark.gpu

GS, JAC = fs2d_amd.GS_LEX, fs2d_amd.JACOBI
DT = 0.0625


def divisor(R, rate):
    a = np.float32(np.float32(DT) * np.float32(R * R)) * np.float32(rate)
    return float(np.float32(1) + np.float32(4) * a)


def unchecked_rate(R):
    """A rate whose divisor takes the corrected quotient."""
    for k in range(1000):
        rate = float(np.float32(1e-6 * 1.01 ** k))
        if not fs2d_amd.division_plan(divisor(R, rate))["checked"]:
            return rate
    raise AssertionError("no unchecked divisor found")


def power_rate(R, d):
    """The rate whose divisor is d, a power of two (R * R is one here)."""
    rate = (d - 1) / 4 / (DT * R * R)
    assert divisor(R, rate) == d
    return rate


def velocities(R, seed, flat):
    rng = np.random.default_rng(seed)
    x = -np.abs(rng.standard_normal((3, R, R), dtype=np.float32)) * np.float32(0.01)
    at = rng.integers(0, 6, x.shape)
    x[at == 0] = -0.0
    x[at == 1] *= np.float32(1e-36)
    if flat:
        x[1:, 3:-3, 3:-3] = -0.0
    return [np.ascontiguousarray(f) for f in x]


def check_step(R, diff, visc, order, kd, kp, O, **options):
    st, z = velocities(R, R, kp > 0), np.full((R, R), -0.0, np.float32)
    want, steps = [x.copy() for x in st], 1 if kp else 2
    for _ in range(steps):
        O.solve(want[0], z, diff, want[1], want[2], z, z, visc, DT, kd, kp,
                oracle.GS_LEX if order == GS else oracle.JACOBI)
    with fs2d_amd.Solver(R, diffuse_iterations=kd, pressure_iterations=kp, order=order, **options) as s:
        s.upload(*st)
        s.set_sources(z, z, z)
        s.step_n(steps, diff, visc, DT)
        got = s.download()
    if visc == 0.0:
        inner = want[1][1:-1, 1:-1]
        assert np.signbit(inner[inner == 0]).any()  # -0 is there to be lost
    for k, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), \
            f"R={R} field {k}: {int(np.sum(a.view(np.uint32) != b.view(np.uint32)))} differ"


@pytest.mark.parametrize("kind", ["zero visc", "zero diff", "power of two visc"])
@pytest.mark.parametrize("order, kp, options", [(GS, 2, {}), (GS, 0, {}), (GS, 2, {"gs_block": 4, "gs_lag": 1}),
                                                (JAC, 2, {"jacobi_block": 8}), (JAC, 0, {"jacobi_block": 4})])
def test_mixed_divisors(kind, order, kp, options, oracle_lib):
    R = 256 if kp else 64
    other = unchecked_rate(R)
    diff, visc = {"zero visc": (other, 0.0), "zero diff": (0.0, other),
                  "power of two visc": (other, power_rate(R, 4.0))}[kind]
    check_step(R, diff, visc, order, 9, kp, oracle_lib, **options)


@pytest.mark.parametrize("d", [1.0, 2.0, 4.0, 1024.0])
@pytest.mark.parametrize("order, options", [(JAC, {"jacobi_kernel": 2, "jacobi_block": 3}), (JAC, {"jacobi_block": 3}),
                                            (GS, {"gs_block": 1}), (GS, {})])
def test_powers_of_two(d, order, options, oracle_lib):
    """One field a launch, the kernels that know only the corrected quotient among them."""
    R = 64
    rate = power_rate(R, d)
    st = velocities(R, 7, False)
    want = [x.copy() for x in st]
    for f in range(3):
        oracle_lib.diffuse(want[f], f, rate, DT, 5, oracle.GS_LEX if order == GS else oracle.JACOBI)
    with fs2d_amd.Solver(R, diffuse_iterations=5, pressure_iterations=2, order=order, **options) as s:
        s.upload(*st)
        for f in range(3):
            s.diffuse(f, rate, DT, 5)
        got = s.download()
    for k, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), \
            f"field {k}: {int(np.sum(a.view(np.uint32) != b.view(np.uint32)))} differ"
