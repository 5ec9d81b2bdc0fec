"""Fields in and out of the device (fs2d_transfer.hip), on both of its ways.

Per call, host arrays of up to 8 MB in all go through pinned memory and larger
ones as whole arrays through a device buffer; R = 836 is the last and R = 837
the first size of three arrays at that line.  Every transfer copies, so every
check is for equal bits, NaN and -0 included, against the arrays themselves.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def fields(R, seed):
    rng = np.random.default_rng(seed)
    out = [rng.standard_normal((R, R), dtype=np.float32) for _ in range(3)]
    for k, x in enumerate(out):
        x[0, 0], x[R - 1, R - 1], x[R // 2, 0] = np.nan, -0.0, np.float32(np.inf) * (1 - 2 * (k & 1))
    return out


def same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


@pytest.mark.parametrize("R", [3, 64, 65, 255, 257, 836, 837, 1100])
def test_host_and_device_round_trips(R):
    x = fields(R, R)
    dev = [torch.from_numpy(a).cuda() for a in fields(R, R + 1)]
    back = [torch.zeros_like(t) for t in dev]
    torch.cuda.synchronize()
    L = fs2d_amd.library()
    with fs2d_amd.Solver(R, diffuse_iterations=2, pressure_iterations=2) as s:
        s.upload(*x)
        assert all(same(a, b) for a, b in zip(x, s.download()))
        assert L.fs2d_hip_upload_device(s._h, *(t.data_ptr() for t in dev)) == 0
        got = s.download()
        assert L.fs2d_hip_download_device(s._h, *(t.data_ptr() for t in back)) == 0
        s.sync()
        assert all(same(a.cpu(), b) and same(a.cpu(), c.cpu()) for a, b, c in zip(dev, got, back))
        # one array named for every field: the last one copied is the one it holds
        assert L.fs2d_hip_download_device(s._h, *(back[0].data_ptr(),) * 3) == 0
        s.sync()
        assert same(back[0].cpu(), dev[2].cpu())


@pytest.mark.parametrize("R", [591, 592, 900])  # six arrays: the last pinned size, the first past it
def test_solve_equals_the_resident_calls(R):
    rng = np.random.default_rng(R)
    x = [rng.standard_normal((R, R), dtype=np.float32) * np.float32(0.01) for _ in range(6)]
    out = [a.copy() for a in x[:3]]
    with fs2d_amd.Solver(R, diffuse_iterations=3, pressure_iterations=3) as s:
        for _ in range(3):
            s.solve(out[0], x[3], 1e-5, out[1], out[2], x[4], x[5], 1e-5, 0.05)
    with fs2d_amd.Solver(R, diffuse_iterations=3, pressure_iterations=3) as s:
        s.upload(*x[:3])
        s.set_sources(*x[3:])
        s.step_n(3, 1e-5, 1e-5, 0.05)
        want = s.download()
    assert all(same(a, b) for a, b in zip(out, want))


def test_batch_round_trip():
    sizes = [3, 66, 300, 900]
    with fs2d_amd.Batch([(R, 4, 0.05, 1e-5, 1e-5) for R in sizes]) as b:
        x = [fields(R, 7 * R) for R in sizes]
        for k in range(len(sizes)):
            b.upload(k, *x[k])
        for k in range(len(sizes)):
            assert all(same(p, q) for p, q in zip(x[k], b.download(k)))
