"""Transfers of arrays that are not what a call's name suggests.

The host calls take whatever memory the runtime can copy: pageable arrays, pinned ones
and device arrays; the device calls take pinned memory too, and arrays anywhere in a
device allocation.  Each is compared with the arrays themselves, for equal bits.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def arrays(R, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((R, R), dtype=np.float32) for _ in range(3)]


def place(kind, a):
    t = torch.from_numpy(a.copy())
    if kind == "pageable":
        return t
    if kind == "pinned":
        return t.pin_memory()
    if kind == "inside":  # 3 floats into an allocation
        whole = torch.zeros(a.size + 8, device="cuda")
        whole[3 : 3 + a.size] = t.flatten().cuda()
        return whole[3 : 3 + a.size].view(a.shape)
    return t.cuda()


HOST = [("pageable",) * 3, ("pinned",) * 3, ("device",) * 3, ("pageable", "pinned", "device"), ("inside", "pageable", "pinned")]
DEVICE = [("device",) * 3, ("pinned",) * 3, ("inside", "pinned", "device")]


@pytest.mark.parametrize("R", [3, 64, 200, 900])
@pytest.mark.parametrize("call, kinds", [("", k) for k in HOST] + [("_device", k) for k in DEVICE])
def test_memory_of_every_kind(R, call, kinds):
    L = fs2d_amd.library()
    x = arrays(R, R)
    src = [place(k, a) for k, a in zip(kinds, x)]
    dst = [place(k, np.zeros_like(a)) for k, a in zip(kinds, x)]
    torch.cuda.synchronize()
    with fs2d_amd.Solver(R, diffuse_iterations=2, pressure_iterations=2) as s:
        assert getattr(L, f"fs2d_hip_upload{call}")(s._h, *(t.data_ptr() for t in src)) == 0
        assert all(np.array_equal(a, b) for a, b in zip(x, s.download()))
        assert getattr(L, f"fs2d_hip_download{call}")(s._h, *(t.data_ptr() for t in dst)) == 0
        s.sync()
        assert all(np.array_equal(a, t.cpu().numpy()) for a, t in zip(x, dst))


@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_solve_and_sources(kind):
    R, x = 130, arrays(130, 1) + arrays(130, 2)
    x = [a * np.float32(0.01) for a in x]
    L = fs2d_amd.library()
    want = [a.copy() for a in x[:3]]
    with fs2d_amd.Solver(R, diffuse_iterations=3, pressure_iterations=3) as s:
        s.solve(want[0], x[3], 1e-5, want[1], want[2], x[4], x[5], 1e-5, 0.05)
    t = [place(kind, a) for a in x]
    torch.cuda.synchronize()
    p = [q.data_ptr() for q in t]
    with fs2d_amd.Solver(R, diffuse_iterations=3, pressure_iterations=3) as s:
        assert L.fs2d_hip_solve(s._h, p[0], p[3], 1e-5, p[1], p[2], p[4], p[5], 1e-5, 0.05) == 0
        s.sync()
        assert all(np.array_equal(a, q.cpu().numpy()) for a, q in zip(want, t))
        s.upload(*x[:3])
        assert L.fs2d_hip_set_sources(s._h, *p[3:]) == 0
        s.step_n(1, 1e-5, 1e-5, 0.05)
        assert all(np.array_equal(a, b) for a, b in zip(want, s.download()))


def test_batch_memory():
    L = fs2d_amd.library()
    x = arrays(66, 5)
    for kind in ("pinned", "device"):
        src, dst = [place(kind, a) for a in x], [place(kind, np.zeros_like(a)) for a in x]
        torch.cuda.synchronize()
        with fs2d_amd.Batch([(10, 4, 0.05, 1e-5, 1e-5), (66, 4, 0.05, 1e-5, 1e-5)]) as b:
            assert L.fs2d_hip_batch_upload(b._h, 1, *(t.data_ptr() for t in src)) == 0
            assert all(np.array_equal(a, c) for a, c in zip(x, b.download(1)))
            assert L.fs2d_hip_batch_download(b._h, 1, *(t.data_ptr() for t in dst)) == 0
            assert all(np.array_equal(a, t.cpu().numpy()) for a, t in zip(x, dst))


def test_a_large_transfer_goes_by_ranges_of_rows():
    """Arrays past the device buffer's 128 MB (a range of 5592 rows of 6000 and the rest),
    and what a handle holds for them."""
    R = 6000
    rng = np.random.default_rng(3)
    x = [rng.integers(0, 1 << 20, (R, R), dtype=np.int32).astype(np.float32) for _ in range(3)]

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    with fs2d_amd.Solver(900) as s:  # whatever the runtime allocates for itself is there afterwards
        s.upload(*(a[:900, :900].copy() for a in x))
        s.download()
    with fs2d_amd.Solver(R) as s:
        before = free()
        s.upload(*x)
        assert all(np.array_equal(a, b) for a, b in zip(x, s.download()))
        assert before - free() <= 132 << 20
