"""Calls on a stream that their caller captures: device arrays in, steps, device arrays
out as one graph of the caller's, replayed with other inputs and with the caller's own
work between the replays, against the same calls made one by one."""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from conftest import bits_equal
from fs2d_amd import workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("order", [fs2d_amd.GS_LEX, fs2d_amd.JACOBI])
@pytest.mark.parametrize("R", [66, 200])
def test_captured_by_the_caller(order, R):
    L = fs2d_amd.library()
    kw = dict(diffuse_iterations=6, pressure_iterations=9, order=order, launch_mode=fs2d_amd.LAUNCH_EAGER,
              jacobi_block=4 if order == fs2d_amd.JACOBI else 0)
    arrays = [torch.zeros((R, R), device="cuda") for _ in range(3)]
    ptrs = [a.data_ptr() for a in arrays]
    states = [W.random_state(R, seed=k, vel_scale=0.05)[:3] for k in range(4)]
    with fs2d_amd.Solver(R, **kw) as s, fs2d_amd.Solver(R, **kw) as plain:
        for t in (s, plain):
            t.set_sources(None, None, None)
            t.upload(*states[0])
            t.step_n(1, 1e-5, 1e-6, 0.01)  # plans and buffers
            t.sync()

        def calls():
            assert L.fs2d_hip_upload_device(s._h, *ptrs) == 0
            s.step_n(2, 1e-5, 1e-6, 0.01)
            assert L.fs2d_hip_download_device(s._h, *ptrs) == 0

        stream = torch.cuda.ExternalStream(s.stream())
        torch.cuda.synchronize()
        for _ in range(4):  # the fields' places cycle: a capture from a state that the replays leave
            calls()
        s.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            calls()
        for k, st in enumerate(states[1:]):
            for a, x in zip(arrays, st):
                a.copy_(torch.from_numpy(x))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            plain.upload(*st)
            plain.step_n(2, 1e-5, 1e-6, 0.01)
            for a, w in zip(arrays, plain.download()):
                assert bits_equal(a.cpu().numpy(), w), k
            (arrays[0] * 2).sum().item()
