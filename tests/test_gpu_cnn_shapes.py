"""The network's kernels at the edges of their tiles.

Shapes whose levels do not fill the 16 x 32 tiles of the weight gradient or the
8- and 16-row tiles of the convolution, the smallest field, and batches past
the pinned buffer.  Gradients are compared with PyTorch's float64 ones: each
value passes through at most 30 roundings to bfloat16 (2^-9 relative), in
quadrature 1.1 %, so a layer's gradient may be off by 10 % of its norm (a lost
tile or tap of one is far more), and the cosine by the square of that.
"""
from __future__ import annotations

import numpy as np
import pytest

from fs2d_amd import pressure_net as PN
from test_gpu_cnn import smooth_field, torch_net

pytestmark = pytest.mark.gpu


def sample(n, h, w, seed):
    rng = np.random.default_rng(seed)
    d = smooth_field(rng, n, h, w) * 1e-3
    target = smooth_field(rng, n, h, w) * 1e-2
    return d, (0.9 * target + smooth_field(rng, n, h, w) * 2e-3).astype(np.float32), target


@pytest.mark.parametrize("n,h,w", [(4, 32, 32), (3, 32, 96), (1, 160, 96), (2, 64, 288)])
def test_gradients_at_ragged_shapes(n, h, w):
    d, prev, target = sample(n, h, w, 11 * h + w)
    with PN.PressureNet(seed=5) as net:
        p = net.params()
        loss = net.train_step(d, prev, target, lr=0.0)
        g = net.grads()
        net.train_step(d, prev, target, lr=0.0)
        assert np.array_equal(g, net.grads())  # sums in a fixed order
    _, _, tloss, layers = torch_net(p, d, prev, target)
    assert abs(loss - float(tloss.detach())) <= 2e-2 * float(tloss.detach())
    for k, ((gw, gb), (wt, bt)) in enumerate(zip(PN.split_params(g), layers)):
        tw = wt.grad.permute(2, 3, 0, 1).reshape(9, gw.shape[1], gw.shape[2]).numpy()
        tb = bt.grad.numpy()
        if k == 0:  # only the two real input channels carry gradient
            tw, gw = tw[:, :, :2], gw[:, :, :2]
        if k == 14:  # only output channel 0
            tw, gw, tb, gb = tw[:, :1], gw[:, :1], tb[:1], gb[:1]
        rel = np.linalg.norm(gw - tw) / np.linalg.norm(tw)
        cos = float((tw * gw).sum() / (np.linalg.norm(tw) * np.linalg.norm(gw)))
        relb = np.linalg.norm(gb - tb) / np.linalg.norm(tb)
        assert rel < 0.1 and cos > 0.99 and relb < 0.1, f"layer {k}: weights {rel:.3e} cos {cos:.4f} bias {relb:.3e}"


@pytest.mark.parametrize("n,h,w", [(2, 1024, 1024), (3, 1024, 1024), (5, 32, 160)])
def test_batch_predicts_as_its_samples(n, h, w):
    """2 x 1024 x 1024 is the largest prediction read back through pinned memory, 3 x 1024 x 1024 past it."""
    rng = np.random.default_rng(n + h)
    d = rng.standard_normal((n, h, w), dtype=np.float32) * np.float32(1e-3)
    prev = rng.standard_normal((n, h, w), dtype=np.float32)
    with PN.PressureNet(seed=3) as net:
        whole = net.predict(d, prev)
        for k in range(n):
            assert np.array_equal(whole[k:k + 1], net.predict(d[k:k + 1], prev[k:k + 1]))
