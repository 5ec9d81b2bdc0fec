"""The network at the ends of what its calls accept, and what they hold for it."""
from __future__ import annotations

import numpy as np
import pytest

from fs2d_amd import pressure_net as PN

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_more_samples_than_a_second_grid_dimension():
    """65 537 samples of the smallest field (the calls accept 262 144): each is
    predicted as it is alone, whatever its place in the batch."""
    n, h, w = 65537, 32, 32
    rng = np.random.default_rng(2)
    few_d = rng.standard_normal((8, h, w), dtype=np.float32) * np.float32(1e-3)
    few_p = rng.standard_normal((8, h, w), dtype=np.float32)
    which = np.arange(n) % 8
    with PN.PressureNet(seed=3) as net:
        whole = net.predict(few_d[which], few_p[which])
        for k in range(8):
            alone = net.predict(few_d[k:k + 1], few_p[k:k + 1])
            assert np.array_equal(whole[k::8], np.broadcast_to(alone, whole[k::8].shape)), k


def test_prediction_holds_no_training_buffers():
    """The partial sums of the weight gradients (75 MB at 512 x 512) come with a shape's first training step."""
    x = np.random.default_rng(1).standard_normal((1, 512, 512), dtype=np.float32)

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    with PN.PressureNet(seed=3) as net:  # whatever the runtime allocates for itself is there afterwards
        net.predict(x, x)
        net.train_step(x, x, x, 0.0)
        free()
    with PN.PressureNet(seed=3) as net:
        net.predict(x, x)
        predicting = free()
        net.predict(x, x)
        assert predicting - free() < 1 << 20
        net.train_step(x, x, x, 0.0)
        assert predicting - free() > 32 << 20
