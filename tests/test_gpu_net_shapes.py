"""The network's convolution kernels at the shapes where their tiles end:
images that are no multiple of the 16-pixel tile or smaller than its halo,
channel counts that leave output tiles partly filled or pad them (40: five
tiles), and layers too wide for an LDS tile (64: 768 input channels).

Every convolution is periodic, so an image laid out twice is the same problem:
each pixel's terms are the same values in the same order, and tiles, halos and
wraps fall elsewhere.  Predictions must be equal bit for bit.  The loss of the
doubled problem is the same mean: its pixel gradients are exactly half (a power
of two through every rounding), twice as many, so the weight gradients agree to
the rounding of their FP32 sums."""
import numpy as np
import pytest

from _gpu_util import banner

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


@pytest.mark.parametrize("axis", [1, 2])
@pytest.mark.parametrize("c0,B,H,W", [(8, 1, 8, 8), (16, 2, 24, 40), (24, 1, 72, 136), (32, 3, 8, 48), (40, 1, 16, 24),
                                      (64, 1, 16, 16)])
def test_doubled_image(c0, B, H, W, axis):
    from mantiis_amd.hip import DeviceArray, Net
    banner(f"network c0={c0}, {B}x{H}x{W} doubled along axis {axis}")
    rng = np.random.default_rng(7)
    x = rng.normal(0, 1, (B, H, W, 3)).astype(np.float32)
    t = rng.normal(0, 0.5, (B, H, W, 2)).astype(np.float32)
    m = (rng.uniform(size=(B, H, W)) > 0.4).astype(np.float32)
    res = []
    for k in (1, 2):
        xs, ts, ms = (np.concatenate([a] * k, axis=axis) for a in (x, t, m))
        net = Net(c0=c0, max_batch=B, max_h=xs.shape[1], max_w=xs.shape[2], seed=3)
        xd, td, md = (DeviceArray.from_numpy(np.ascontiguousarray(a)) for a in (xs, ts, ms))
        out = DeviceArray(xs.shape[:3] + (2,))
        net.forward(xd, out)
        loss = net.backward(td, md)
        res.append((out.numpy(), loss, net.grads()))
    (o1, l1, g1), (o2, l2, g2) = res
    assert np.array_equal(np.concatenate([o1, o1], axis=axis), o2)
    n = 2 * B * H * W  # terms of a sum, each addition rounded to 2^-24
    assert abs(l1 - l2) <= n * 2.0**-24 * abs(l1)
    assert rel(g2, g1) <= n * 2.0**-24
