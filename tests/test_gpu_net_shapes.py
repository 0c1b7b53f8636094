"""The network's convolution kernels at the shapes where their tiles end:
images that are no multiple of the 16-pixel tile or smaller than its halo,
channel counts that leave output tiles partly filled or pad them (40: five
tiles), and layers too wide for an LDS tile (64: 768 input channels)."""
import os
import sys

import numpy as np
import pytest

from _gpu_util import banner

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import unet_oracle as U  # noqa: E402

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


@pytest.mark.parametrize("c0,B,H,W", [(8, 1, 8, 8), (16, 2, 24, 40), (24, 1, 72, 136), (32, 3, 8, 48), (40, 1, 16, 24),
                                      (64, 1, 16, 16)])
def test_forward_backward_shapes(c0, B, H, W):
    from mantiis_amd.hip import DeviceArray, Net
    banner(f"network c0={c0}, {B}x{H}x{W}: forward, loss and every gradient vs the CPU oracle")
    net = Net(c0=c0, max_batch=B, max_h=H, max_w=W, seed=3)
    rng = np.random.default_rng(7)
    x = rng.normal(0, 1, (B, H, W, 3)).astype(np.float32)
    t = rng.normal(0, 0.5, (B, H, W, 2)).astype(np.float32)
    m = (rng.uniform(size=(B, H, W)) > 0.4).astype(np.float32)
    xd, td, md = (DeviceArray.from_numpy(a) for a in (x, t, m))
    out = DeviceArray((B, H, W, 2))
    net.forward(xd, out)
    loss = net.backward(td, md)
    g = net.grads()
    o_out, o_loss, o_g = U.forward_backward(net.params(), c0, x, t, m, use_bf16=True)
    # device and oracle differ in FP32 summation order, which can move an
    # activation by one BF16 rounding (2^-9 relative)
    assert rel(out.numpy(), o_out) < 2.0**-9 and abs(loss - o_loss) <= 2.0**-8 * abs(o_loss)
    off = 0
    for i, (cin, cout, k, relu) in enumerate(U.layer_table(c0)):
        nw = k * k * cout * cin
        # two roundings a layer on the way back, 15 layers
        assert rel(g[off:off + nw], o_g[off:off + nw]) < 15 * 2.0**-8, (i, "weights")
        assert rel(g[off + nw:off + nw + cout], o_g[off + nw:off + nw + cout]) < 15 * 2.0**-8, (i, "bias")
        off += nw + cout
