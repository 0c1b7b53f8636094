"""The network against the CPU oracle at the widths and sizes that select every
form of the convolution kernels: one to six output-channel tiles per block and
several blocks of them, partly filled tiles (40: five), operands from memory
(64 and above: 768 input channels), and tiles of 4, 8 and 16 rows (images large
enough for two blocks per CU).

With general weights two correct networks part ways: an FP32 sum in another
order now and then falls on the other side of a BF16 rounding or of a ReLU, and
the next layers multiply that.  Here every FP32 sum is exact, whatever its
order: inputs and biases are small integers, each output channel has eight
weights +-1 somewhere among its (offset, channel) terms and zeros elsewhere, and
the output's error is a small integer over a power of two, so that values stay
multiples of 2^-6 below 2^18 on the way forward (three poolings, 2 bits each)
and within as many bits on the way back.  The predictions must then be the
oracle's bit for bit, and so is every BF16 operand of the backward products.  A
weight gradient is an FP32 sum of n = B H W such products, each addition rounded
to 2^-24; a channel, offset or tile out of place changes it by order one."""
import os
import sys

import numpy as np
import pytest

from _gpu_util import banner

pytestmark = pytest.mark.gpu
sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import unet_oracle as U  # noqa: E402


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


def params(c0, rng):
    out = []
    for cin, cout, k, _ in U.layer_table(c0):
        w = np.zeros((k * k, cout, cin), np.float32)
        for co in range(cout):
            for t in rng.choice(k * k * cin, 8, replace=False):
                w[t // cin, co, t % cin] = rng.choice([-1.0, 1.0])
        out += [w.reshape(-1), rng.integers(-1, 2, cout).astype(np.float32)]
    return np.concatenate(out)


def problem(c0, B, H, W):
    """Parameters, input, target, mask, and the oracle's output, loss and gradients."""
    rng = np.random.default_rng(c0 + H)
    p = params(c0, rng)
    x = rng.integers(-1, 3, (B, H, W, 3)).astype(np.float32)
    m = np.zeros(B * H * W, np.float32)  # a power of two of ones
    m[rng.permutation(m.size)[:1 << (m.size.bit_length() - 2)]] = 1.0
    m = m.reshape(B, H, W)
    out = U.forward_backward(p, c0, x, np.zeros((B, H, W, 2), np.float32), m, need_grad=False)[0]
    t = out - rng.integers(-3, 4, out.shape).astype(np.float32)
    return p, x, t, m, U.forward_backward(p, c0, x, t, m)


@pytest.mark.parametrize("c0,B,H,W", [(8, 1, 8, 8), (16, 3, 40, 24), (24, 1, 16, 24), (32, 2, 24, 40), (40, 1, 16, 24),
                                      (64, 1, 16, 16), (96, 1, 8, 16), (8, 2, 256, 256), (24, 1, 256, 256),
                                      (24, 2, 256, 256)])
def test_network_matches_oracle(c0, B, H, W):
    from mantiis_amd.hip import DeviceArray, Net
    banner(f"network c0={c0}, {B}x{H}x{W}: forward, loss and every layer's gradient vs the CPU oracle")
    p, x, t, m, (o_out, o_loss, o_g) = problem(c0, B, H, W)
    net = Net(c0=c0, max_batch=B, max_h=H, max_w=W, seed=3)
    net.set_params(p)
    xd, td, md = (DeviceArray.from_numpy(a) for a in (x, t, m))
    out = DeviceArray((B, H, W, 2))
    net.forward(xd, out)
    loss = net.backward(td, md)
    g = net.grads()
    net.close()
    assert np.array_equal(out.numpy(), o_out)
    n = B * H * W
    assert abs(loss - o_loss) <= 2 * n * 2.0**-24 * o_loss
    off = 0
    for i, (cin, cout, k, _) in enumerate(U.layer_table(c0)):
        for name, size in (("weights", k * k * cout * cin), ("biases", cout)):
            e = rel(g[off:off + size], o_g[off:off + size])
            print("layer", i, name, "rel", e)
            assert e <= n * 2.0**-24, (i, name)
            off += size
