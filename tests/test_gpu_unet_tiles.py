"""The U-Net convolutions' tile shapes: a batch large enough for the widest tile
(256 pixels x 64 channels) and its images one at a time (128 x 32) go through
different kernels with one order of sums, so their outputs are equal bit for
bit; the one-image outputs are checked against the restatement in test_unet.py.
The gradients of a batch are the mean of its images' gradients: with a power of
two of images every BF16 value only changes its exponent, so the two differ by
the FP32 sums over pixels, which the batch splits otherwise."""
import numpy as np
import pytest

from oracle import unet_ref as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,H,W,B", [(4, 128, 256, 16), (3, 64, 64, 9), (2, 32, 96, 33)])
def test_batch_equals_single_images(levels, H, W, B):
    from codeare_amd.warmstart import UNet
    rng = np.random.default_rng(levels * 100 + B)
    net = UNet(H, W, levels=levels, max_batch=B, seed=3)
    net.set_params(U.init_params(levels, 3))
    x = (rng.normal(size=(B, H, W)) + 1j * rng.normal(size=(B, H, W))).astype(np.complex64)
    y = net.forward(x)
    assert np.isfinite(y.view(np.float32)).all()
    for i in (0, B // 2, B - 1):
        assert np.array_equal(net.forward(x[i])[0], y[i])


@pytest.mark.parametrize("levels,H,W,B", [(4, 128, 256, 8), (2, 32, 96, 16), (3, 64, 64, 2),
                                           (5, 256, 256, 2), (6, 512, 512, 2)])   # 512 and 1024 channels
def test_batch_gradient_is_mean_of_images(levels, H, W, B):
    """Sums of 1e5 FP32 products in two orders: 1e-5 of the gradient's norm per layer block."""
    from codeare_amd.warmstart import UNet
    rng = np.random.default_rng(levels * 10 + B)
    net = UNet(H, W, levels=levels, max_batch=B, seed=4)
    net.set_params(U.init_params(levels, 4))
    x, t = ((rng.normal(size=(B, H, W)) + 1j * rng.normal(size=(B, H, W))).astype(np.complex64) for _ in range(2))
    loss = net.gradients(x, t)
    g = net.grads().astype(np.float64)
    one = np.zeros_like(g)
    ls = 0.0
    for i in range(B):
        ls += net.gradients(x[i], t[i]) / B
        one += net.grads().astype(np.float64) / B
    assert abs(loss - ls) <= 1e-9 * ls
    off = 0
    for ca, cb, co in U.layer_table(levels):
        for n in (9 * co * (ca + cb), co):
            e = np.linalg.norm(g[off:off + n] - one[off:off + n]) / np.linalg.norm(one[off:off + n])
            assert e <= 1e-5, (ca, cb, co, n, e)
            off += n
    assert np.linalg.norm(g[off:] - one[off:]) <= 1e-5 * np.linalg.norm(one[off:])
