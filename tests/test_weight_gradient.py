"""The weight- and bias-gradient kernel at the edges of its tiles (4 or 8 rows x
32 columns, 32 or 64 channels a block, rows shared by the waves or not).  Small
whole numbers keep every product and partial sum exact in f32, so the result
equals the float64 oracle."""
import numpy as np
import pytest

from oracle import conv_ref as cr
from tests.test_surrogate import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,Ci,Co", [(1, 1, 32, 32, 32), (2, 9, 64, 32, 32), (1, 5, 32, 64, 32), (2, 3, 64, 32, 64),
                                         (1, 4, 32, 64, 64), (3, 7, 96, 64, 64), (1, 2, 32, 128, 96),
                                         (2, 6, 32, 96, 128), (1, 65, 32, 32, 32)])
def test_weight_gradient_exact(N, H, W, Ci, Co):
    print(f"case: weight gradient {N}x{H}x{W} {Ci}->{Co}", flush=True)
    rng = np.random.default_rng(N * 1000 + H * 100 + Ci + Co)
    x = rng.integers(-4, 5, (N, H, W, Ci)).astype(np.float32)
    g = rng.integers(-4, 5, (N, H, W, Co)).astype(np.float32)
    got = _run(2, N, H, W, Ci, Co, x, g, None, None).reshape(9, Co, Ci)
    assert np.array_equal(got, cr.conv3x3_wgrad(x, g))


@pytest.mark.parametrize("B,H", [(1, 8), (3, 40)])
def test_head_bias_gradient(B, H):
    """The head's bias gradient is the sum over pixels of the loss gradient, which
    is stored in bf16; summed in f32 here and in float64 there."""
    from lbm_amd.surrogate import UNet
    print(f"case: head bias gradient {B}x{H}x256", flush=True)
    rng = np.random.default_rng(B + H)
    net = UNet(B, H, 256, seed=5)
    x = rng.standard_normal((B, H, 256, 8)).astype(np.float32)
    t = rng.standard_normal((B, H, 256, 3)).astype(np.float32)
    w = (rng.random((B, H, 256)) < 0.9).astype(np.float32)
    y = net.forward(x)
    _, grads = net.loss_grad(x, t, w)
    inv = np.float32(1.0 / w.astype(np.float64).sum())
    gout = cr.bf16(np.float32(2.0) * w[..., None] * (y - t) * inv)
    bound = B * H * 256 * 2.0 ** -24 * np.abs(gout).sum((0, 1, 2))
    assert (np.abs(grads[-32:-29] - gout.sum((0, 1, 2))) <= bound).all()
    assert not grads[-29:].any()


def test_minibatch_gradient_is_the_mean_of_its_images():
    """Loss and gradients of two images are the means of each image's own (equal
    weight sums), at a height that leaves one row at the coarsest level; the two
    runs split their sums differently, and bf16 rounding of the loss gradient
    (scaled by the weight sum, here a power of two apart) is the same in both."""
    from lbm_amd.surrogate import UNet
    print("case: minibatch gradient", flush=True)
    rng = np.random.default_rng(3)
    one, two = UNet(1, 8, 256, seed=9), UNet(2, 8, 256, seed=9)
    x = rng.standard_normal((2, 8, 256, 8)).astype(np.float32)
    t = rng.standard_normal((2, 8, 256, 3)).astype(np.float32)
    w = np.ones((2, 8, 256), np.float32)
    loss, grad = two.loss_grad(x, t, w)
    single = [one.loss_grad(x[i:i + 1], t[i:i + 1], w[i:i + 1]) for i in range(2)]
    mean = (single[0][1].astype(np.float64) + single[1][1]) / 2
    assert abs(loss - (single[0][0] + single[1][0]) / 2) < 1e-5 * loss
    assert np.linalg.norm(grad - mean) < 1e-5 * np.linalg.norm(mean)


def test_zero_loss_weights_are_refused():
    from lbm_amd._native import LbmError, LBM_EINVAL
    from lbm_amd.surrogate import UNet
    print("case: zero loss weights", flush=True)
    net = UNet(1, 8, 256, seed=2)
    before = net.get_params()
    x, t = np.zeros((1, 8, 256, 8), np.float32), np.zeros((1, 8, 256, 3), np.float32)
    with pytest.raises(LbmError) as e:
        net.train_step(x, t, np.zeros((1, 8, 256), np.float32), 1e-3)
    assert e.value.code == LBM_EINVAL
    assert np.array_equal(net.get_params(), before)
