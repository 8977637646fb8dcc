"""Loss weights that do not sum to a positive number are refused before the network
runs: such a call takes the copies' time and no more, leaves the parameters and
what the caller passed for the results alone, and the next call is a fresh
network's."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weight", [0.0, -1.0, float("nan")])
def test_refused_before_the_work(weight):
    from lbm_amd._native import LbmError, LBM_EINVAL
    from lbm_amd.surrogate import UNet
    print(f"case: refused gradient, weight {weight}", flush=True)
    B, H, W = 8, 256, 256
    rng = np.random.default_rng(5)
    x = rng.standard_normal((B, H, W, 8)).astype(np.float32)
    t = rng.standard_normal((B, H, W, 3)).astype(np.float32)
    ones, bad = np.ones((B, H, W), np.float32), np.full((B, H, W), weight, np.float32)
    net = UNet(B, H, W, seed=4)
    loss, grad = net.loss_grad(x, t, ones)

    def median(f):
        took = []
        for _ in range(7):
            t0 = time.perf_counter()
            f()
            took.append(time.perf_counter() - t0)
        return float(np.median(took))

    def refused():
        with pytest.raises(LbmError) as e:
            net.loss_grad(x, t, bad)
        assert e.value.code == LBM_EINVAL
    good = median(lambda: net.loss_grad(x, t, ones))
    short = median(refused)
    print(f"accepted {good * 1e6:.0f} us, refused {short * 1e6:.0f} us", flush=True)
    assert short < 0.7 * good  # (the work is two thirds of an accepted call)
    again, grad2 = net.loss_grad(x, t, ones)
    assert abs(again - loss) <= 1e-6 * loss and np.array_equal(grad2, grad)
    net.close()
