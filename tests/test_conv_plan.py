"""The block shapes the 3x3 convolution picks by itself, at the smallest image
that takes each and with partial tiles in its rows.  Small whole numbers keep
every product and partial sum exact in f32, so the result equals the oracle; an
image a few rows shorter takes the neighbouring choice and must agree as well."""
import numpy as np
import pytest

from oracle import conv_ref as cr
from tests.test_surrogate import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,Ci,Co", [(4, 253, 256, 32, 64), (1, 125, 256, 32, 64),  # two waves of channels
                                         (1, 124, 256, 32, 64), (1, 187, 256, 64, 64),  # LDS weights, two by two
                                         (1, 184, 256, 64, 64), (1, 190, 256, 64, 64),
                                         (5, 228, 256, 32, 32), (3, 178, 256, 32, 64),  # runs of two row tiles
                                         (1, 91, 128, 96, 128), (1, 7, 32, 64, 96)])
def test_chosen_block_shapes_exact(N, H, W, Ci, Co):
    print(f"case: conv plan {N}x{H}x{W} {Ci}->{Co}", flush=True)
    rng = np.random.default_rng(H + Ci + Co)
    x = rng.integers(-4, 5, (N, H, W, Ci)).astype(np.float32)
    w = rng.integers(-3, 4, (9, Co, Ci)).astype(np.float32)
    b = rng.integers(-9, 10, Co).astype(np.float32)
    want = cr.conv3x3(x, w, b)
    got = _run(0, N, H, W, Ci, Co, x, None, w, b).reshape(want.shape)
    assert np.array_equal(got, want)
    if H % 2 == 0:  # with the average pool: the chosen shape may differ, the stored output not
        both = _run(1 << 12, N, H, W, Ci, Co, x, None, w, b, size=want.size * 5 // 4)
        full = both[:want.size].reshape(want.shape)
        assert np.array_equal(full, cr.bf16(want))
        pool = cr.bf16(np.float32(0.25) * ((full[:, 0::2, 0::2] + full[:, 0::2, 1::2]) +
                                           (full[:, 1::2, 0::2] + full[:, 1::2, 1::2])))
        assert np.array_equal(both[want.size:].reshape(pool.shape), pool)
