"""The ReLU gate in the epilogue of the input gradient, for every kernel that
conv3_plan picks by itself (at the smallest image that takes it, with partial
tiles) and for the pass that adds a split's partial sums.  Small whole numbers
make every sum exact, so the result equals the oracle's rounded to bf16; the
activations hold zeros of both signs, tiny and huge values, infinities and NaN."""
import numpy as np
import pytest

from oracle import conv_ref as cr
from tests.test_surrogate import _run

pytestmark = pytest.mark.gpu

GATE = 1 << 14


@pytest.mark.parametrize("N,H,W,Ci,Co", [(1, 253, 256, 32, 32), (5, 229, 256, 32, 32),  # k_conv3_rows, one and two tiles a run
                                         (1, 125, 256, 64, 32), (3, 178, 256, 64, 32),  # two waves of channels
                                         (1, 7, 64, 32, 32), (1, 93, 128, 96, 32),      # one input chunk, small
                                         (1, 187, 256, 64, 64), (2, 125, 128, 128, 64),  # LDS weights, two by two
                                         (1, 93, 128, 32, 64), (1, 61, 256, 96, 96),    # LDS weights, one by one
                                         (1, 5, 32, 64, 128), (1, 9, 32, 32, 256),      # split input channels
                                         (2, 33, 96, 96, 64)])
def test_gated_input_gradient_exact(N, H, W, Ci, Co):
    print(f"case: gated input gradient {N}x{H}x{W} {Co}->{Ci}", flush=True)
    rng = np.random.default_rng(H + 3 * Ci + Co)
    g = rng.integers(-3, 4, (N, H, W, Co)).astype(np.float32)
    w = rng.integers(-2, 3, (9, Co, Ci)).astype(np.float32)
    act = rng.integers(-3, 4, (N, H, W, Ci)).astype(np.float32)
    odd = np.array([0.0, -0.0, 1e-38, -1e-38, 3e38, -3e38, np.inf, -np.inf, np.nan], np.float32)
    at = rng.random(act.shape) < 0.05
    act[at] = rng.choice(odd, int(at.sum()))
    want = np.where(cr.bf16(act) > 0, cr.bf16(cr.conv3x3_dgrad(g, w)), 0.0)
    got = _run(1 | GATE, N, H, W, Ci, Co, g, act, w, None).reshape(want.shape)
    assert np.array_equal(got, want)


def test_a_gate_needs_a_gradient_and_an_activation():
    from lbm_amd import _native as Nn
    import ctypes
    lib = Nn.load()
    a = np.zeros(9 * 32 * 32 + 32 * 32 * 32, np.float32)
    p = a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
    for mode, act in ((GATE, p), (2 | GATE, p), (1 | GATE, None), (1 | 1 << 15, p)):
        assert lib.lbm_conv3x3_test(mode, 1, 2, 32, 32, 32, p, act, p, None, p, 0) == Nn.LBM_EINVAL
