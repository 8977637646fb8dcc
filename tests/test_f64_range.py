"""The FP64 collision's velocities share one reciprocal while density and momenta
are of ordinary size; every other wave divides.  Inflow speeds from none over
the subnormal to the absurd, and the unstable flows that the fast ones become
(densities near zero and below, infinities, NaN), against the CPU FP64 oracle
bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("u", [0.0, -0.0, 5e-324, 1e-300, -1e-160, 1e-30, -0.3, 0.9, -7.5, 300.0, 2.0 ** 10, 2.0 ** 21,
                               1e60, -1e160, float("inf"), float("nan")])
def test_collision_bits(u, mode):
    from lbm_amd import LBM64
    print(f"case: f64 range {u} mode {mode}", flush=True)
    X, Y = 150, 40
    rng = np.random.default_rng(7)
    mask = (rng.random((Y, X)) < 0.03).astype(np.uint8)
    for omega in (0.6, 1.9):
        g, o = LBM64(omega, X, Y, u, boundary=mode), oracle.Oracle64(X, Y, omega, u, mode)
        g.set_mask(mask)
        o.set_solid(mask)
        for n in (1, 2, 5, 30):
            g.step(n)
            o.step(n)
            got, exp = g.read_f(), o.state()
            same = (got.view(np.uint64) == exp.view(np.uint64)) | (np.isnan(got) & np.isnan(exp))
            assert same.all(), f"omega {omega}: {(~same).sum()} values differ after a call of {n}"
        g.close()
