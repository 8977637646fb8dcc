"""The f32 collision's velocities share one reciprocal while density and momenta
are of ordinary size; every other wave divides.  Populations over the whole f32
range, rest, sign changes, infinities and NaN among them, collide to the oracle's
bits (one step from a written state is the collision of every cell)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [(-1, 0), (-6, 3), (-30, 10), (-60, 40), (-140, 0), (0, 100)])
@pytest.mark.parametrize("kind", ["mixed signs", "positive", "sparse", "special"])
def test_collision_bits(scale, kind):
    from lbm_amd import LBM
    print(f"case: collision range 2^{scale} {kind}", flush=True)
    X, Y = 192, 64
    rng = np.random.default_rng(scale[1] * 1000 - scale[0])
    f = np.ldexp(rng.random((9, Y, X)) + 0.5, rng.integers(scale[0], scale[1] + 1, (9, Y, X))).astype(np.float32)
    if kind == "mixed signs":
        f *= rng.choice([-1.0, 1.0], f.shape).astype(np.float32)
    elif kind == "sparse":
        f *= rng.random(f.shape) < 0.4
    elif kind == "special":
        f[rng.random(f.shape) < 0.01] = np.inf
        f[rng.random(f.shape) < 0.01] = np.nan
    mask = np.zeros((Y, X), np.uint8)
    mask[0] = mask[-1] = 1
    g, r = LBM(1.3, X, Y), oracle.RefCPU(X, Y, 1.3)
    r.set_mask(mask.astype(np.uint32))
    for s in (0, 1):
        r.set_set(s, f)
    g.write_f(f)
    for n in (1, 2):  # one step: the collision of every cell; two more: through every step kernel
        g.step(n)
        r.step(n)
        got, exp = g.read_f(), r.state()
        same = (got.view(np.uint32) == exp.view(np.uint32)) | (np.isnan(got) & np.isnan(exp))
        assert same.all(), f"{(~same).sum()} values differ after a call of {n}"
