"""Host copies of device planes: padded rows (width not a multiple of 64) go
through a dense staging copy, unpadded ones straight out; both must hand over
every cell of every plane.  The expected values come from the populations."""
import numpy as np
import pytest

from lbm_amd import LBM, Batch, SummaryStat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 3), (63, 5), (64, 7), (65, 3), (255, 9), (256, 4), (257, 6), (1021, 17)])
def test_planes_and_masks(nx, ny):
    print(f"case: read-back {nx}x{ny}", flush=True)
    rng = np.random.default_rng(nx * 1000 + ny)
    mask = (rng.random((ny, nx)) < 0.2).astype(np.uint8)
    odd = mask * np.uint8(1) + (mask == 0) * np.uint8(7)  # any value but 1 is fluid
    g, b = LBM(1.2, nx, ny, u_init=0.05), Batch([(nx, ny, 1.2, 0.05), (70, 5, 1.2, 0.05)])
    g.mask = odd
    b.set_mask(0, odd)
    assert np.array_equal(g.mask, mask)
    f = (rng.random((9, ny, nx)) * 0.1 + 0.1).astype(np.float32)
    g.write_f(f)
    assert np.array_equal(g.read_f(), f)
    ux = (f[2] + f[8]) - f[0] - f[6] + (f[5] - f[3])
    jx, jy, rho = g.moments()
    assert np.array_equal(jx, ux)
    gx, gy, grho = g.fields()[1], g.fields()[2], g.fields()[0]
    assert np.array_equal(grho, rho) and np.array_equal(gx, jx / rho) and np.array_equal(gy, jy / rho)
    g.step(1)
    assert np.array_equal(g.moments(lagged=True)[0], ux)
    assert np.array_equal(g.calculate_summary(SummaryStat.Ux), ux)
    g.custom_speed(0.05)
    g.step(4)
    b.step(4)
    for p, q in zip(g.moments(lagged=True), b.moments(0)):
        assert np.array_equal(p, q)
