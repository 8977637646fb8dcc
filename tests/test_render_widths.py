"""The colour plane at widths around its blocks of 256 cells, against the CPU
restatement of the colour maps bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("X", [5, 255, 256, 257, 513])
def test_render_at_block_edges(X):
    from lbm_amd import LBM
    from oracle import colormap_ref
    print(f"case: render width {X}", flush=True)
    rng = np.random.default_rng(X)
    mask = (rng.random((9, X)) < 0.2).astype(np.uint8)
    g = LBM(1.6, X, 9)
    g.mask = mask
    g.custom_speed(0.08)
    g.step(20)
    for cmap in range(3):
        for stat in (0, 4):
            rgb = g.render(stat, cmap)
            want = colormap_ref.colormap(cmap, g.calculate_summary(stat), mask)
            assert np.array_equal(rgb.view(np.uint32), want.view(np.uint32)), (cmap, stat)
    g.close()
