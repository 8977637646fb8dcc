"""The FP64 solver's several steps per launch against the CPU FP64 oracle bit
for bit, at sizes that take each block shape, with regions that end at every
edge of the grid, both outlets, and call lengths of one, three and more launches."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny", [(64, 16), (63, 15), (129, 700), (655, 331), (1501, 803)])
def test_block_shapes_and_launch_counts(nx, ny, mode):
    from lbm_amd import LBM64
    print(f"case: f64 tile {nx}x{ny} mode {mode}", flush=True)
    rng = np.random.default_rng(nx + ny + mode)
    g, o = LBM64(1.5, nx, ny, 0.06, boundary=mode), oracle.Oracle64(nx, ny, 1.5, 0.06, mode)
    mask = (rng.random((ny, nx)) < 0.02).astype(np.uint8)
    mask[ny // 3:ny // 2, nx // 3:nx // 2] = 1  # rows of a wave that are solid throughout
    g.set_mask(mask)
    o.set_solid(mask)
    for n in (8, 11, 25):
        g.step(n)
        o.step(n)
        assert np.array_equal(g.read_f().view(np.uint64), o.state().view(np.uint64)), f"after a call of {n}"
