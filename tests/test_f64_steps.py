"""The FP64 solver's fused passes against the CPU FP64 oracle bit for bit: calls
of odd and even length, grids open at every edge, masks changed between calls,
both outlets."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny", [(3, 3), (40, 5), (257, 33)])
def test_call_lengths_and_mask_changes(nx, ny, mode):
    from lbm_amd import LBM64
    print(f"case: f64 call lengths {nx}x{ny} mode {mode}", flush=True)
    rng = np.random.default_rng(nx + ny + mode)
    g, o = LBM64(1.3, nx, ny, 0.07, boundary=mode), oracle.Oracle64(nx, ny, 1.3, 0.07, mode)
    for n in (1, 2, 3, 4, 9, 10, 0, 1):
        mask = (rng.random((ny, nx)) < 0.15).astype(np.uint8)
        g.set_mask(mask)
        o.set_solid(mask)
        g.step(n)
        o.step(n)
        assert np.array_equal(g.read_f().view(np.uint64), o.state().view(np.uint64)), f"after a call of {n}"
