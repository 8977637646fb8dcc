"""A grid gives back every buffer its calls allocated: the device's free memory
after rounds of create, use of every buffer and destroy."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _free():
    from lbm_amd import _native as N
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert N.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_no_buffer_outlives_its_grid():
    from lbm_amd import LBM
    print("case: buffers after destroy", flush=True)

    def use():
        g = LBM(1.6, 2048, 1024)
        g.step(5)
        g.render()
        g.fields()
        g.conservation()
        g.snapshot()
        for slot in (0, 1):
            g.velocity_mark(slot)
        g.velocity_skill()
        g.close()
    use()  # what the library keeps for the process
    before = _free()
    for _ in range(12):
        use()
    # (a plane kept back would be 8 MB a grid, 100 MB in all)
    assert before - _free() < 16 << 20
