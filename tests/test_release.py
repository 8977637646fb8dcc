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


def test_network_memory():
    """A network holds 36 MB of parameters, optimiser state and bf16 copies, its
    tensors, and workspaces for its own layers (55 MB in all at 8 x 256), not 38 MB
    more for a 256-channel layer at the full resolution, which it has none of."""
    from lbm_amd.surrogate import UNet
    print("case: network memory", flush=True)
    first = UNet(1, 8, 256, seed=1)  # (modules and the runtime's own buffers)
    nets, before = [], _free()
    for _ in range(4):
        nets.append(UNet(1, 8, 256, seed=1))
    held = (before - _free()) / 4
    print(f"held per network: {held / 2 ** 20:.1f} MB", flush=True)
    for n in nets + [first]:
        n.close()
    assert held < 64 << 20
