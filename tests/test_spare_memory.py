"""The two sets a small untuned grid or batch takes unasked stand in nothing's way
on a card that is nearly full: what could be allocated without them -- a variant
of several steps, an autotuner's snapshot, the grid's own buffers -- still can,
and the state's bits do not depend on it.  The card is filled by a count the
library keeps (LBM_TEST_MEM_HIDDEN); no memory is really taken."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
X, Y = 1536, 1024
SET = 9 * X * (Y + 2) * 4  # a state set with its two spare rows
PLANE = X * Y * 4
SLACK = 12 * MB  # allocations are rounded up to 2 MB


class only_free:
    """All but `bytes` of the device's free memory hidden from the library."""

    def __init__(self, bytes_):
        self.bytes = int(bytes_)

    def __enter__(self):
        from lbm_amd import _native as N
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert N.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        os.environ["LBM_TEST_MEM_HIDDEN"] = str(free.value - self.bytes)

    def __exit__(self, *exc):
        os.environ.pop("LBM_TEST_MEM_HIDDEN", None)


def _grid():
    from lbm_amd import LBM, gen_circles
    g = LBM(1.6, X, Y)
    g.mask = gen_circles(X, Y, 5, 8, 8, 40)
    g.custom_speed(0.06)
    return g


def _batch():
    from lbm_amd import Batch, gen_circles
    b = Batch([(X, 700, 1.6, 0.06), (X, Y - 700, 1.5, 0.05)])
    b.set_mask(0, gen_circles(X, 700, 5, 8, 8, 40))
    return b


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


@pytest.mark.parametrize("make,several", [(_grid, 8), (_batch, 6)])
def test_a_several_step_variant_while_the_default_pair_is_held(make, several):
    """Less than two sets are free, but the object holds a pair already."""
    print(f"case: variant {several} on a full card", flush=True)
    g, ref = make(), make()
    for o in (g, ref):
        o.step(20)
    with only_free(SET):
        g.variant = several
    assert g.variant == several
    for o in (g, ref):
        o.step(21)
    r = (lambda o: o.read_f()) if make is _grid else (lambda o: o.read_f(0))
    assert _same(r(g), r(ref))
    g.close()
    ref.close()


@pytest.mark.parametrize("make", [_grid, _batch])
def test_autotuning_while_the_default_pair_is_held(make):
    """The snapshot (two sets and the moments) does not fit beside the pair."""
    print("case: autotune on a full card", flush=True)
    g, ref = make(), make()
    for o in (g, ref):
        o.step(20)
    with only_free(SET + 3 * PLANE):
        best, ms = g.autotune(5)
    assert g.variant == best and np.isfinite(ms[0])
    for o in (g, ref):
        o.step(21)
    r = (lambda o: o.read_f()) if make is _grid else (lambda o: o.read_f(0))
    assert _same(r(g), r(ref))
    g.close()
    ref.close()


def test_a_grid_leaves_room_for_its_own_buffers():
    """Created where two more sets fit but little else would after them: every
    call that needs memory of its own is still answered, with the same bits."""
    print("case: grid on a full card", flush=True)
    def program(g):
        g.step(20)
        g.snapshot()
        g.velocity_mark(0)
        out = [*g.fields(), g.render()]
        g.step(21)
        return out + [g.read_f(), np.float32(g.velocity_change())]

    # the grid's own allocations, then its snapshot, moments, staging, colours, marks
    own = 2 * SET + 4 * PLANE + 2 * X * Y
    later = 2 * SET + 3 * PLANE + 3 * PLANE + 4 * PLANE + 3 * PLANE + 4 * PLANE
    with only_free(own + later + 3 * SLACK):
        g = _grid()
        got = program(g)
    ref = _grid()
    assert all(_same(p, q) for p, q in zip(got, program(ref)))
    g.close()
    ref.close()
