"""A batch whose segment lists cannot be allocated (after a mask change, or for
another tile width) reports it and goes on with the lists it has: the same call
without the shortage, and calls that need no new list, give a fresh batch's bits."""
import ctypes
import gc
import os
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _settled_free():
    """The device's free bytes once what earlier objects gave back has arrived."""
    from lbm_amd import _native as N
    gc.collect()
    seen = []
    while len(seen) < 100 and (len(seen) < 4 or len(set(seen[-4:])) > 1):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert N.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        seen.append(free.value)
        time.sleep(0.02)
    return seen[-1]


def _batch(masks):
    from lbm_amd import Batch
    b = Batch([(300, 90, 1.6, 0.05), (700, 64, 1.5, 0.04)])
    for i, m in enumerate(masks):
        b.set_mask(i, m)
    return b


@pytest.mark.parametrize("widths", [(0, 2), (2, 4), (4, 0)])
def test_lists_that_cannot_be_made(widths):
    from lbm_amd import gen_circles
    from lbm_amd._native import LbmError, LBM_ENOMEM
    print(f"case: lists without memory {widths}", flush=True)
    masks = [gen_circles(300, 90, 1, 4, 4, 9), gen_circles(700, 64, 2, 5, 4, 9)]
    other = gen_circles(300, 90, 9, 6, 4, 9)
    b, ref = _batch(masks), _batch(masks)
    b.variant = ref.variant = widths[0]

    def short(call):
        os.environ["LBM_TEST_ALLOC_LIMIT"] = "512"
        try:
            with pytest.raises(LbmError) as e:
                call()
        finally:
            os.environ.pop("LBM_TEST_ALLOC_LIMIT", None)
        assert e.value.code == LBM_ENOMEM

    def same():
        for d in range(2):
            assert np.array_equal(b.read_f(d).view(np.uint32), ref.read_f(d).view(np.uint32))
    for o in (b, ref):
        o.step(5)
    same()
    b.variant = widths[1]  # another tile width: its lists do not fit
    short(lambda: b.step(3))
    held = [_batch(masks) for _ in range(2)]  # (memory given back by mistake would go to these)
    for h in held:
        h.variant = widths[0]
        h.step(2)
    b.variant = widths[0]  # back to the lists it has
    for o in (b, ref):
        o.step(4)
    same()
    for o in (b, ref):
        o.set_mask(0, other)
    short(lambda: b.step(2))
    for o in (b, ref):
        o.step(6)
    same()
    for o in [b, ref, *held]:
        o.close()


def test_a_tuning_call_that_fails_midway_restores_the_state():
    """The lists of the second tile width do not fit beside the first ones: the
    call fails after steps of its own, and the state, the moments and the step
    count are as before it."""
    from lbm_amd import Batch, PRECISION_F16S
    from lbm_amd import _native as N
    print("case: tuning call that fails midway", flush=True)
    X, Y = 8192, 16384  # a list of every segment: 17 MB
    o = [Batch([(X, Y, 1.6, 0.05)], precision=PRECISION_F16S) for _ in range(2)]
    for b in o:
        b.step(3)
    b, ref = o
    snapshot = 2 * 9 * X * Y * 2 + 3 * X * Y * 4
    os.environ["LBM_TEST_MEM_HIDDEN"] = str(_settled_free() - snapshot - (6 << 20))
    try:
        with pytest.raises(N.LbmError) as e:
            b.autotune(3)
    finally:
        os.environ.pop("LBM_TEST_MEM_HIDDEN", None)
    assert e.value.code == N.LBM_ENOMEM and b.variant == 0 and b.step_count == 3
    for p, q in zip(b.moments(0), ref.moments(0)):
        assert np.array_equal(p, q)
    for x in o:
        x.step(2)
    for p, q in zip(b.moments(0), ref.moments(0)):
        assert np.array_equal(p, q)
    for x in o:
        x.close()
