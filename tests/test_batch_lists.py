"""A batch whose segment lists cannot be allocated (after a mask change, or for
another tile width) reports it and goes on with the lists it has: the same call
without the shortage, and calls that need no new list, give a fresh batch's bits."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
