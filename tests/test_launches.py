"""lbm_launches / lbm_batch_launches name the launches a call makes: one a step
with the one-step kernels, fewer with several steps a launch."""
import ctypes

import pytest


def test_null_arguments():
    from lbm_amd import _native as N
    lib, n = N.load(), ctypes.c_uint32()
    assert lib.lbm_launches(None, 5, ctypes.byref(n)) == N.LBM_EINVAL
    assert lib.lbm_batch_launches(None, 5, ctypes.byref(n)) == N.LBM_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [False, True])
def test_launches_of_a_call(batch):
    from lbm_amd import LBM, Batch
    print(f"case: launches, batch {batch}", flush=True)
    o = Batch([(400, 160, 1.6, 0.05), (96, 64, 1.5, 0.04)]) if batch else LBM(1.6, 400, 160)
    several = 6 if batch else 8
    o.step(3)  # a stream is pending
    for variant in (None, several, several + 1, 0, several - 1):
        if variant is not None:
            o.variant = variant
        one = variant is not None and variant < several
        assert [o.launches(n) for n in (0, 1)] == [0, 1]
        for n in range(2, 70):
            k = o.launches(n)
            if one:
                assert k == n
            else:
                assert 2 * k <= n <= 8 * k
    o.close()


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [False, True])
def test_a_short_tuning_call_keeps_the_default(batch):
    """Two steps cannot compare the several-step kernels: they pick the variant
    of single steps and no more.  Three and above decide for every call; a
    variant that was set is replaced as before."""
    from lbm_amd import LBM, Batch
    print(f"case: short tuning call, batch {batch}", flush=True)
    o = Batch([(400, 160, 1.6, 0.05), (96, 64, 1.5, 0.04)]) if batch else LBM(1.6, 400, 160)
    several = 6 if batch else 8
    o.step(3)
    untuned = [o.launches(n) for n in range(70)]
    assert untuned[60] < 60
    best, _ = o.autotune(2)
    assert best < several and o.variant == best
    assert [o.launches(n) for n in range(70)] == untuned
    best, _ = o.autotune(3)
    assert o.variant == best and (o.launches(60) == 60) == (best < several)
    o.variant = several
    best, _ = o.autotune(2)
    assert best < several and o.launches(60) == 60
    o.close()
