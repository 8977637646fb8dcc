"""Several steps per launch (k_tile): both parity sets and the lagged moments
equal the one-step kernel's bit for bit, at widths and heights around the
regions' (64 columns; 16, 32 or 36 rows), with rows open or walled, random
obstacles, from a written state (S-form) and from a stepped one (P-form), by the
default path and by both variants, for calls of one to several launches."""
import numpy as np
import pytest

from tests.test_gpu_parity import both_sets, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("nx,ny", [(3, 3), (62, 15), (63, 14), (64, 16), (65, 31), (117, 33), (119, 35), (121, 37),
                                   (200, 70)])
def test_tile_equals_one_step(nx, ny, precision, boundary):
    from lbm_amd import LBM
    print(f"case: tile {nx}x{ny} precision {precision} boundary {boundary}", flush=True)
    rng = np.random.default_rng(nx * 100 + ny)
    for walls in (True, False):
        mask = (rng.random((ny, nx)) < 0.06).astype(np.uint8)
        if walls:
            mask[0] = mask[-1] = 1
        noise = 1 + 0.01 * rng.standard_normal((9, ny, nx))
        grids = []
        for variant in (0, None, 8, 9):
            g = LBM(1.6, nx, ny, precision=precision, boundary=boundary)
            g.mask = mask
            g.custom_speed(0.07)
            g.write_f((g.read_f() * noise).astype(np.float32))
            if variant is not None:
                g.variant = variant
            grids.append(g)
        for n in (2, 3, 8, 9, 1, 25):
            for g in grids:
                g.step(n)
            want, mom = both_sets(grids[0]), grids[0].moments(True)
            for g, v in zip(grids[1:], ("default", 8, 9)):
                assert np.array_equal(both_sets(g), want), (walls, v, n)
                assert all(same_bits(a, b) for a, b in zip(g.moments(True), mom)), (walls, v, n)
        for g in grids:
            g.paint(np.array([nx // 2 + nx * (ny // 2), 1], np.uint32))  # a mask change inside the run
            g.step(6)
        want = both_sets(grids[0])
        for g, v in zip(grids[1:], ("default", 8, 9)):
            assert np.array_equal(both_sets(g), want), (walls, v, "after paint")
            g.close()
        grids[0].close()


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("boundary", [0, 1])
def test_batch_tile_equals_one_step(precision, boundary):
    """Seventy domains around the regions' sizes (more than one wave of block
    counts to search): the default path and both tile variants give the one-step
    variants' populations and moments, through mask changes between calls."""
    from lbm_amd import Batch
    print(f"case: batch tile precision {precision} boundary {boundary}", flush=True)
    rng = np.random.default_rng(precision * 2 + boundary)
    sizes = [(3, 3), (62, 15), (63, 14), (64, 16), (65, 31), (121, 37), (200, 70)] * 10
    doms = [(nx, ny, rng.uniform(1.2, 1.7), rng.uniform(0.02, 0.08)) for nx, ny in sizes]
    batches = []
    for variant in (0, None, 6, 7):
        b = Batch(doms, precision=precision, boundary=boundary)
        if variant is not None:
            b.variant = variant
        batches.append(b)
    for n in (8, 9, 2, 1, 25, 6):
        for i in rng.choice(len(doms), 40, replace=False):
            mask = (rng.random((doms[i][1], doms[i][0])) < 0.06).astype(np.uint8)
            for b in batches:
                b.set_mask(i, mask)
        for b in batches:
            b.step(n)
        for i in range(0, len(doms), 3):
            want = batches[0].moments(i)
            for b, v in zip(batches[1:], ("default", 6, 7)):
                assert all(same_bits(p, q) for p, q in zip(b.moments(i), want)), (i, v, n)
    for i in range(len(doms)):
        want = batches[0].read_f(i)
        for b, v in zip(batches[1:], ("default", 6, 7)):
            assert same_bits(b.read_f(i), want), (i, v)
    for b in batches:
        b.close()
