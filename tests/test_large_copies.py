"""Host copies large enough for the pinned chunks (4 MB out, 8 MB in), through
the public calls: every byte of odd sizes, in both directions, more than once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_state_images_round_trip():
    """Five pieces of padded planes in and out; each image as it was saved, and the
    restored grid steps on with the same bits."""
    from lbm_amd import LBM, gen_circles
    print("case: state images of 50 MB", flush=True)
    X, Y = 1021, 513
    a, b = LBM(1.6, X, Y), LBM(1.6, X, Y)
    a.mask = gen_circles(X, Y, 3, 6, 6, 30)
    a.custom_speed(0.06)
    for n in (7, 12):
        a.step(n)
        image = a.save_state()
        assert len(image) > 40 << 20
        b.load_state(image)
        assert b.save_state() == image
        a.step(9)
        b.step(9)
        assert np.array_equal(a.read_f().view(np.uint32), b.read_f().view(np.uint32))
    a.close()
    b.close()


def test_planes_in_and_out():
    from lbm_amd import LBM
    print("case: planes of 9 MB in and out", flush=True)
    X, Y = 1543, 1531  # one population plane: 9.4 MB
    g = LBM(1.2, X, Y)
    rng = np.random.default_rng(1)
    for _ in range(2):
        f = rng.random((9, Y, X), np.float32)
        g.write_f(f)
        assert np.array_equal(g.read_f(), f)
    g.close()


def test_network_inputs():
    """Fields of 8.4 MB in, 3.1 MB out: the images of a batch one by one give the
    batch's predictions."""
    from lbm_amd.surrogate import UNet
    print("case: network inputs of 8.4 MB", flush=True)
    rng = np.random.default_rng(2)
    many, one = UNet(4, 256, 256, seed=3), UNet(1, 256, 256, seed=3)
    for _ in range(2):
        x = rng.standard_normal((4, 256, 256, 8)).astype(np.float32)
        y = many.forward(x)
        for i in range(4):
            single = one.forward(x[i:i + 1])[0]
            # (another split of the sums at 4 images: bf16 roundings apart)
            assert np.linalg.norm(y[i] - single) <= 0.02 * np.linalg.norm(single)
    many.close()
    one.close()
