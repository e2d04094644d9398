"""unpack_patch2col and pack_col2patch on images and patch rows shorter than a 16-byte pack: packs of the column matrix that
span patch rows and images, a thread a pixel of the image; every window that has an instance of its own, pitched images and
matrices, sizes around a workgroup. Bit-exact against the oracle."""
import numpy as np
import pytest

from checkers import Checker

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def G():
    import mshadow_amd
    g = mshadow_amd.load_cases()
    g.set_device(0)
    return g


@pytest.fixture(scope="module")
def O():
    return Checker("orc")


# n, c, h, w, (ky, kx), (sy, sx), (dy, dx), (pad_y, pad_x); images of up to 7 halves or 3 floats, patch rows of up to 7 and 3
GEOMETRIES = [
    (5, 3, 7, 7, (3, 3), (1, 1), (1, 1), (1, 1)), (37, 2, 7, 7, (1, 1), (1, 1), (1, 1), (0, 0)), (3, 5, 9, 7, (5, 5), (1, 1), (1, 1), (2, 2)),
    (4, 3, 30, 7, (7, 7), (2, 2), (1, 1), (3, 3)), (6, 2, 7, 5, (3, 3), (2, 2), (1, 1), (1, 1)), (2, 3, 16, 2, (3, 2), (1, 1), (1, 1), (1, 1)),
    (3, 2, 20, 1, (3, 1), (1, 1), (1, 1), (1, 0)), (2, 2, 13, 6, (4, 3), (3, 2), (1, 1), (0, 1)), (1, 1, 3, 3, (3, 3), (1, 1), (1, 1), (0, 0)),
    (9, 2, 12, 3, (5, 3), (1, 1), (1, 1), (2, 1)), (5, 4, 8, 14, (3, 3), (2, 2), (1, 1), (1, 1)), (4, 3, 11, 9, (3, 3), (1, 1), (1, 1), (0, 0)),
    (70, 3, 5, 15, (3, 3), (2, 2), (1, 1), (1, 1)), (3, 2, 12, 7, (3, 3), (1, 1), (2, 2), (2, 2)), (2, 2, 9, 7, (7, 7), (1, 1), (1, 1), (3, 3)),
    (2, 3, 15, 13, (4, 4), (4, 4), (1, 1), (1, 1)), (85, 2, 6, 2, (2, 2), (2, 2), (1, 1), (0, 0))]


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("geom", GEOMETRIES)
def test_both_directions(G, O, geom, half):
    n, c, h, w, k, s, d, p = geom
    rng = np.random.default_rng(n + 10 * h + w)
    oh, ow = ((a + 2 * q - (e * (b - 1) + 1)) // t + 1 for a, b, t, e, q in zip((h, w), k, s, d, p))
    dtype = np.uint16 if half else f32
    make = (lambda *shape: O.float2half(rng.standard_normal(shape).astype(f32))) if half else \
        (lambda *shape: rng.standard_normal(shape).astype(f32))
    args = (*k, *s, *d, *p)
    img = make(n, c, h, w)
    want = np.zeros((c * k[0] * k[1], n * oh * ow), dtype)
    O.im2col(want, img, *args)
    for pad in (0, 3):
        got = G.buffer(want.shape, dtype, pad)
        G.im2col(got, G.to_device(img, pad), *args)
        assert np.array_equal(got.download(), want), f"im2col pad {pad}"
    col = make(*want.shape)
    back = np.zeros((n, c, h, w), dtype)
    O.col2im(back, col, *args)
    for pad in (0, 3):
        got = G.buffer(back.shape, dtype, pad)
        G.col2im(got, G.to_device(col, pad), *args)
        assert np.array_equal(got.download(), back), f"col2im pad {pad}"
