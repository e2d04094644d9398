"""sumall_except_dim<1> of half_t planes whose pixels are even in number, the rows of even and of odd length:
dense ones are walked as one row, pitched ones are not. Bit-exact against the oracle."""
import numpy as np
import pytest

from checkers import MAX, PLUSTO, SAVETO, SUM, Checker
from gpu_util import assert_bits_equal, f32, normal, uniform

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import mshadow_amd
    g = mshadow_amd.load_cases()
    g.set_device(0)
    return g


@pytest.fixture(scope="module")
def O():
    return Checker("orc")


# even rows, which dense planes walk as one row too: a segment per lane of one, four, sixteen and 64
EVEN = [(1, 195, 512, 130), (3, 193, 148, 150), (16, 192, 66, 64), (20, 200, 58, 58), (65, 7, 34, 32)]
# odd rows on the ring, dealt out by kept index (192 and more) and by segments (fewer), and where they stay
# with the kernel of expressions: fewer than 16 images, more than 256 kept indices, planes of fewer than 512
# pixels, less than 65536 elements per kept index
ODD = [(16, 192, 66, 63), (20, 200, 58, 57), (33, 5, 40, 55), (65, 194, 32, 33), (65, 7, 34, 31),
       (15, 200, 60, 75), (16, 200, 60, 75), (20, 256, 58, 57), (20, 257, 58, 57), (129, 194, 34, 15), (128, 194, 2, 257),
       (16, 194, 2, 2049), (16, 194, 2, 2047), (128, 3, 512, 1), (127, 3, 512, 1), (1, 195, 512, 129), (3, 193, 148, 149),
       (32768, 3, 2, 1), (32767, 3, 2, 1)]


@pytest.mark.parametrize("n,c,h,w", EVEN + ODD)
@pytest.mark.parametrize("extra", [0, 1])
def test_half_planes_of_odd_rows(G, O, n, c, h, w, extra):
    x = O.float2half(normal(80, (n, c, h, w)))
    src = G.to_device(x, extra)
    start = O.float2half(uniform(81, (c,)) + f32(2))
    scale = int(O.float2half(np.array([0.75], f32))[0])
    for reducer, saver in ((SUM, SAVETO), (SUM, PLUSTO), (MAX, SAVETO)):
        want, dst = start.copy(), G.to_device(start)
        O.reduce_keep_highdim(want, x, reducer, saver, 0.75)
        G.case_reduce_keep_highdim(dst, src, reducer, saver, scale)
        assert_bits_equal(dst.download(), want, f"{(n, c, h, w)} pitch+{extra}")
