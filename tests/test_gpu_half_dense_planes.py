"""sumall_except_dim<1> of half_t planes whose rows are of odd length and whose pixels are even in number:
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


# a segment per lane of one, four, sixteen and 64; fewer and more kept indices than are dealt out by segments;
# planes of two pixels and of whole 16-byte packs; the least work per kept index that takes the ring, and less
@pytest.mark.parametrize("n,c,h,w", [(1, 195, 512, 129), (3, 193, 148, 149), (16, 192, 66, 63), (20, 200, 58, 57),
                                     (65, 7, 34, 31), (33, 5, 40, 55), (32768, 3, 2, 1), (32767, 3, 2, 1), (65, 194, 32, 33)])
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
