"""Stride-1 pooling and its gradient at the planes where the dispatch changes kernels (pixels of a plane,
width, rows of a strip). Bit-exact against the oracle."""
import numpy as np
import pytest

from checkers import MAX, MIN, SUM, Checker
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


PLANES = [(7, 7), (5, 24), (8, 23), (16, 16), (17, 15), (17, 16), (33, 17), (31, 33), (32, 32), (25, 41), (100, 14), (147, 7),
          (15, 64), (16, 64), (65, 65), (17, 256), (20, 257), (49, 31)]


def check(G, O, planes, h, w, k, reducers):
    # few distinct values: equal maxima inside a window, zeros of both signs
    src = np.round(uniform(80 + k, (planes, h, w)) * f32(4)) / f32(4)
    grad = normal(81, (planes, h - k + 1, w - k + 1))
    for reducer in reducers:
        want = np.empty(grad.shape, f32)
        O.pool(want, src, k, k, 1, 1, reducer)
        pooled = G.buffer(want.shape, f32)
        G.pool(pooled, G.to_device(src), k, k, 1, 1, reducer)
        assert_bits_equal(pooled.download(), want, f"pool {h}x{w} k{k} reducer {reducer}")
        want_dst = np.empty_like(src)
        O.unpool(want_dst, src, want, grad, k, k, 1, 1, reducer)
        dst = G.buffer(src.shape, f32)
        G.unpool(dst, G.to_device(src), pooled, G.to_device(grad), k, k, 1, 1, reducer)
        assert_bits_equal(dst.download(), want_dst, f"unpool {h}x{w} k{k} reducer {reducer}")


@pytest.mark.parametrize("h,w", PLANES)
@pytest.mark.parametrize("k", [2, 3, 5])
def test_stride_one_pooling(G, O, h, w, k):
    check(G, O, 5, h, w, k, (MAX, SUM, MIN))


# planes enough for full groups of them, on both sides of the pixels from which the columns kernel pays; strips
# of the 5x5 gradient by the waves there are; more low planes than waves of one turn, and as many
@pytest.mark.parametrize("planes,h,w,k", [(5200, 61, 17, 2), (5119, 61, 17, 3), (4200, 88, 16, 3), (5200, 34, 33, 2), (3100, 8, 160, 3),
                                          (300, 11, 130, 2), (2048, 7, 160, 5), (2049, 7, 160, 5), (2100, 40, 20, 5),
                                          (9000, 16, 20, 5), (700, 33, 16, 5), (40, 130, 64, 5), (2049, 9, 141, 5),
                                          (11364, 32, 33, 2)])
def test_stride_one_pooling_of_many_planes(G, O, planes, h, w, k):
    check(G, O, planes, h, w, k, (MAX,))


# few low planes of the 5x5 gradient and wide low planes of the forward pass, around the pixels at which the
# dispatch changes kernels
@pytest.mark.parametrize("planes,h,w,k", [(200, 6, 16, 5), (416, 6, 16, 5), (417, 6, 16, 5), (585, 8, 32, 5), (586, 8, 32, 5), (208, 9, 32, 5),
                                          (209, 9, 32, 5), (78, 16, 32, 5), (79, 16, 32, 5), (20, 9, 64, 5), (20, 9, 65, 5), (5, 17, 20, 5),
                                          (4300, 9, 155, 2), (4300, 11, 161, 3), (4300, 12, 146, 3), (4300, 10, 136, 2), (4300, 8, 195, 2)])
def test_stride_one_pooling_of_low_planes(G, O, planes, h, w, k):
    check(G, O, planes, h, w, k, (MAX,))
