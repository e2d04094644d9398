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


@pytest.mark.parametrize("h,w", PLANES)
@pytest.mark.parametrize("k", [2, 3, 5])
def test_stride_one_pooling(G, O, h, w, k):
    planes = 5
    # few distinct values: equal maxima inside a window, zeros of both signs
    src = np.round(uniform(80 + k, (planes, h, w)) * f32(4)) / f32(4)
    grad = normal(81, (planes, h - k + 1, w - k + 1))
    for reducer in (MAX, SUM, MIN):
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
