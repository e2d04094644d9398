"""pool<Reducer> on half_t tensors: the windows with a kernel of their own and their neighbours that have
none, rows of four outputs and more, strips that end inside a plane, values whose order counts - zeros
of both signs, NaN, infinities. Bit-exact against the oracle."""
import numpy as np
import pytest

from checkers import MAX, MIN, SUM, Checker
from gpu_util import f32, uniform

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


WINDOWS = [(2, 1), (3, 1), (5, 1), (2, 2), (3, 2), (5, 2), (4, 2), (3, 3)]


def test_half_pool_of_many_narrow_planes(G, O):
    """2x2 by two on rows of ten, more of them than fit L2: the map kernel"""
    img = O.float2half(uniform(95, (22000, 64, 10)))
    want = np.empty((22000, 32, 5), np.uint16)
    O.pool(want, img, 2, 2, 2, 2, MAX)
    dst = G.buffer(want.shape, np.uint16)
    G.case_pool(dst, G.to_device(img), 2, 2, 2, 2, MAX)
    assert np.array_equal(dst.download(), want)


@pytest.mark.parametrize("k,s", WINDOWS)
@pytest.mark.parametrize("h,w", [(5, 5), (7, 11), (9, 10), (12, 13), (13, 13), (17, 33), (24, 8), (40, 67)])
def test_half_pool(G, O, h, w, k, s):
    planes = 7
    img = O.float2half(uniform(90 + w, (planes, h, w)))
    rng = np.random.default_rng(h * w)
    odd = img[3:6].reshape(3, -1)   # three planes with what the order of comparisons shows
    odd[0][rng.random(h * w) < 0.7] = 0x8000
    odd[0][rng.random(h * w) < 0.3] = 0x0000
    odd[1][rng.random(h * w) < 0.1] = 0x7e01
    odd[1][rng.random(h * w) < 0.1] = 0xfd00   # a signalling NaN
    odd[2][:] = rng.choice(np.array([0xfc00, 0x7c00, 0xfbff, 0x0001, 0x8001], np.uint16), h * w)
    src = G.to_device(img, 3)
    ph, pw = (h - k) // s + 1, (w - k) // s + 1
    for reducer in (MAX, MIN, SUM):
        want = np.empty((planes, ph, pw), np.uint16)
        O.pool(want, img, k, k, s, s, reducer)
        dst = G.buffer(want.shape, np.uint16, 1)
        G.case_pool(dst, src, k, k, s, s, reducer)
        got = dst.download()
        nan = np.isnan(O.half2float(want).astype(f32))
        assert np.array_equal(np.isnan(O.half2float(got).astype(f32)), nan)
        assert np.array_equal(got[~nan], want[~nan]), f"{h}x{w} k{k} s{s} reducer {reducer}"


# threads enough for strips of eight, four, two rows of outputs and of one (half of that with a step of two)
@pytest.mark.parametrize("planes", [7400, 4500, 2300, 300])
@pytest.mark.parametrize("k,s", WINDOWS[:6])
def test_half_pool_strips(G, O, planes, k, s):
    h, w = 21, 23
    img = O.float2half(uniform(96, (planes, h, w)))
    img[::7, 3:9, 5] = 0x8000
    img[::11, 17, ::6] = 0x7e01
    ph, pw = (h - k) // s + 1, (w - k) // s + 1
    want = np.empty((planes, ph, pw), np.uint16)
    O.pool(want, img, k, k, s, s, MAX)
    dst = G.buffer(want.shape, np.uint16)
    G.case_pool(dst, G.to_device(img), k, k, s, s, MAX)
    got = dst.download()
    nan = np.isnan(O.half2float(want).astype(f32))
    assert np.array_equal(np.isnan(O.half2float(got).astype(f32)), nan)
    assert np.array_equal(got[~nan], want[~nan])
