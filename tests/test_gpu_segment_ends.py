"""Sums over dense planes by waves of eight and sixteen planes: the ends of planes behind their last whole slice, a few packs
at a time with floats selected by the plane's length, halves by whole packs and one by one, of every length modulo two
slices; and shapes of few kept indices, of 5 to 16 planes an index and of one, which other kernels had. Bit-exact against the
oracle, sums, maxima and minima, -0 and NaN among the values."""
import numpy as np
import pytest

from checkers import MAX, MIN, SAVETO, SUM, Checker

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


# (n, c, len): ends of 0 to 63 floats and 0 to 127 halves, with and without a whole slice in front (7 kept indices of 9 planes
# for short planes, 200 of 7 for the others), eight planes a wave from 512 values on
ENDS = [(70, 9, n) for n in (8, 9, 11, 15, 16, 17, 23, 24, 31, 33)] + \
       [(7, 200, n) for n in (64, 65, 71, 72, 73, 79, 80, 127, 128, 129, 135, 143, 191, 255, 257, 511)] + \
       [(7, 200, n) for n in (512, 513, 520, 575, 577, 639, 640, 641, 767, 769)]
ROUTES = [(6, 1519, 320), (12, 300, 592), (16, 400, 140), (5, 260, 1300), (9, 16, 1280), (24, 24, 2208), (28, 184, 1536), (47, 40, 640),
          (17, 56, 672), (2, 700, 2048), (3, 270, 2000), (1, 536, 700), (1, 72, 1392), (114, 246, 600), (2, 52, 1536), (64, 320, 72)]


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n,c,length", ENDS + ROUTES)
def test_planes(G, O, n, c, length, half):
    rng = np.random.default_rng(n * 3 + c + length)
    x = rng.standard_normal((n, c, length, 1)).astype(f32)
    x[:, 1::6] = -0.0
    x[:, 2::7, -1] = 3.0           # the last value decides
    x[n // 2, 3, -1] = np.nan
    if half:
        x = O.float2half(x)
    src = G.to_device(x)
    dtype = np.uint16 if half else f32
    for reducer in (SUM, MAX, MIN):
        want, dst = np.zeros(c, dtype), G.buffer((c,), dtype)
        with np.errstate(all="ignore"):
            O.reduce_keep_highdim(want, x, reducer, SAVETO, 1.0)
        if half:
            G.case_reduce_keep_highdim(dst, src, reducer, scale=0x3C00)
        else:
            G.reduce_keep_highdim(dst, src, reducer)
        got = dst.download()
        bits = np.uint16 if half else np.uint32
        as_float = (lambda v: v.view(np.float16)) if half else (lambda v: v)
        same = (got.view(bits) == want.view(bits)) | (np.isnan(as_float(got)) & np.isnan(as_float(want)))
        assert same.all(), (reducer, [(i, got[i], want[i]) for i in np.flatnonzero(~same)[:5]])
