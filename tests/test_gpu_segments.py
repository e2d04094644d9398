"""sumall_except_dim<1> and its kin over dense planes by ReduceSegmentsKernel: bit for bit the oracle's two serial levels, at the
edges of what a wave and a slice take and of the rule that sends shapes there."""
import numpy as np
import pytest

from checkers import MAX, MIN, MINUSTO, PLUSTO, SAVETO, SUM, Checker
pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def G():
    import mshadow_amd
    g = mshadow_amd.load_cases()
    assert g.device_count() >= 1, "no GPU visible"
    g.set_device(0)
    return g


@pytest.fixture(scope="module")
def O():
    return Checker("orc")


# slices of 64 and 128 floats (128 and 256 halves): shorter planes, whole slices, one element more; n around whole groups of
# sixteen lanes, one round of a workgroup and several; kept indices that do not fill the last workgroup; and neighbours of
# each that the rule leaves to the other kernels
SHAPES = [(100, 100, 1, 4), (100, 100, 1, 8), (33, 270, 1, 9), (17, 300, 3, 21), (17, 301, 8, 8), (17, 302, 5, 13), (48, 257, 1, 127),
          (49, 258, 1, 128), (49, 259, 3, 43), (3, 700, 16, 16), (2, 1100, 257, 1), (4, 800, 1, 255), (1, 1100, 29, 31), (1, 2049, 20, 20),
          (250, 300, 9, 9), (300, 60, 7, 7), (257, 90, 10, 11), (2048, 9, 5, 5), (2049, 9, 5, 5), (600, 193, 2, 33), (700, 300, 4, 24),
          (70, 384, 31, 33), (20, 400, 50, 51), (19, 304, 72, 80), (5, 600, 130, 101), (13, 530, 74, 69), (60, 190, 30, 50), (16, 400, 15, 10),
          # few kept indices: eight and sixteen planes a wave, one round of sixteen waves and several, more planes than the split
          # kernel has room for, and shapes that it takes
          (128, 17, 28, 28), (129, 17, 28, 28), (256, 16, 32, 32), (300, 9, 24, 25), (2048, 9, 16, 16), (1100, 61, 9, 7), (1101, 60, 11, 12),
          (2048, 5, 28, 28), (48, 200, 41, 40), (44, 250, 40, 40)]


@pytest.mark.parametrize("n,c,h,w", SHAPES)
def test_planes_are_summed_in_order(G, O, n, c, h, w):
    rng = np.random.default_rng(n * 7 + c)
    x = rng.standard_normal((n, c, h, w)).astype(f32)
    x[:, 1::5] *= 1e-3
    x[n // 2, 2, -1, -1] = np.inf
    x[n // 3, 3, h // 2, 0] = np.nan
    x[:, 4] = -0.0
    want = np.empty(c, f32)
    src = G.to_device(x)
    for reducer in (SUM, MAX) if n % 2 else (SUM, MIN):
        with np.errstate(all="ignore"):
            O.reduce_keep_highdim(want, x, reducer, SAVETO, 1.0)
        dst = G.buffer((c,), f32)
        G.reduce_keep_highdim(dst, src, reducer)
        got = dst.download()
        same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
        assert same.all(), (reducer, [(i, got[i], want[i]) for i in np.flatnonzero(~same)[:5]])
    # a tensor that begins in the middle of a pack, and a scale and savers of its own
    saver = PLUSTO if c % 2 else MINUSTO
    flat = rng.standard_normal(n * c * h * w + 1).astype(f32)
    whole = G.to_device(flat[None, :])
    start = rng.standard_normal(c).astype(f32)
    want = start.copy()
    O.reduce_keep_highdim(want, np.ascontiguousarray(flat[1:]).reshape(n, c, h, w), SUM, saver, 0.3)
    dst = G.to_device(start)
    G.check(G.dll.mshadow_hip_reduce_keep_highdim_f32(dst.ptr, whole.ptr + 4, w, n, c, h, w, SUM, saver, 0.3, None))
    assert np.array_equal(dst.download().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,c,h,w", SHAPES)
def test_half_planes_are_summed_in_order(G, O, n, c, h, w):
    rng = np.random.default_rng(n * 11 + c)
    x = O.float2half(rng.standard_normal((n, c, h, w)).astype(f32))
    want = np.empty(c, np.uint16)
    O.reduce_keep_highdim(want, x, SUM, SAVETO, 1.0)
    dst = G.buffer((c,), np.uint16)
    G.case_reduce_keep_highdim(dst, G.to_device(x), scale=0x3C00)
    assert np.array_equal(dst.download(), want)
