"""unpool of 2 x 2 and 3 x 3 windows by two at the edges of its packs and with pooled tensors of fewer windows than fit, and Softmax
of short rows that share cache lines: against the oracle, bit for bit (Softmax 1e-5, and the same whatever the alignment)."""
import numpy as np
import pytest

from checkers import MAX, MIN, SUM, Checker
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


# one plane whose last pack ends the tensor, odd and even widths from a pack on, heights that cut the last window, pitched rows
@pytest.mark.parametrize("planes,h,w,pad", [(1, 4, 4, 0), (1, 5, 5, 0), (1, 4, 7, 0), (3, 7, 6, 0), (2, 9, 9, 3), (5, 13, 13, 0), (64, 55, 55, 0),
                                            (7, 27, 27, 1), (3, 8, 66, 2), (2, 6, 255, 0), (3, 10, 16, 4), (1, 3, 4, 0)])
@pytest.mark.parametrize("k", [2, 3])
def test_unpool_by_two(G, O, planes, h, w, pad, k):
    rng = np.random.default_rng(h * 100 + w + k)
    x = rng.integers(-3, 4, (planes, h, w)).astype(f32)      # equal values in a window
    x[rng.random(x.shape) < 0.1] = -0.0
    ph, pw = (h - k) // 2 + 1, (w - k) // 2 + 1
    for reducer in (MAX, SUM, MIN):
        pooled = np.empty((planes, ph, pw), f32)
        O.pool(pooled, x, k, k, 2, 2, reducer)
        grad = rng.standard_normal(pooled.shape).astype(f32)
        want = np.empty_like(x)
        O.unpool(want, x, pooled, grad, k, k, 2, 2, reducer)
        dst = G.buffer(x.shape, f32, pad)
        G.unpool(dst, G.to_device(x, pad), G.to_device(pooled, pad), G.to_device(grad), k, k, 2, 2, reducer)
        assert np.array_equal(dst.download().view(np.uint32), want.view(np.uint32)), reducer


# pooled rows and columns left out at the end, several packs of them, with one column left and one or two windows in all; widths
# of whole packs and not; a gradient with a pitch of its own
@pytest.mark.parametrize("planes,h,w,ph,pw,pad,gpad", [(3, 8, 16, 3, 8, 0, 0), (3, 8, 16, 4, 6, 0, 1), (2, 9, 13, 2, 3, 1, 0), (2, 12, 12, 1, 6, 0, 3),
                                                       (5, 10, 10, 4, 1, 2, 2), (1, 8, 8, 1, 1, 0, 0), (2, 8, 8, 1, 1, 0, 0), (1, 8, 9, 2, 1, 0, 0),
                                                       (1, 8, 9, 1, 2, 0, 5), (64, 27, 27, 12, 11, 0, 0), (64, 28, 28, 12, 12, 0, 1)])
@pytest.mark.parametrize("k", [2, 3])
def test_unpool_by_two_of_fewer_windows(G, O, planes, h, w, ph, pw, pad, gpad, k):
    rng = np.random.default_rng(h * 1000 + w * 10 + k)
    x = rng.integers(-3, 4, (planes, h, w)).astype(f32)
    whole = np.empty((planes, (h - k) // 2 + 1, (w - k) // 2 + 1), f32)
    O.pool(whole, x, k, k, 2, 2, MAX)
    pooled = whole[:, :ph, :pw].copy()
    ph, pw = pooled.shape[1:]
    grad = rng.standard_normal(pooled.shape).astype(f32)
    want = np.empty_like(x)
    O.unpool(want, x, pooled, grad, k, k, 2, 2, MAX)
    dst = G.buffer(x.shape, f32, pad)
    G.unpool(dst, G.to_device(x, pad), G.to_device(pooled, gpad // 2), G.to_device(grad, gpad), k, k, 2, 2, MAX)
    assert np.array_equal(dst.download().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(8201, 33), (8200, 127), (16390, 129), (16391, 255), (8193, 64)])
def test_softmax_of_short_rows_at_any_alignment(G, O, rows, cols):
    x = (np.random.default_rng(cols).standard_normal((rows, cols)) * 3).astype(f32)
    want = np.empty_like(x)
    O.softmax(want, x)
    out = []
    for pad in (0, 1, 4 - cols % 4):
        dst = G.buffer(x.shape, f32, pad)
        G.softmax(dst, G.to_device(x, pad))
        out.append(dst.download())
    assert all(np.array_equal(o.view(np.uint32), out[0].view(np.uint32)) for o in out)
    assert (np.abs(out[0].astype(np.float64) - want) <= 1e-5 * want).all()
