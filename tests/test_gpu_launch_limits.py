"""Matrices of so many rows that a thread, a wave or a workgroup for each would be 2^32 threads or more,
which one launch cannot have: every row is worked on all the same. Up to 69 GB, in place where that is
possible; rows at both ends, on both sides of the limit and in between are compared with the oracle, the
others hold whatever the memory held."""
from types import SimpleNamespace

import numpy as np
import pytest

from checkers import Checker
from gpu_util import assert_bits_equal, f32
from mshadow_amd.capi import DeviceBuffer, HipError

pytestmark = pytest.mark.gpu
SOME = 40


@pytest.fixture(scope="module")
def G():
    import mshadow_amd
    g = mshadow_amd.load_cases()
    g.set_device(0)
    return g


@pytest.fixture(scope="module")
def O():
    return Checker("orc")


def pieces(G, m, limit):
    """SOME rows of m here and there, as buffers of their own"""
    starts = sorted({0, 1000, m.rows // 2 - 7, limit - SOME // 2, m.rows - SOME})
    return [SimpleNamespace(lib=G, ptr=m.ptr + r * m.cols * m.dtype.itemsize, stride=m.cols, rows=SOME, cols=m.cols,
                            dtype=m.dtype, shape=(SOME, m.cols)) for r in starts]


def logits(O, cols, dtype):
    x = (np.random.default_rng(cols).standard_normal((SOME, cols), dtype=f32) * f32(3)).astype(f32)
    return O.float2half(x) if dtype == np.uint16 else x


@pytest.mark.parametrize("limit,cols", [(1 << 27, 3)])
def test_half_softmax(G, O, limit, cols):
    x = logits(O, cols, np.uint16)
    want = np.empty_like(x)
    O.softmax(want, x)
    m = G.buffer((limit + 64, cols), np.uint16)
    at = pieces(G, m, limit)
    for p in at:
        DeviceBuffer.upload(p, x)
    G.case_softmax(m, m)
    for p in at:
        assert_bits_equal(DeviceBuffer.download(p), want)


@pytest.mark.parametrize("limit,cols", [(1 << 28, 33), (1 << 26, 257)])
def test_softmax_and_row_sums(G, O, limit, cols):
    x = logits(O, cols, f32)
    want = np.empty_like(x)
    O.softmax(want, x)
    m = G.buffer((limit + 64, cols), f32)
    at = pieces(G, m, limit)
    for p in at:
        DeviceBuffer.upload(p, np.abs(x))
    sums = G.buffer((m.rows, 1), f32)
    G.softmax_rowsum(sums, m)
    right = np.cumsum(np.abs(x), axis=1, dtype=f32)[:, -1:]
    for p in pieces(G, sums, limit):
        assert_bits_equal(DeviceBuffer.download(p), right)
    for p in at:
        DeviceBuffer.upload(p, x)
    G.softmax(m, m)
    for p in at:   # the bound of the short rows' test: exponential, sum and quotient
        assert np.max(np.abs(DeviceBuffer.download(p).astype(np.float64) - want) / want) < 1e-6


@pytest.mark.parametrize("dtype,cols", [(np.uint16, 1025), (np.float32, 513)])
def test_softmax_gradient(G, O, dtype, cols):
    limit = 1 << 24
    prob = logits(O, cols, dtype)
    label = np.arange(SOME) % cols
    label = O.float2half(label.astype(f32)) if dtype == np.uint16 else label.astype(f32)
    want = np.empty_like(prob)
    O.softmax_grad(want, prob, label)
    m, labels = G.buffer((limit + 64, cols), dtype), G.buffer((limit + 64, 1), dtype, fill=0)
    at = pieces(G, m, limit)
    for p, l in zip(at, pieces(G, labels, limit)):
        DeviceBuffer.upload(p, prob)
        DeviceBuffer.upload(l, label.reshape(-1, 1))
    (G.case_softmax_grad if dtype == np.uint16 else G.softmax_grad)(m, m, labels)
    for p in at:
        assert_bits_equal(DeviceBuffer.download(p), want)


def test_columns_of_two_rows(G):
    """where no call takes less than 2^32 threads the launch is refused, not cut short"""
    m, dst = G.buffer((2, 870_000_000), f32), G.buffer((870_000_000,), f32)
    with pytest.raises(HipError, match="2\\^32"):
        G.reduce_keep_lowest(dst, m)


@pytest.mark.parametrize("n", [1, 3])
def test_kept_indices(G, O, n):
    limit, cols = 1 << 24, 3
    x = logits(O, cols, f32)
    m = G.buffer((n, limit + 64, 1, cols), f32, fill=0)
    rows = SimpleNamespace(ptr=m.ptr, rows=limit + 64, cols=cols, dtype=m.dtype)
    for p in pieces(G, rows, limit):
        DeviceBuffer.upload(p, x)
    dst = G.buffer((limit + 64, 1), f32)
    G.reduce_keep_highdim(dst, m)
    for p in pieces(G, dst, limit):
        assert_bits_equal(DeviceBuffer.download(p), np.cumsum(x, axis=1, dtype=f32)[:, -1:])
