"""Softmax on half_t rows kept on chip: every width of workgroup the dispatch takes, at its first and
last column and at rows that start at any column of an aligned pack, for rows of every kind the sum
in 16 bits can meet; its gradient on rows of any length and start. Bit-exact against the oracle."""
from types import SimpleNamespace

import numpy as np
import pytest

from checkers import Checker
from gpu_util import f32
from mshadow_amd.capi import DeviceBuffer

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


def part(buf, cols, shift):
    """the `cols` columns of a device buffer from column `shift` on"""
    return SimpleNamespace(ptr=buf.ptr + shift * buf.dtype.itemsize, stride=buf.stride, rows=buf.rows, cols=cols,
                           dtype=buf.dtype, shape=(buf.rows, cols))


def logits(kind, rows, cols):
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((rows, cols), dtype=f32) * f32({"flat": 0.1, "wide": 6.0}.get(kind, 3.0))
    if kind == "equal":
        x[:] = f32(-0.5)
    elif kind == "rising":
        x = np.sort(x, axis=1)
    elif kind == "ties":      # terms 1, 1/2, 3/8, ... of few bits: half-way cases all along
        x = np.log(rng.choice(np.array([1, 0.75, 0.5, 0.375, 0.0625], f32), (rows, cols))).astype(f32)
    elif kind == "late":      # nothing but zero terms in front of the largest
        x[:, : cols // 2] = -np.inf
    return x


def check(G, O, x, shift, dst_shift):
    rows, cols = x.shape
    x = O.float2half(x)
    want = np.empty_like(x)
    O.softmax(want, x)
    wide = np.full((rows, cols + 9), 0x3c00, np.uint16)
    wide[:, shift:shift + cols] = x
    src, dst = G.to_device(wide), G.to_device(np.full((rows, cols + 9), 0x1234, np.uint16))
    G.case_softmax(part(dst, cols, dst_shift), part(src, cols, shift))
    got = dst.download()
    inside = got[:, dst_shift:dst_shift + cols]
    nan = np.isnan(O.half2float(want))
    assert np.array_equal(np.isnan(O.half2float(inside)), nan)
    assert np.array_equal(inside[~nan], want[~nan]), f"{np.count_nonzero(inside != want)} of {want.size} differ"
    assert np.all(got[:, :dst_shift] == 0x1234) and np.all(got[:, dst_shift + cols:] == 0x1234), "written outside"
    G.case_softmax(part(src, cols, shift), part(src, cols, shift))  # in place
    assert np.array_equal(src.download()[:, shift:shift + cols], inside)


# 129: the shortest; runs of 512 columns in one, two, three, four waves of eight, three, four, eight and
# sixteen of sixteen; one column more than the longest goes to the kernel of other lengths
COLS = [129, 264, 505, 512, 1024, 1025, 2049, 4090, 4097, 8192, 8193, 12288, 12290, 16384, 16385, 24577, 32761, 32769,
        65529, 65537, 131065, 131066, 131072]


@pytest.mark.parametrize("cols", COLS)
def test_half_rows_widths(G, O, cols):
    rows = 2 if cols > 20000 else 5
    for shift, dst_shift in ((0, 0), (1, 1), (5, 2), (8, 0)):
        check(G, O, logits("normal", rows, cols), shift, dst_shift)


@pytest.mark.parametrize("cols", [1, 7, 8, 9, 12, 15, 17, 31, 63, 101, 127, 128, 132099])
def test_half_rows_that_end_inside_a_pack(G, O, cols):
    """rows of the kernel of other lengths, several to a workgroup; the longest ends just behind a tile"""
    rows = 2 if cols > 20000 else 37
    for shift, dst_shift in ((0, 0), (1, 1), (5, 2), (8, 3)):
        check(G, O, logits("normal", rows, cols), shift, dst_shift)


@pytest.mark.parametrize("kind", ["flat", "wide", "equal", "rising", "ties", "late"])
@pytest.mark.parametrize("cols", [300, 1500, 5000, 15000, 31000, 50257])
def test_half_rows_kinds(G, O, cols, kind):
    check(G, O, logits(kind, 3, cols), 0, 0)


def test_half_rows_special_values(G, O):
    """a NaN anywhere, an infinite maximum and rows of -infinity make every result of the row NaN"""
    x = logits("normal", 7, 3000)
    x[0, 0], x[1, 2999], x[2, 1234], x[3, 77], x[4, 5] = np.nan, np.nan, np.nan, np.inf, -np.inf
    x[5] = -np.inf
    check(G, O, x, 3, 3)


def test_half_rows_every_exponential(G, O):
    """x - max takes every binary16 value from -0 down to -infinity, and one wrong exponential shows in
    its quotient: a row that begins with 2^k columns of the maximum has a sum of 2^k, and terms of at
    most half an ulp of that, 2^(k-11), leave it there. Divided by 2^k a term of 2^(k-14) or more keeps
    all its bits; the smaller ones are in the row whose sum is one."""
    every = np.arange(0x8000, 0x7c01 + 0x8000, dtype=np.uint32).astype(np.uint16)
    d = O.half2float(every).astype(f32)
    with np.errstate(divide="ignore"):
        log2 = np.log2(np.exp(d.astype(np.float64)))
    row_of = np.clip(np.ceil(log2 + 11.5), 0, 11)
    x = np.full((12, 2048 + d.size), -np.inf, f32)
    quotients = np.zeros(x.shape, f32)
    for k in range(12):
        piece = d[row_of == k]
        x[k, :1 << k] = 0.0
        x[k, 1 << k:(1 << k) + piece.size] = piece
        quotients[k] = O.half2float(O.float2half(np.exp(x[k]))) * f32(2.0 ** -k)
    used = 2048 + int(max(np.count_nonzero(row_of == k) for k in range(12)))
    x, quotients = x[:, :used], quotients[:, :used]
    want = O.float2half(x)
    O.softmax(want, O.float2half(x))
    assert np.array_equal(O.half2float(want), quotients)   # nothing of a term is lost
    check(G, O, x, 0, 0)


def test_half_rows_more_than_a_launch_takes(G, O):
    """a wave per row of these is more threads than one launch may have (fewer than 2^32). In place; rows at
    both ends and in between are looked at, the others hold whatever the memory held."""
    rows, cols, some = (1 << 26) + 1024, 129, 100
    x = O.float2half(logits("normal", some, cols))
    want = np.empty_like(x)
    O.softmax(want, x)
    m = G.buffer((rows, cols), np.uint16)
    at = [SimpleNamespace(lib=G, ptr=m.ptr + r * cols * 2, stride=cols, rows=some, cols=cols, dtype=m.dtype, shape=x.shape)
          for r in (0, 1000, rows // 2 - 7, (1 << 26) - 50, rows - some)]
    for piece in at:
        DeviceBuffer.upload(piece, x)
    G.case_softmax(m, m)
    for piece in at:
        assert np.array_equal(DeviceBuffer.download(piece), want)


@pytest.mark.parametrize("rows,cols", [(300, 1), (300, 7), (300, 8), (513, 9), (129, 33), (65, 511), (33, 1000), (9, 1024),
                                       (9, 1025), (5, 2047), (3, 4097), (2, 50257)])
def test_half_gradient_rows(G, O, rows, cols):
    rng = np.random.default_rng(rows)
    prob = O.float2half(rng.random((rows, cols), dtype=f32))
    lab = rng.integers(-1, min(cols, 2048) + 1, rows).astype(f32)   # a few outside the row
    want = np.empty_like(prob)
    O.softmax_grad(want, prob, O.float2half(lab))
    for shift in (0, 1, 6):
        wide = np.zeros((rows, cols + 7), np.uint16)
        wide[:, shift:shift + cols] = prob
        src, dst = G.to_device(wide), G.to_device(np.full_like(wide, 0x1234))
        G.case_softmax_grad(part(dst, cols, 7 - shift), part(src, cols, shift), G.to_device(O.float2half(lab)))
        got = dst.download()
        assert np.array_equal(got[:, 7 - shift:7 - shift + cols], want)
        assert np.all(got[:, :7 - shift] == 0x1234) and np.all(got[:, 7 - shift + cols:] == 0x1234)


# both sides of the numbers of rows and columns at which the dispatch changes kernels
@pytest.mark.parametrize("rows,cols", [(64, 100), (65, 100), (64, 101), (65, 15), (65, 63), (6144, 11), (6145, 11), (6145, 7), (6144, 12),
                                       (3240, 129), (3241, 129), (6144, 256), (6145, 256), (6144, 257)])
def test_half_rows_routes(G, O, rows, cols):
    for shift, dst_shift in ((0, 0), (5, 2)):
        check(G, O, logits("normal", rows, cols), shift, dst_shift)


@pytest.mark.parametrize("rows,cols", [(3241, 248), (4352, 264), (4353, 264), (4353, 352), (4353, 360), (5376, 400), (5377, 400),
                                       (5377, 408), (8192, 376), (8193, 376)])
def test_half_rows_routes_of_whole_packs(G, O, rows, cols):
    x = O.float2half(logits("normal", rows, cols))
    want = np.empty_like(x)
    O.softmax(want, x)
    src = G.to_device(x)
    G.case_softmax(src, src)
    assert np.array_equal(src.download(), want)


@pytest.mark.parametrize("rows,cols", [(1536, 21), (1537, 20), (1537, 21), (1537, 96), (1537, 511), (1537, 1024)])
def test_half_gradient_routes(G, O, rows, cols):
    test_half_gradient_rows(G, O, rows, cols)
