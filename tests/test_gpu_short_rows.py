"""The left-to-right row sums and the Softmax of short float rows at the edges of the dispatch: a thread,
a part of a wave, a wave per row, by columns and by the number of rows. Sums are bit-exact against a
serial float32 sum, whatever the terms are."""
import numpy as np
import pytest

from checkers import Checker
from gpu_util import assert_bits_equal, f32

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


def terms(kind, rows, cols):
    rng = np.random.default_rng(cols)
    x = np.exp(rng.standard_normal((rows, cols), dtype=f32) * f32(3) - f32(6))
    if kind == "ties":       # few bits and a wide range: half-way cases
        x = np.ldexp(f32(1), rng.integers(-30, 3, (rows, cols))).astype(f32)
    elif kind == "signed":
        x *= rng.choice(np.array([-1, 1], f32), (rows, cols))
    elif kind == "extremes":  # subnormal, zero and huge terms; infinities and NaN in some rows
        with np.errstate(over="ignore"):
            x *= np.ldexp(f32(1), rng.integers(-140, 120, (rows, cols))).astype(f32)
        x[::3, cols // 2] = 0.0
        x[1::7, cols // 3] = np.inf
        x[2::11, cols - 1] = np.nan
    return x


# rows around 16, 64 and 6 times the 256 CUs; columns around every kernel's own
@pytest.mark.parametrize("cols", [1, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 3072, 3073])
@pytest.mark.parametrize("kind", ["normal", "ties", "signed", "extremes"])
def test_row_sums(G, cols, kind):
    for rows in ((7, 1537) if cols > 512 else (7, 4099) if cols <= 128 else (7, 16387)):
        x = terms(kind, rows, cols)
        with np.errstate(all="ignore"):
            want = np.cumsum(x, axis=1, dtype=f32)[:, -1]
        sums = G.buffer((rows,), f32)
        G.softmax_rowsum(sums, G.to_device(x))
        got = sums.download()
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert_bits_equal(got[~nan], want[~nan], f"{kind} {rows}x{cols}")


@pytest.mark.parametrize("rows", [1, 255, 257, 5000])
def test_row_sums_of_no_terms(G, rows):
    """rows without a column sum to zero, and no term is read: there may be no tensor at all"""
    x = G.to_device(np.full((rows, 4), 3.0, f32))
    for terms_ptr, pitch in ((x.ptr, 4), (x.ptr, 0), (None, 0)):
        sums = G.to_device(np.full(rows, 7.0, f32))
        G.check(G.dll.mshadow_hip_softmax_rowsum_f32(sums.ptr, terms_ptr, pitch, rows, 0, None))
        assert_bits_equal(sums.download(), np.zeros(rows, f32), f"{rows} rows, pitch {pitch}")


@pytest.mark.parametrize("rows,cols", [(7, 10), (5000, 16), (9, 50), (4096, 64), (4097, 64), (33, 128), (5000, 101), (70, 200),
                                       (16385, 200), (3, 512), (1535, 513), (1536, 700), (2000, 2304), (2000, 3072)])
def test_softmax_short_rows(G, O, rows, cols):
    x = (np.random.default_rng(rows).standard_normal((rows, cols), dtype=f32) * f32(3)).astype(f32)
    want = np.empty_like(x)
    O.softmax(want, x)
    dst = G.buffer(x.shape, f32)
    G.softmax(dst, G.to_device(x))
    got = dst.download().astype(np.float64)
    # the exponential within 3 ulp, the sum of such terms and the quotient within one each: 4e-7 together
    assert np.max(np.abs(got - want) / want) < 1e-6


@pytest.mark.parametrize("cols", [1, 8, 9, 12, 13, 16, 17, 20, 21, 24, 25, 28, 29, 32])
def test_rows_of_a_thread(G, O, cols):
    """at the lengths that a thread's registers are cut to: Softmax, in place and not, and the row sums, pitched and ending
    where the tensor ends"""
    rows = 515
    x = (np.random.default_rng(cols).standard_normal((rows, cols), dtype=f32) * f32(3)).astype(f32)
    x[::7, -1] = x[::7].max(axis=1) + f32(1)
    want = np.empty_like(x)
    O.softmax(want, x)
    terms = np.exp(x)
    sums = np.zeros(rows, f32)
    for i in range(cols):
        sums = sums + terms[:, i]
    for pad in (0, 3):
        src = G.to_device(x, pad)
        dst = G.buffer(x.shape, f32, pad)
        G.softmax(dst, src)
        got = dst.download()
        assert np.max(np.abs(got.astype(np.float64) - want) / want) < 1e-6   # as above
        G.softmax(src, src)
        assert_bits_equal(src.download(), got, f"{cols} columns in place")
        out = G.buffer((rows,), f32)
        t = G.to_device(terms, pad)
        G.check(G.dll.mshadow_hip_softmax_rowsum_f32(out.ptr, t.ptr, cols + pad, rows, cols, None))
        assert_bits_equal(out.download(), sums, f"{cols} columns")
