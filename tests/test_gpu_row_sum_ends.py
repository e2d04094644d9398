"""Row sums that end just above a power of two in rows that do not fill their kernel's slabs: the chunks behind the end,
zeros whose binade is not certain there, enter no list of addends. Bit for bit the serial sum."""
import numpy as np
import pytest

from gpu_util import assert_bits_equal

pytestmark = pytest.mark.gpu
f32 = np.float32


# little and much of the slabs unused: a slab and a chunk, one column, all but one column
@pytest.mark.parametrize("cols", [3073, 5000, 8191, 8193, 10000, 16385, 16808, 30001, 32769, 40000, 65281, 70001, 100003])
def test_row_sums_that_end_above_a_power_of_two(cols):
    import mshadow_amd
    G = mshadow_amd.load_cases()
    G.set_device(0)
    rng = np.random.default_rng(cols)
    rows = []
    for above in (0.0, 1e-6, 1e-5, 1e-4, 3e-4, 1e-3, 5e-3):
        t = np.exp((rng.standard_normal(cols) - 4) * 3)
        t = np.minimum(t, 1)
        rows.append(t * (2.0 ** np.floor(np.log2(t.sum())) * (1 + above) / t.sum()))
        rows.append(np.where(np.arange(cols) < cols // 3, rows[-1], 0) * 4)   # zeros within the row
    terms = np.array(rows, f32)
    want = np.array([np.add.accumulate(r, dtype=f32)[-1] for r in terms])
    sums = G.buffer((len(terms),), f32)
    G.softmax_rowsum(sums, G.to_device(terms))
    assert_bits_equal(sums.download(), want, f"{cols} columns")
    # Softmax of rows whose largest term is a power of two, so that its terms, divided by that, end there too. The probability of
    # that term is 1 / sum. Against the same serial sum of numpy's exponentials, which differ from the device's by few ulps: two sums
    # with roundings of their own, uniform in half an ulp (2^-24 of the sum) to either side, so 2^-24 sqrt(cols / 3) off the exact one
    # each; six times what both are off together, and 8 ulps for the exponentials and the quotient.
    rest = terms[:, 1:].astype(np.float64)
    total = terms.astype(np.float64).sum(1)
    largest = 2.0 ** np.ceil(np.log2(rest.max(1)))
    rest *= ((total - largest) / rest.sum(1))[:, None]
    largest = np.where(rest.max(1) > largest, 2 * largest, largest)
    x = np.log(np.maximum(np.column_stack([largest, rest]) / largest[:, None], 1e-30)).astype(f32)
    assert np.all(x.max(1) == 0) and np.all(x[:, 0] == 0)
    want = np.array([np.add.accumulate(np.exp(r), dtype=f32)[-1] for r in x]).astype(np.float64)
    p = G.buffer(x.shape, f32)
    G.softmax(p, G.to_device(x))
    got = p.download().astype(np.float64)
    bound = 6 * np.sqrt(2 * cols / 3) * 2.0 ** -24 + 8 * 2.0 ** -24
    assert np.all(np.abs(got[:, 0] * want - 1) < bound), np.abs(got[:, 0] * want - 1).max() / bound
    ratio = got * want[:, None] / np.exp(x.astype(np.float64))
    normal = got > 2.0 ** -120   # not where quotients round to subnormals
    assert np.all(np.abs(ratio[normal] - 1) < bound)
