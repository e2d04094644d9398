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
    x = np.log(np.maximum(terms, 1e-30)).astype(f32)   # the softmax of the same rows sums to 1
    p = G.buffer(x.shape, f32)
    G.softmax(p, G.to_device(x))
    got = p.download().astype(np.float64).sum(1)
    assert np.all(np.abs(got - 1) < cols * 2.0 ** -24)   # a sum's cols roundings of at most half an ulp
