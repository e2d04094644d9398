"""Softmax of rows that are kept partly in LDS (32769 to 51200 columns with more rows than compute units, 65537 to 110592
columns), of the wider workgroups that up to two rows a compute unit take, and of the other rows of 1025 to 8192 columns, a
workgroup or a wave each: bit for bit what the kernel that goes
stretch by stretch gives for the same logits with columns of -inf behind them, whose terms are zeros at the end of the sum
and which change neither the maximum nor a quotient. That kernel's row sums are tested against the serial sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32
STRETCHED = 131072 + 7


@pytest.fixture(scope="module")
def G():
    import mshadow_amd
    g = mshadow_amd.load_cases()
    assert g.device_count() >= 1, "no GPU visible"
    g.set_device(0)
    return g


@pytest.fixture(scope="module")
def stream(G):
    s = G.stream_create()
    yield s
    G.stream_destroy(s)


def _logits(rows, cols, seed):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((rows, cols)) * 3).astype(f32)
    x[1 % rows] = np.log(rng.uniform(1e-6, 1, cols))                      # sums through many binades, evenly
    x[2 % rows] = 0.0                                                     # 1 + 1 + ...: every sum a whole number
    x[3 % rows, : cols - 1] = -40.0                                       # one term above next to nothing, at the end
    x[3 % rows, cols - 1] = 0.0
    # sums that pass 2 at once and then stay a little above it: more addends than the row's list holds
    x[4 % rows] = np.log(1e-5 / cols)
    x[4 % rows, :2] = 0.0
    x[5 % rows, cols // 2] = np.inf
    x[6 % rows, cols // 3] = np.nan
    x[7 % rows, ::3] = -np.inf
    return x


# around the first column in LDS, the ends of a slab, whole and ragged packs, the last column that fits
SHAPES = [(280, 32769, 0), (280, 36864, 0), (270, 36867, 1), (260, 50257, 0), (300, 51199, 2), (300, 51200, 0),
          (9, 65537, 0), (9, 65540, 3), (260, 70001, 0), (9, 81917, 0), (9, 81920, 0), (9, 81921, 1), (9, 94209, 0), (520, 90001, 0),
          (9, 110589, 0), (9, 110592, 0),
          # wider workgroups for few rows
          (9, 1025, 0), (9, 2047, 1), (9, 2048, 0), (500, 3001, 0), (9, 4096, 0), (9, 8191, 2), (9, 16384, 0), (9, 16385, 0), (9, 32767, 0),
          # a workgroup a row beyond those few rows, at its borders with the kernel of a wave a row
          (1535, 1025, 0), (1200, 2047, 1), (600, 2048, 0), (1023, 2049, 2), (1023, 3072, 0), (1100, 3073, 0), (513, 4096, 1),
          (600, 4097, 0), (513, 8191, 0), (513, 8192, 3),
          # a wave a row, up to 4, 8, 10 and 12 packs a lane
          (1536, 1024, 0), (1536, 1025, 0), (1537, 2047, 1), (1600, 2048, 0), (1024, 2049, 0), (1025, 2303, 2), (1101, 2560, 0),
          (1024, 2561, 3), (1026, 2815, 0), (1024, 3072, 0)]


@pytest.mark.parametrize("rows,cols,pad", SHAPES)
def test_rows_in_lds_are_the_stretched_rows(G, stream, rows, cols, pad):
    few = 9
    x = np.tile(_logits(few, cols, cols), ((rows + few - 1) // few, 1))[:rows]
    long = np.full((few, STRETCHED), -np.inf, f32)
    long[:, :cols] = x[:few]
    want = G.buffer(long.shape, f32)
    G.softmax(want, G.to_device(long), stream)
    want = want.download(stream)[:, :cols]
    src = G.to_device(x, pad)
    dst = G.buffer(x.shape, f32, pad)
    G.softmax(dst, src, stream)
    got = dst.download(stream)
    for r in range(rows):
        w = want[r % few]
        same = (got[r].view(np.uint32) == w.view(np.uint32)) | (np.isnan(got[r]) & np.isnan(w))
        assert same.all(), (r, np.flatnonzero(~same)[:5])
    G.softmax(src, src, stream)   # in place
    assert np.array_equal(src.download(stream).view(np.uint32), got.view(np.uint32))
