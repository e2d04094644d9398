"""sum_rows at the edges of its strips of columns: every width of strip the dispatch takes (by the
number of columns), rows around a block, a slot and a full ring, and rows that start at any element.
Bit-exact against the oracle, like every reduction: the order of the additions is the CPU path's."""
from types import SimpleNamespace

import numpy as np
import pytest

from checkers import MAX, PLUSTO, SAVETO, SUM, Checker
from gpu_util import assert_bits_equal, f32, normal, uniform

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


# strips of 16, 32 and 64 columns (up to 4096 and 8192 columns and beyond), the last one not full,
# and the short ring (up to 1024 rows, more than 32768 columns); 6144 rows and more of up to 4096 float
# columns, 4000 of up to 64 and 2400 of one take the kernel of long chains, whose stages have 512 rows
SHAPES = [(1, 16), (15, 17), (16, 1), (64, 15), (65, 4096), (129, 4097), (257, 33), (2047, 40), (2048, 4097),
          (63, 8192), (64, 8193), (320, 8255), (513, 9000), (1024, 32769), (1025, 32775), (32, 32800), (97, 33000),
          (2399, 1), (2400, 1), (3999, 10), (4000, 64), (4001, 65), (6143, 65), (6144, 70), (6145, 1),
          (6657, 33), (8191, 1000), (6150, 4095)]


def offset_view(buf, cols, shift):
    """the `cols` columns of a device buffer from column `shift` on"""
    return SimpleNamespace(ptr=buf.ptr + shift * buf.dtype.itemsize, stride=buf.stride, rows=buf.rows, cols=cols,
                           dtype=buf.dtype, shape=(buf.rows, cols))


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("half", [False, True])
def test_sum_rows_strips(G, O, rows, cols, half):
    for extra, shift in ((0, 0), (1, 1), (2, 1), (3, 0), (4, 2)):
        wide = normal(70 + extra, (rows, cols + extra))
        start = uniform(71, (cols,)) + f32(2)
        scale = 0.75
        if half:
            wide, start = O.float2half(wide), O.float2half(start)
            scale = int(O.float2half(np.array([scale], f32))[0])
        m = np.ascontiguousarray(wide[:, shift:shift + cols])
        src = G.to_device(wide)
        for reducer, saver in ((SUM, SAVETO), (SUM, PLUSTO), (MAX, SAVETO)):
            want, dst = start.copy(), G.to_device(start)
            O.reduce_keep_lowest(want, m, reducer, saver, 0.75)
            if half:
                G.case_reduce_keep_lowest(dst, offset_view(src, cols, shift), reducer, saver, scale)
            else:
                G.reduce_keep_lowest(dst, offset_view(src, cols, shift), reducer, saver, scale)
            assert_bits_equal(dst.download(), want, f"{rows}x{cols} half={half} pitch+{extra} start+{shift}")


# long chains in strips of 16 that the kernel of other sources sums: both sides of the rows and strips from which the
# strips are dealt in eighths
@pytest.mark.parametrize("rows,cols", [(16383, 17), (16384, 17), (16384, 128), (16390, 1785), (16384, 1793)])
def test_half_sum_rows_long_chains(G, O, rows, cols):
    m = O.float2half(uniform(77, (rows, cols)))
    want = np.zeros(cols, np.uint16)
    dst = G.to_device(want)
    O.reduce_keep_lowest(want, m, SUM, SAVETO, 0.75)
    G.case_reduce_keep_lowest(dst, G.to_device(m), SUM, SAVETO, int(O.float2half(np.array([0.75], f32))[0]))
    assert_bits_equal(dst.download(), want, f"{rows}x{cols}")
