"""sum_rows of long float columns, which are summed by chunks of 128 rows: maps from the sum in front of a chunk to
the sum behind it, looked up one after the other, or the chunk's terms where there is no map. Bit-exact against the
oracle's serial sum on both sides of the dispatch's border and of tiles, chunks, workgroups and blocks of the walk,
and on columns that take each of the ways a chunk can go."""
import threading
import time
from types import SimpleNamespace

import numpy as np
import pytest

from checkers import MINUSTO, PLUSTO, SAVETO, SUM, Checker
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


def terms(kind, rows, cols, seed):
    rng = np.random.default_rng(seed)
    m = rng.standard_normal((rows, cols), dtype=f32)
    if kind == "gradient":
        p = np.exp(m * 3)
        m = (p / np.maximum(p.sum(1, keepdims=True), f32(90 * 8))).astype(f32)
        m[np.arange(rows), rng.integers(0, max(cols, 8), rows) % cols] -= (rng.random(rows) < 0.3).astype(f32)
    elif kind == "constant":      # every rounding goes the same way: the sums drift away from the expected ones
        m[:] = f32(0.1) * (1 + np.arange(cols, dtype=f32))
    elif kind == "alternating":
        m = np.abs(m) * np.where(np.arange(rows) % 2, f32(-1), f32(1))[:, None]
    elif kind == "cancelling":    # sums of exactly nothing or one term: no map either
        m[:] = np.where(np.arange(rows) % 2, f32(-1), f32(1))[:, None] * (1 + np.arange(cols, dtype=f32) / 8)
    elif kind == "late":          # such rows from another chunk on in every column
        start = rows // 3 + 97 * (np.arange(cols) % 23)
        back = np.where(np.arange(rows) % 2, f32(-1e6), f32(1e6))[:, None] * (1 + np.arange(cols, dtype=f32))
        m = np.where(np.arange(rows)[:, None] >= start, back, m).astype(f32)
    elif kind == "few":           # such columns among others that have maps
        m[:, 5::23] = np.where(np.arange(rows) % 2, f32(-3), f32(3))[:, None]
    elif kind == "overflow":
        m = (np.abs(m) * f32(3e34)).astype(f32)
    elif kind == "zeros":         # nothing to add, of either sign, with a few terms between
        m[:] = np.where(rng.random((1, cols)) < 0.5, f32(-0.0), f32(0.0))
        m[rows // 3] = rng.integers(-1, 2, cols)
        m[rows // 2, ::3] = f32(0.0)
    elif kind == "ties":
        m = np.round(m * 64).astype(f32) / 64 + f32(2.0 ** -18)
    elif kind == "wide":
        m = (m * np.exp2(rng.integers(-40, 40, m.shape))).astype(f32)
    elif kind == "tiny":
        m = (m * f32(1e-38)).astype(f32)
    elif kind == "infinite":
        m[rng.integers(0, rows, cols), np.arange(cols)] = np.where(np.arange(cols) % 3 == 0, -np.inf, np.inf)
        m[rows - 1, ::4] = np.nan
    return np.ascontiguousarray(m)


# with 10 columns from 6335 rows on, with 64 from 6545, with 1000 from 15455 (tests/host/column_chunk_plan_check.cc looks these up);
# chunks of 128 rows, workgroups of four chunks and 64 columns, blocks of 16 chunks; up to two columns a compute unit (512) the walk
# takes a block's maps at once, beyond that four; bands of 8192 chunks of up to 64 columns, 512 of up to 1024
SHAPES = [(6300, 10), (6400, 10), (6528, 64), (6656, 64), (6657, 65), (6783, 63), (8192, 1), (8193, 3), (8320, 129), (10240, 128),
          (9200, 512), (9200, 513), (16384, 1000), (20481, 17), (33000, 300), (65536, 1000), (65537, 1000), (1048576, 3),
          (1048577, 3), (2097281, 5)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_long_columns(G, O, rows, cols):
    for kind, extra, shift in (("normal", 0, 0), ("gradient", 3, 1)):
        wide = terms(kind, rows, cols + extra, 7)
        m = np.ascontiguousarray(wide[:, shift:shift + cols])
        src = G.to_device(wide)
        view = SimpleNamespace(ptr=src.ptr + shift * 4, stride=src.stride, rows=rows, cols=cols, dtype=src.dtype,
                               shape=(rows, cols))
        start = np.random.default_rng(8).standard_normal(cols, dtype=f32)
        for saver in (SAVETO, PLUSTO, MINUSTO) if rows * cols < 1 << 24 else (PLUSTO,):
            want, dst = start.copy(), G.to_device(start)
            O.reduce_keep_lowest(want, m, SUM, saver, 0.75)
            G.reduce_keep_lowest(dst, view, SUM, saver, 0.75)
            assert_bits_equal(dst.download(), want, f"{rows}x{cols} {kind} saver {saver}")


@pytest.mark.parametrize("rows,cols", [(12345, 70), (9300, 300), (16411, 999)])
@pytest.mark.parametrize("kind", ["constant", "alternating", "cancelling", "late", "few", "overflow", "zeros", "ties", "wide",
                                  "tiny", "infinite"])
def test_columns_whose_chunks_have_no_map(G, O, kind, rows, cols):
    m = terms(kind, rows, cols, 11)
    src = G.to_device(m)
    for saver in (SAVETO, PLUSTO):   # the second with the scratch memory as the first call left it
        want, dst = np.full(cols, 7, f32), G.to_device(np.full(cols, 7, f32))
        with np.errstate(all="ignore"):
            O.reduce_keep_lowest(want, m, SUM, saver, 0.75)
        G.reduce_keep_lowest(dst, src, SUM, saver, 0.75)
        got = dst.download()
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert_bits_equal(got[~nan], want[~nan], kind)


@pytest.mark.parametrize("kind", ["constant", "infinite"])
def test_time_without_usable_maps(G, kind):
    """Columns whose roundings all go one way, or that meet an infinity or a NaN, are no slower than others: 50 and 57 us where
    drawn terms take 54, and 148 and 263 when their terms were read from the matrix column by column. The bound is twice
    the time of drawn terms, of 40 calls each, the least of six."""
    rows, cols = 16384, 1000

    def least(m):
        src, dst = G.to_device(m), G.buffer((cols,), f32)
        times = []
        for _ in range(6):
            G.device_sync()
            t0 = time.perf_counter()
            for _ in range(40):
                G.reduce_keep_lowest(dst, src)
            G.device_sync()
            times.append(time.perf_counter() - t0)
        return min(times)

    assert least(terms(kind, rows, cols, 3)) < 2 * least(terms("normal", rows, cols, 3))


@pytest.mark.parametrize("kind", ["constant", "cancelling", "late", "few", "infinite"])
def test_bands_of_columns_without_maps(G, O, kind):
    """a column that is chained in one band and walked in the next, or was left infinite or NaN by the one before"""
    rows, cols = 66001, 1000   # two bands of 260 chunks and less
    m = terms("normal", rows, cols, 5)
    m[rows // 4:3 * rows // 4] = terms(kind, 3 * rows // 4 - rows // 4, cols, 6)
    want, dst = np.full(cols, 7, f32), G.to_device(np.full(cols, 7, f32))
    with np.errstate(all="ignore"):
        O.reduce_keep_lowest(want, m, SUM, PLUSTO, 0.75)
    G.reduce_keep_lowest(dst, G.to_device(m), SUM, PLUSTO, 0.75)
    got = dst.download()
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert_bits_equal(got[~nan], want[~nan], kind)


def test_streams_threads_and_recording(G, O):
    """streams have scratch memory of their own, more of them than there is such memory for among them; threads that
    share a stream do not come between each other's launches; a recorded call does without"""
    mats = [terms("normal", 7000 + 300 * i, 40, 20 + i) for i in range(6)]
    want = []
    for m in mats:
        w = np.empty(40, f32)
        O.reduce_keep_lowest(w, m)
        want.append(w)
    src = [G.to_device(m) for m in mats]
    out = [G.buffer((40,), f32) for _ in mats]
    streams = [G.stream_create() for _ in mats]
    for _ in range(3):
        for i, s in enumerate(streams):
            G.reduce_keep_lowest(out[i], src[i], stream=s)
    for i, s in enumerate(streams):
        G.stream_sync(s)
        assert_bits_equal(out[i].download(), want[i], f"stream {i}")

    def work(i):
        G.set_device(0)
        for _ in range(20):
            G.reduce_keep_lowest(out[i], src[i], stream=streams[0])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    G.stream_sync(streams[0])
    for i in range(4):
        assert_bits_equal(out[i].download(), want[i], f"thread {i}")

    # a slot of its own in the recording stream, which sums others' columns while its recording is replayed beside it
    G.graph_begin(streams[1])
    G.reduce_keep_lowest(out[2], src[2], stream=streams[1])
    G.reduce_keep_lowest(out[4], src[4], stream=streams[0])   # not recorded, while the same thread records
    graph = G.graph_end(streams[1])
    G.stream_sync(streams[0])
    assert_bits_equal(out[4].download(), want[4], "beside a recording")
    for _ in range(5):
        G.fill(out[2], 3.0, streams[2])
        for i in range(6):
            G.graph_launch(graph, streams[2])
            G.reduce_keep_lowest(out[3], src[3], stream=streams[1])
        G.stream_sync(streams[1])
        G.stream_sync(streams[2])
        assert_bits_equal(out[2].download(), want[2], "replayed")
        assert_bits_equal(out[3].download(), want[3], "beside a replay")
    G.graph_destroy(graph)
    for s in streams:
        G.stream_destroy(s)


def test_slots_of_streams_that_go_away(G, O):
    """a stream destroyed with sums queued gives its scratch memory to the next one only when they are done"""
    rows, cols = 20000, 200
    mats = [terms(k, rows, cols, 30 + i) for i, k in enumerate(("normal", "gradient"))]
    want = []
    for m in mats:
        w = np.empty(cols, f32)
        O.reduce_keep_lowest(w, m)
        want.append(w)
    src = [G.to_device(m) for m in mats]
    out = [G.buffer((cols,), f32) for _ in mats]
    for _ in range(6):   # more of them than slots
        a, b = G.stream_create(), G.stream_create()
        for _ in range(8):
            G.reduce_keep_lowest(out[0], src[0], stream=a)
        G.stream_destroy(a)
        c = G.stream_create()
        G.reduce_keep_lowest(out[1], src[1], stream=c)
        G.reduce_keep_lowest(out[0], src[0], stream=b)
        G.device_sync()
        for i in range(2):
            assert_bits_equal(out[i].download(), want[i], f"stream {i}")
        G.stream_destroy(b)
        G.stream_destroy(c)
