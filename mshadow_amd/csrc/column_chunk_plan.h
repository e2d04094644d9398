/*
 * Which column sums go by chunks of 128 rows (column_chunk_kernels.h), and in which bands of rows: plain C++, so that a
 * host program can look at the choice without a GPU.
 */
#ifndef MSHADOW_AMD_CSRC_COLUMN_CHUNK_PLAN_H_
#define MSHADOW_AMD_CSRC_COLUMN_CHUNK_PLAN_H_

#include <stdint.h>

#include "column_chunks.h"

namespace mshadow_hipk {

/*! \brief a workgroup has four chunks of 64 columns, a wave each */
const int kChunkWaves = 4;
const uint32_t kColumnsPerTile = 64;
/*! \brief columns of a strip that is chained */
const uint32_t kChunkStrip = 16;

/*! \brief what the scratch memory of a call has room for: cells are (chunk, column), the columns padded to whole tiles */
const uint32_t kChunkCells = 1u << 19;
const uint32_t kChunkCopies = 1u << 14;
const uint32_t kChunkGroupCells = kChunkCells / kChunkWaves * 3 / 2;  // groups of fewer than four chunks among them
const uint32_t kMostChunkColumns = 1536;

/*! \brief a band of rows, and the columns */
struct ChunkShape {
  uint32_t rows, cols, stride;
  uint32_t chunks, groups, tiles;
  uint32_t copies;     // copies a (chunk, tile) has room for
  uint32_t strips;     // strips of 16 columns that may be chained, 0: none
  uint32_t most_bare;  // bare chunks of a column that is walked
  uint32_t begun, more;  // whether rows in front of and behind the band are other bands'
};

/*! \brief rows of the bands that a matrix is summed in, but for the last, which may have fewer: of about the same size, whole
 *  workgroups of chunks, so many that the scratch memory holds a band's cells */
inline uint32_t ChunkBandRows(uint32_t rows, uint32_t cols) {
  const uint64_t group_rows = static_cast<uint64_t>(kChunkWaves) * column_chunks::kRows;
  const uint32_t tiles = (cols + kColumnsPerTile - 1) / kColumnsPerTile;
  const uint64_t most = kChunkCells / (tiles * kColumnsPerTile) / kChunkWaves * group_rows;
  const uint64_t bands = (rows + most - 1) / most;
  return static_cast<uint32_t>(((rows + bands - 1) / bands + group_rows - 1) / group_rows * group_rows);
}
inline ChunkShape MakeChunkShape(uint32_t rows, uint32_t cols, uint32_t stride, uint32_t cus) {
  ChunkShape g;
  g.rows = rows;
  g.cols = cols;
  g.stride = stride;
  g.chunks = (rows + column_chunks::kRows - 1) / column_chunks::kRows;
  g.groups = (g.chunks + kChunkWaves - 1) / kChunkWaves;
  g.tiles = (cols + kColumnsPerTile - 1) / kColumnsPerTile;
  const uint32_t room = kChunkCopies / (g.chunks * g.tiles);
  g.copies = room < kColumnsPerTile ? room : kColumnsPerTile;
  /* A bare chunk's terms, read from the matrix 4 bytes of a cache line at a time, take 0.5 us where a column has a CU to itself,
     1.2 us where all of 512 columns have such chunks, 2.3 us of 1000 (65536 x 1000: 1180 us in all). In a strip of 16 columns
     128 terms of each take 0.53 us. */
  g.strips = cols <= cus ? 0u : (cols + kChunkStrip - 1) / kChunkStrip;
  g.most_bare = static_cast<uint32_t>(static_cast<uint64_t>(g.chunks) * cus / cols) + 8u;
  g.begun = g.more = 0u;
  return g;
}

/*! \brief where the chunks are the sooner way. Measured, us (MI355X; a classifier's gradients), without and with:
 *  131072 x 10 448 and 99, 131072 x 100 470 and 109, 65536 x 1000 232 and 169, 30000 x 100 114 and 44, 16384 x 1000
 *  64 and 53, 16384 x 100 65 and 30, 8192 x 100 36 and 23, 8192 x 10 34 and 26; level at 8192 x 1000 and 4096 x 64,
 *  slower at 16384 x 4096 (72 and 180: its reads alone take as long as its chain). Without, a row takes 3.5 ns; with,
 *  0.8 ns, 1.6 ps a column for the second read of the matrix and the less than full rate of the first, and
 *  17 us for the three launches of a band. Several bands only where they win a tenth: 65537 x 1000 232 and 167, 131072 x 1000
 *  460 and 334, 131072 x 513 474 and 233, 100000 x 700 362 and 205, 1048577 x 10 3510 and 710, but 60000 x 1200 210 and 176 to
 *  192, 60000 x 1300 212 and 206 to 216. More than six columns a CU walk in turns.
 *  What the terms are can take the gain away. Columns with roundings that all go one way (equal terms, 1 / 0.9 nine times of
 *  ten), or with an infinity or a NaN: 16384 x 1000 63 and 48 to 57, 65536 x 1000 230 and 140 to 199, 131072 x 10 450 and 90 to
 *  190. Columns that have no map throughout, their sums back at nothing after every other term, pay for the first two launches in
 *  vain: 6800 x 10 29 and 42, 16384 x 100 64 and 79, 16384 x 1000 62 and 110, 40000 x 1200 142 and 265, 65536 x 1000 231 and 406,
 *  131072 x 100 464 and 504; with one such column in a hundred nearly as much. */
inline bool ColumnChunksAreSooner(uint32_t rows, uint32_t cols, uint32_t cus) {
  if (cols > 6u * cus || cols > kMostChunkColumns || static_cast<double>(rows) * (2700.0 - 1.6 * cols) <= 17e6) return false;
  const uint32_t band = ChunkBandRows(rows, cols), bands = (rows + band - 1) / band;
  return bands == 1 || static_cast<double>(rows) * (2350.0 - 1.6 * cols) > 17e6 * bands;
}

}  // namespace mshadow_hipk

#endif  // MSHADOW_AMD_CSRC_COLUMN_CHUNK_PLAN_H_
