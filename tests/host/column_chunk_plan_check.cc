// Which column sums go by chunks, and in which bands of rows (csrc/column_chunk_plan.h): the shapes that the GPU tests take for
// summed that way and for not, both sides of what the scratch memory holds, and that every band fits it.
#include <cstdio>
#include <random>

#include "../../mshadow_amd/csrc/column_chunk_plan.h"

using namespace mshadow_hipk;

static const uint32_t kCus = 256;
static int g_wrong = 0;

static void Expect(uint32_t rows, uint32_t cols, bool sooner, uint32_t bands) {
  const uint32_t per = ChunkBandRows(rows, cols);
  const bool use = ColumnChunksAreSooner(rows, cols, kCus);
  if (use == sooner && (!use || (rows + per - 1) / per == bands)) return;
  ++g_wrong;
  printf("%u x %u: %d in bands of %u\n", rows, cols, use, per);
}

int main() {
  // tests/test_gpu_column_chunks.py: without, at the edges of tiles, chunks, workgroups and of the walk's blocks
  const uint32_t without[][2] = {{6300, 10}, {6528, 64}, {8192, 1000}, {4096, 64}, {16384, 4096}, {131072, 1537}};
  for (const auto &s : without) Expect(s[0], s[1], false, 0);
  const uint32_t one[][2] = {{6400, 10}, {6656, 64}, {6657, 65}, {6783, 63}, {8192, 1}, {8193, 3}, {8320, 129}, {10240, 128}, {9200, 512},
                             {9200, 513}, {16384, 1000}, {20481, 17}, {33000, 300}, {12345, 70}, {9300, 300}, {16411, 999}};
  for (const auto &s : one) Expect(s[0], s[1], true, 1);
  // the last that one band holds, and the first of two: 8192 chunks of a tile, 512 of sixteen
  Expect(1048576, 3, true, 1);
  Expect(1048577, 3, true, 2);
  Expect(65536, 1000, true, 1);
  Expect(65537, 1000, true, 2);
  Expect(131072, 512, true, 1);
  Expect(131072, 513, true, 2);
  Expect(2097281, 5, true, 3);
  Expect(66001, 1000, true, 2);
  Expect(131072, 1000, true, 2);
  Expect(100000, 700, true, 2);
  Expect(60000, 1300, false, 0);

  std::mt19937 rng(4);
  for (int i = 0; i < 1000000; ++i) {
    const uint32_t rows = 1 + (rng() >> (1 + rng() % 25)), cols = 1 + rng() % kMostChunkColumns;
    if (!ColumnChunksAreSooner(rows, cols, kCus)) continue;
    const uint32_t per = ChunkBandRows(rows, cols);
    bool fits = per >= 1 && per % (kChunkWaves * column_chunks::kRows) == 0;
    const uint32_t left = fits ? (rows - 1) % per + 1 : 1;
    for (const uint32_t band : {rows < per ? rows : per, left}) {
      const ChunkShape g = MakeChunkShape(band, cols, cols, kCus);
      const uint64_t cells = static_cast<uint64_t>(g.chunks) * g.tiles, padded = cells * kColumnsPerTile;
      fits = fits && padded <= kChunkCells && g.copies >= 1 && cells * g.copies <= kChunkCopies &&
             static_cast<uint64_t>(g.groups) * g.tiles * kColumnsPerTile <= kChunkGroupCells && cols <= kMostChunkColumns &&
             static_cast<uint64_t>(g.chunks) * column_chunks::kRows < (1ull << 32);
    }
    if (!fits && ++g_wrong < 10) printf("%u x %u in bands of %u does not fit\n", rows, cols, per);
  }
  if (g_wrong == 0) printf("OK\n");
  return g_wrong != 0;
}
