/*
 * sum_rows of long float columns by chunks of 128 rows (column_chunks.h has the arithmetic), in three
 * launches: the chunks' sums in any order, their maps, and a walk down every column. The matrix is read twice, by
 * all CUs, where a strip of columns a workgroup leaves most of them idle; the sequence of a column is left
 * to one wave, which takes a chunk in 60 ns, and one that has no map in 500, where 128 dependent adds
 * take 450. 65536 x 1000: 48, 58 and 63 us (the last by the column with the fewest maps). Where the scratch memory does not
 * hold the cells of all rows, they go band by band, the three launches each, from the sums that the walk of the band before left.
 */
#ifndef MSHADOW_AMD_CSRC_COLUMN_CHUNK_KERNELS_H_
#define MSHADOW_AMD_CSRC_COLUMN_CHUNK_KERNELS_H_

#include <float.h>

#include <mshadow/hip/kernels/common.h>
#include <mshadow/hip/kernels/reduce_dma.h>

#include "column_chunk_plan.h"

namespace mshadow_hipk {

using column_chunks::Map;
using column_chunks::Step;
using column_chunks::Windows;
using mshadow::hip::kWave;

struct ColumnChunkScratch {
  Map map[kChunkCells];                             // [column][chunk], what the walk reads
  float copy[kChunkCopies][column_chunks::kRows];   // terms of chunks that are added one by one
  float before[kChunkCells];                        // [chunk][column]: sum of the workgroup's chunks in front
  float group[kChunkGroupCells];                    // [workgroup of chunks][column]
  uint32_t bare[kMostChunkColumns];                 // of a column: chunks that have neither a map nor a copy
  float carry[kMostChunkColumns];                   // a column's sum behind the bands so far
};
static_assert(kChunkStrip == mshadow::hip::kLowestCols, "a strip of the walk is one of the chain kernel's");

/*! \brief a column's terms of N rows: all loads under way together */
template <uint32_t N>
__device__ __forceinline__ void LoadRows(float (&t)[N], const float *src, const ChunkShape &g, uint32_t row0,
                                         uint32_t x) {
  /* a row's address is the wave's, the column's offset a lane's (32 bits: the instruction adds them) */
  const uint32_t at = x * static_cast<uint32_t>(sizeof(float));
  const size_t pitch = static_cast<size_t>(g.stride) * sizeof(float);
  const char *p = reinterpret_cast<const char *>(src) + row0 * pitch;
#pragma unroll
  for (uint32_t i = 0; i < N; ++i) {
    t[i] = *reinterpret_cast<const float *>(p + at);
    p += pitch;
  }
}
/*! \brief whether all rows of a chunk are there: a last one of fewer is added term by term, and nothing waits for its
 *  sum */
__device__ __forceinline__ bool IsWhole(const ChunkShape &g, uint32_t chunk) {
  return (chunk + 1u) * column_chunks::kRows <= g.rows;
}

/*! \brief rows whose loads are under way together in the launch that only sums */
const uint32_t kSumsAtOnce = 32;

/*! \brief the sums of the chunks, in any order of adds: per workgroup of four chunks the sum of those in
 *  front of each, and of all. Bound by its read of the matrix: 65536 x 1000 48 us, 5.5 TB/s; four columns a lane, which
 *  leaves a quarter of the waves, 57. */
__global__ void __launch_bounds__(kChunkWaves *kWave)
    ColumnChunkSumsKernel(const float *src, ChunkShape g, float *before, float *group, uint32_t *bare) {
  __shared__ float sums[kChunkWaves][kWave];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & (kWave - 1);
  const uint32_t piece = mshadow::hip::StripOfBlock(blockIdx.x, gridDim.x);
  const uint32_t at = piece / g.tiles, tile = piece % g.tiles;
  const uint32_t chunk = at * kChunkWaves + wave, pitch = g.tiles * kColumnsPerTile;
  const uint32_t column = tile * kColumnsPerTile + lane;
  const uint32_t x = column < g.cols ? column : g.cols - 1;
  float sum = 0.0f;
  if (IsWhole(g, chunk)) {
    float part[kSumsAtOnce] = {0.0f};
    for (uint32_t i = 0; i < static_cast<uint32_t>(column_chunks::kRows); i += kSumsAtOnce) {
      float t[kSumsAtOnce];
      LoadRows(t, src, g, chunk * column_chunks::kRows + i, x);
#pragma unroll
      for (uint32_t k = 0; k < kSumsAtOnce; ++k) part[k] += t[k];
    }
#pragma unroll
    for (uint32_t step = 1; step < kSumsAtOnce; step *= 2) {
#pragma unroll
      for (uint32_t k = 0; k < kSumsAtOnce; k += 2 * step) part[k] += part[k + step];
    }
    sum = part[0];
  }
  if (at == 0 && wave == 0 && column < g.cols) bare[column] = 0u;
  sums[wave][lane] = sum;
  __syncthreads();
  float front = 0.0f;
  for (uint32_t w = 0; w < wave; ++w) front += sums[w][lane];
  if (chunk < g.chunks) before[static_cast<size_t>(chunk) * pitch + column] = front;
  if (wave == kChunkWaves - 1) group[static_cast<size_t>(at) * pitch + column] = front + sum;
}

/*! \brief the maps of the chunks. A wave keeps its chunk of 64 columns in registers, so that terms to be added
 *  one by one can be copied out; sixteen instructions a term, which the reads hide (58 us on 65536 x 1000, 4.5 TB/s; with
 *  fourteen, without the third window, 55). Workgroups go through
 *  the matrix from its end: what the launch before read last is still in the memory-side cache. */
__global__ void __launch_bounds__(kChunkWaves *kWave, 3)
    ColumnChunkMapsKernel(const float *src, ChunkShape g, const float *before, const float *group, Map *map,
                          float (*copy)[column_chunks::kRows], uint32_t *bare, const float *carry) {
  __shared__ float part[3][kChunkWaves][kWave];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & (kWave - 1);
  const uint32_t piece = gridDim.x - 1u - mshadow::hip::StripOfBlock(blockIdx.x, gridDim.x);
  const uint32_t at = piece / g.tiles, tile = piece % g.tiles;
  const uint32_t chunk = at * kChunkWaves + wave, pitch = g.tiles * kColumnsPerTile;
  const uint32_t column = tile * kColumnsPerTile + lane;
  const uint32_t x = column < g.cols ? column : g.cols - 1;
  const bool live = chunk < g.chunks;
  /* the sums in front: a quarter of the groups a wave, with the largest and smallest sum on the way */
  {
    const uint32_t each = (at + kChunkWaves - 1) / kChunkWaves;
    const uint32_t first = wave * each, end = first + each < at ? first + each : at;
    float sum = 0.0f, high = 0.0f, low = 0.0f;
    const float *p = group + static_cast<size_t>(first) * pitch + column;
    uint32_t i = first;
    for (; i + 8 <= end; i += 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = p[static_cast<size_t>(k) * pitch];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        sum += v[k];
        high = fmaxf(high, sum);
        low = fminf(low, sum);
      }
      p += static_cast<size_t>(8) * pitch;
    }
    for (; i < end; ++i) {
      sum += *p;
      high = fmaxf(high, sum);
      low = fminf(low, sum);
      p += pitch;
    }
    part[0][wave][lane] = sum;
    part[1][wave][lane] = high;
    part[2][wave][lane] = low;
  }
  float t[column_chunks::kRows];
  const float inside = live ? before[static_cast<size_t>(chunk) * pitch + column] : 0.0f;
  const bool whole = IsWhole(g, chunk);
  if (whole) LoadRows(t, src, g, chunk * column_chunks::kRows, x);
  __syncthreads();
  if (!live) return;
  float a = g.begun != 0u ? carry[x] : 0.0f, most = 0.0f;
#pragma unroll
  for (int w = 0; w < kChunkWaves; ++w) {
    most = fmaxf(most, fmaxf(fabsf(a + part[1][w][lane]), fabsf(a + part[2][w][lane])));
    a += part[0][w][lane];
  }
  a += inside;
  if (!whole) {
    const Map m = {a, 0.0f, 0u, column_chunks::How(true, 0u, column_chunks::kInMatrix)};
    if (column < g.cols) map[static_cast<size_t>(column) * g.chunks + chunk] = m;
    return;
  }
  most = fmaxf(most, fabsf(a));
  const float rows_before = static_cast<float>(chunk * column_chunks::kRows);
  Windows j = {column_chunks::kMaxWindow + 1u, 0u};
  if (column_chunks::StartsOnGrid(a)) j = column_chunks::WindowsFor(a, most, rows_before, sqrtf(rows_before));
  const bool tried = j.second <= column_chunks::kMaxWindow;
  if (!tried) j.second = j.third = column_chunks::kMinWindow;
  column_chunks::Chains chains;
  chains.Start(tried ? a : 1.0f, j);
  /* all that is needed of these behind the chains, in one register: there are 168 for three waves a SIMD */
  uint32_t windows = j.second | j.third << 8 | (tried ? 1u << 16 : 0u);
  asm volatile("" : "+v"(windows), "+v"(a));
#pragma unroll
  for (int i = 0; i < column_chunks::kRows; ++i) {
    chains.Add(t[i]);
    if (i % 4 == 3) {
      /* else the compiler runs one chain after the other, makes trees of the maxima and ors, and keeps
         every sum until then (256 registers and as many spilled) */
      asm volatile("" : "+v"(chains.differ), "+v"(chains.far), "+v"(chains.farthest), "+v"(chains.most));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  Map m;
  bool wide;
  j.second = windows & 255u;
  j.third = windows >> 8 & 255u;
  const bool known = chains.Finish(windows >> 16 != 0u ? a : 1.0f, j, &m, &wide) && windows >> 16 != 0u;
  if (!known) {
    uint32_t where = column_chunks::kInMatrix;
    float term = 0.0f;
#pragma unroll
    for (int i = 0; i < column_chunks::kRows; ++i) term = fmaxf(term, fabsf(t[i]));
    const bool nan = chains.s[0] != chains.s[0];
    if (term == 0.0f && !nan) {
      bool plus = false;
#pragma unroll
      for (int i = 0; i < column_chunks::kRows; ++i) plus = plus || __float_as_uint(t[i]) == 0u;
      where = plus ? column_chunks::kPlusZero : column_chunks::kNothing;
    }
    m.how = column_chunks::How(true, 0u, where);
    m.a = a;
    m.shift = term <= FLT_MAX && !nan ? 1u : 0u;
  }
  /* copies of the terms that will or may be asked for */
  const bool copied = column < g.cols && !(known && wide) && column_chunks::WhereOf(m.how) == column_chunks::kInMatrix;
  const uint32_t place = mshadow::hip::LanesBelow(__ballot(copied));
  if (copied && place < g.copies) {
    const uint32_t slot = (chunk * g.tiles + tile) * g.copies + place;
    float4 *to = reinterpret_cast<float4 *>(copy[slot]);
#pragma unroll
    for (int i = 0; i < column_chunks::kRows; i += 4) to[i / 4] = make_float4(t[i], t[i + 1], t[i + 2], t[i + 3]);
    m.how = column_chunks::How(!known, column_chunks::WindowOf(m.how), column_chunks::kKept + slot);
  } else if (copied && !known && column_chunks::Exponent(a) != 255u) {
    __hip_atomic_fetch_add(bare + column, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (column < g.cols) map[static_cast<size_t>(column) * g.chunks + chunk] = m;
}

__device__ __forceinline__ void WaveLdsFence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
/*! \brief columns up to which the walk takes its maps sixteen at once */
inline uint32_t ColumnsOfWideWalk(uint32_t cus) { return 2u * cus; }
/*! \brief stages of a strip's chain, in the LDS that a CU has for each of two or six columns: the longer they are the less
 *  often their first reads are waited for (65536 x 1000 in stages of 64, 96 and 128 rows: 5.1, 4.5 and 4.0 ns a row; but with
 *  128 a CU holds four workgroups, and 30000 x 1000 columns that have maps take 86 us instead of 76) */
typedef mshadow::hip::DmaRing<5, 2048, 2> StripRingOfTwo;
typedef mshadow::hip::DmaRing<4, 1536, 2> StripRingOfSix;

/*! \brief 128 additions, the terms read from LDS a block of 32 ahead */
__device__ __forceinline__ void AddTerms(float *sum, const float4 *term) {
  const int kBlock = 8, kBlocks = column_chunks::kRows / 4 / kBlock;
  float4 v[2][kBlock];
#pragma unroll
  for (int k = 0; k < kBlock; ++k) v[0][k] = term[k];
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    if (b + 1 < kBlocks) {
#pragma unroll
      for (int k = 0; k < kBlock; ++k) v[(b + 1) & 1][k] = term[(b + 1) * kBlock + k];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kBlock; ++k) {
      *sum += v[b & 1][k].x;
      *sum += v[b & 1][k].y;
      *sum += v[b & 1][k].z;
      *sum += v[b & 1][k].w;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

/*! \brief chunks the walk takes between two barriers; blocks on their way or in use; waves that bring them in turn */
const uint32_t kWalkBlock = 16;
const uint32_t kWalkLoaders = 2;
const uint32_t kWalkRing = kWalkLoaders + 1;
/*! \brief in the place of a window: the terms are here; there are none; there are only zeros, a +0 among them; the sum in
 *  front is expected to be infinite or NaN, which mostly asks for no terms */
const uint32_t kWalkTerms = 0xbf800000u, kWalkNothing = 0xc0000000u, kWalkPlusZero = 0xc0400000u, kWalkNoSum = 0xc0800000u;
struct WalkBlock {
  float4 step[kWalkBlock];  // Step's a, inverse, e0, grid
  uint2 rest[kWalkBlock];   // Step's shift, window
  uint32_t here;            // bit c: the terms of chunk c are here
  float4 term[kWalkBlock][column_chunks::kRows / 4];  // of the chunks that are added term by term
};

/*! \brief whether a column has so many chunks that ask for the matrix that it is left to the chain */
__device__ __forceinline__ bool TakesChain(uint32_t bare, const ChunkShape &g) { return g.strips != 0u && bare > g.most_bare; }

/*! \brief the sums themselves: a wave walks down a column, every lane with the same sum, and reads nothing but
 *  LDS. Two more bring it the maps, and the terms of the chunks that have none: a block each in turn,
 *  asked for two blocks ahead. Bound by the walk's sequence: a wave alone issues an instruction every 3.5 ns. The
 *  first workgroups have a strip of 16 columns each, of which they add those that TakesChain from top to bottom.
 *  AT_ONCE: maps in registers together. All of a block where two columns a CU at most leave the registers for it
 *  (65536 x 64 of columns with a map for every chunk 28.9 us, 35.0 with eight; 30000 x 100 gradients 25.2 and 27.8), four
 *  where four have to share a CU (65536 x 1000 gradients 61 to 64 us, with eight 58 to 76, with sixteen 80: columns then wait
 *  for others to end). */
template <typename Saver, uint32_t AT_ONCE, typename StripRing>
__global__ void __launch_bounds__((1 + kWalkLoaders) * kWave)
    ColumnChunkWalkKernel(float *dst, const float *src, ChunkShape g, const Map *map,
                          const float (*copy)[column_chunks::kRows], const uint32_t *bare, float *carry, float scale) {
  __shared__ union {
    WalkBlock ring[kWalkRing];
    __attribute__((aligned(16))) float strip[StripRing::kSlots][StripRing::kElems];
  } lds;
  __shared__ uint32_t misses;  // chunks whose map did not cover the sum
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & (kWave - 1);
  if (blockIdx.x < g.strips) {
    const uint32_t x0 = mshadow::hip::StripOfBlock(blockIdx.x, g.strips) * kChunkStrip;
    const bool chain = lane < kChunkStrip && x0 + lane < g.cols && TakesChain(bare[x0 + lane], g);
    if (__ballot(chain) == 0ull) return;
    const float from = chain && g.begun != 0u ? carry[x0 + lane] : -0.0f;
    mshadow::hip::LowestDmaFold<mshadow::red::sum, StripRing, true>(
        lds.strip, src, g.stride, g.rows, g.cols, x0, chain, from, [=](float sum, uint32_t l) {
          if (g.more != 0u) carry[x0 + l] = sum;
          else Saver::template Save<float>(dst[x0 + l], sum * scale);
        });
    return;
  }
  WalkBlock *ring = lds.ring;
  const uint32_t x = blockIdx.x - g.strips;
  const uint32_t blocks = (g.chunks + kWalkBlock - 1) / kWalkBlock;
  const Map *mine = map + static_cast<size_t>(x) * g.chunks;
  auto fetch = [&](uint32_t block) {
    const uint32_t c = block * kWalkBlock + lane % kWalkBlock;
    return mine[c < g.chunks ? c : g.chunks - 1];
  };
  Map now = {};
  if (wave != 0) now = fetch(wave - 1);
  if (TakesChain(bare[x], g)) return;
  if (threadIdx.x == 0) misses = 0u;
  __syncthreads();

  if (wave != 0) {
    for (uint32_t b = 0; b < blocks + kWalkLoaders; ++b) {
      if (b % kWalkLoaders == wave - 1) {
        if (b < blocks) {
          WalkBlock *to = &ring[b % kWalkRing];
          const uint32_t first = b * kWalkBlock;
          /* where the maps keep missing the sum, every chunk's terms */
          const uint32_t missed =
              __hip_atomic_load(&misses, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          const bool all = __builtin_amdgcn_readfirstlane(missed > 8u && missed * 4u > first ? 1u : 0u) != 0u;
          const bool live = lane < kWalkBlock && first + lane < g.chunks;
          const bool mapped = !column_chunks::IsByTerms(now.how);
          const uint32_t where = column_chunks::WhereOf(now.how);
          const bool nothing = where == column_chunks::kNothing, plus = where == column_chunks::kPlusZero;
          const bool no_sum = !mapped && column_chunks::Exponent(now.a) == 255u;
          unsigned long long wanted =
              __ballot(live && !no_sum && (where >= column_chunks::kKept ||
                                           (where == column_chunks::kInMatrix && (all || !mapped))));
          if (lane < kWalkBlock) {
            const Step st = column_chunks::StepOf(now);
            const uint32_t window = !live || nothing ? kWalkNothing
                                    : plus           ? kWalkPlusZero
                                    : no_sum         ? kWalkNoSum
                                    : mapped         ? __float_as_uint(st.window)
                                                     : kWalkTerms;
            to->step[lane] = make_float4(st.a, st.inverse, st.e0, st.grid);
            to->rest[lane] = make_uint2(st.shift, window);
            to->here = static_cast<uint32_t>(wanted);
          }
          while (wanted != 0ull) {
            const uint32_t c = __builtin_ctzll(wanted);
            wanted &= wanted - 1ull;
            const uint32_t place = mshadow::hip::ReadLaneU32(where, c);
            float *term = reinterpret_cast<float *>(to->term[c]);
            const uint32_t row0 = (first + c) * column_chunks::kRows;
            if (place >= column_chunks::kKept) {
              const float *from = copy[place - column_chunks::kKept];
              mshadow::hip::LoadDwordToLds(from + lane, term);
              mshadow::hip::LoadDwordToLds(from + kWave + lane, term + kWave);
            } else if (row0 + column_chunks::kRows <= g.rows) {
              const float *from = src + static_cast<size_t>(row0 + lane) * g.stride + x;
              mshadow::hip::LoadDwordToLds(from, term);
              mshadow::hip::LoadDwordToLds(from + static_cast<size_t>(kWave) * g.stride, term + kWave);
            } else {
              for (uint32_t i = lane; i < static_cast<uint32_t>(column_chunks::kRows); i += kWave) {
                term[i] = row0 + i < g.rows ? src[static_cast<size_t>(row0 + i) * g.stride + x] : -0.0f;
              }
            }
          }
          now = fetch(b + kWalkLoaders);
        }
      }
      /* the walk comes to a block kWalkLoaders steps behind its turn */
      if ((b + 1u) % kWalkLoaders == wave - 1) mshadow::hip::WaitAllLanded();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      mshadow::hip::BareBarrier();
    }
    mshadow::hip::WaitAllLanded();  // no load is under way when the workgroup's LDS is handed on
    return;
  }

  uint32_t missed = 0u;
  float sum = g.begun != 0u ? carry[x] : -0.0f;  // the identity: the reference starts from the first term
  for (uint32_t b = 0; b < blocks + kWalkLoaders; ++b) {
    if (b >= kWalkLoaders) {
      WalkBlock *blk = &ring[(b - kWalkLoaders) % kWalkRing];
      const uint32_t first = (b - kWalkLoaders) * kWalkBlock;
      const uint32_t count = g.chunks - first < kWalkBlock ? g.chunks - first : kWalkBlock;
      for (uint32_t c = 0; c < count; c += AT_ONCE) {
        float4 va[AT_ONCE];
        uint2 vb[AT_ONCE];
#pragma unroll
        for (uint32_t i = 0; i < AT_ONCE; ++i) {
          va[i] = blk->step[c + i];
          vb[i] = blk->rest[c + i];
        }
#pragma unroll
        for (uint32_t i = 0; i < AT_ONCE; ++i) {
          const Step m = {va[i].x, va[i].y, va[i].z, va[i].w, vb[i].x, __uint_as_float(vb[i].y)};
          float to;
          if (__ballot(column_chunks::Apply(m, sum, &to)) != 0ull) {
            sum = to;
            continue;
          }
          const uint32_t window = __builtin_amdgcn_readfirstlane(vb[i].y);
          if (window == kWalkNothing) continue;
          if (window == kWalkPlusZero) {
            sum += 0.0f;
            continue;
          }
          float4 *term = blk->term[c + i];
          if (window != kWalkTerms) {
            /* The map does not cover the sum, or there is none. A sum that is infinite or NaN stays what it is, but for an
               infinity that meets another or a NaN. */
            if (column_chunks::Exponent(sum) == 255u &&
                (sum != sum || window != kWalkNoSum || __builtin_amdgcn_readfirstlane(vb[i].x) != 0u)) {
              continue;
            }
            if ((__builtin_amdgcn_readfirstlane(blk->here) >> (c + i) & 1u) == 0u) {
              const uint32_t row0 = (first + c + i) * column_chunks::kRows;
              for (uint32_t k = lane; k < static_cast<uint32_t>(column_chunks::kRows); k += kWave) {
                reinterpret_cast<float *>(term)[k] =
                    row0 + k < g.rows ? src[static_cast<size_t>(row0 + k) * g.stride + x] : -0.0f;
              }
            }
            /* enough of these and the other waves bring all terms */
            __hip_atomic_store(&misses, ++missed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            WaveLdsFence();
          }
          AddTerms(&sum, term);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    mshadow::hip::BareBarrier();
  }
  if (lane == 0) {
    if (g.more != 0u) carry[x] = sum;
    else Saver::template Save<float>(dst[x], sum * scale);
  }
}

}  // namespace mshadow_hipk

#endif  // MSHADOW_AMD_CSRC_COLUMN_CHUNK_KERNELS_H_
