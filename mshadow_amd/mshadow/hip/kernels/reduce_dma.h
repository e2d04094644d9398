/*
 * Reduce-to-1D of a plain float tensor with the loads delivered straight into LDS.
 *
 * Same order of operations as the kernels in reduce.h (one serial chain per output, see
 * there for why), different plumbing. When the source is a tensor in memory - not an
 * expression that has to be evaluated in registers - the loader waves use the
 * global-load-to-LDS instruction of gfx950: the data never passes through VGPRs, so the
 * depth of the pipeline is limited by LDS (a ring of 128 KB: up to six stages = 96 KB
 * per CU in flight) instead of by registers and by what the compiler can prove
 * about loop-carried loads. Roles are fixed per wave:
 *   waves 1..8  issue the loads of stage i, wait (by count) for their own loads of
 *               an earlier stage to have landed, and meet the barrier; they never read LDS,
 *               fetch nothing past the last stage and exit with no load outstanding;
 *   wave 0      after the barrier folds that stage from its slot with 128-bit LDS reads,
 *               one dependent add per element; it never touches global memory.
 * A slot is refilled two barriers after the chain has finished with it.
 *
 * The load instruction places lane l's dword at (wave base + 4 l) in LDS, so the layout
 * of a slot is chosen per kernel such that the lanes of one instruction fetch full
 * 64-byte runs of global memory AND a chain lane finds four consecutive operands in one
 * 16-byte LDS word.
 *
 * The barrier here is the bare instruction: the usual workgroup fence in front of it
 * would wait for every outstanding load, which is exactly what the ring avoids. Ordering
 * is by construction: a loader's wait-by-count precedes its barrier, and the chain's LDS
 * reads have returned (their sums depend on them) before it reaches the next barrier.
 */
#ifndef MSHADOW_HIP_KERNELS_REDUCE_DMA_H_
#define MSHADOW_HIP_KERNELS_REDUCE_DMA_H_

#include "../../core/fastdiv.h"
#include "./common.h"
#include "./reduce.h"

namespace mshadow {
namespace hip {

/*! \brief loader waves per workgroup (one more wave runs the chains) */
const int kDmaLoaders = 8;
const int kDmaThreads = (kDmaLoaders + 1) * kWave;
/*! \brief LDS ring of SLOTS slots of ELEMS floats each (128 KB in all): SLOTS - 2 stages
 *  are in flight. KeepHighDim is bound by HBM and takes many small stages (deep queue);
 *  KeepLowest is bound by its chain of dependent adds and takes few large ones, so that
 *  the LDS latency at the start of a stage is paid less often. */
template <int SLOTS_, int ELEMS_, int LOADERS_ = kDmaLoaders>
struct DmaRing {
  static const int kLoaders = LOADERS_;
  static const int kSlots = SLOTS_;
  static const int kElems = ELEMS_;
  static const int kAhead = SLOTS_ - 2;
  /*! \brief load instructions per loader wave per stage (64 dwords each) */
  static const int kPerWave = ELEMS_ / kWave / LOADERS_;
  static_assert(kAhead * kPerWave < 64, "the wait-by-count immediate has 6 bits");
};
typedef DmaRing<4, 8192> LowestRing;
typedef DmaRing<8, 4096> HighDimRing;

/*! \brief cache policy of the loads: non-temporal (the data passes through once; measured
 *  38 us against 43 us for the (64,256,56,56) reduction) */
const int kDmaCachePolicy = 2;
/*! \brief lane l of the wave fetches the 4 bytes at gsrc_of_lane into the l-th dword behind
 *  lds_wave_base */
__device__ __forceinline__ void LoadDwordToLds(const void *gsrc_of_lane, void *lds_wave_base) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void *)gsrc_of_lane,
      (__attribute__((address_space(3))) void *)lds_wave_base, 4, 0, kDmaCachePolicy);
}
template <int BYTES>
__device__ __forceinline__ void LoadLaneToLds(const void *gsrc_of_lane, void *lds_wave_base) {
  const __attribute__((address_space(1))) void *from =
      (const __attribute__((address_space(1))) void *)gsrc_of_lane;
  __attribute__((address_space(3))) void *to = (__attribute__((address_space(3))) void *)lds_wave_base;
  if (BYTES == 16) {
    __builtin_amdgcn_global_load_lds(from, to, 16, 0, kDmaCachePolicy);
  } else {
    __builtin_amdgcn_global_load_lds(from, to, 4, 0, kDmaCachePolicy);
  }
}

/*! \brief all but the newest kAhead stages of this wave's loads have landed */
template <typename Ring>
__device__ __forceinline__ void WaitStageLanded() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Ring::kAhead * Ring::kPerWave) : "memory");
}
/*! \brief every load of this wave has landed (used once the last stage has been issued:
 *  nothing is fetched past the end, and no load is outstanding when the wave exits and
 *  the workgroup's LDS is handed to the next one) */
__device__ __forceinline__ void WaitAllLanded() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void BareBarrier() { asm volatile("s_barrier" ::: "memory"); }

/* ------------------------------------------------------------------ KeepLowest
 * 16 columns per workgroup. A stage is 512 rows; one load instruction covers a group of
 * four rows: lane l fetches row 4 g + (l & 3), column l >> 2, so the slot holds
 * [group][column][row & 3] and a chain lane reads rows 4g..4g+3 of its column as one
 * 128-bit word, 64 floats from the next group. */
/*! \brief a workgroup of 1 + Ring::kLoaders waves; lane l of wave 0 folds column x0 + l if that is `wanted`, and calls
 *  done(result, l). BEGUN: on from `res`; else from the first row. */
template <typename Reducer, typename Ring, bool BEGUN, typename Done>
__device__ __forceinline__ void LowestDmaFold(float (*ring)[Ring::kElems], const float *src, uint32_t stride, uint32_t rows,
                                              uint32_t cols, uint32_t x0, bool wanted, float res, Done done) {
  const int kDmaSlots = Ring::kSlots, kDmaAhead = Ring::kAhead, kDmaPerWave = Ring::kPerWave;
  const int CW = kLowestCols;
  const int TR = Ring::kElems / CW;

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t nstage = (rows + TR - 1) / TR;
  const uint32_t nstep = nstage == 0 ? 0 : nstage + kDmaAhead;

  if (wave != 0) {
    const uint32_t lw = wave - 1;
    const uint32_t r = lane & 3;
    /* out-of-range columns and rows re-read the last valid one: never consumed */
    const uint32_t xc = (x0 + (lane >> 2) < cols) ? x0 + (lane >> 2) : cols - 1;
    const float *colp = src + xc;
    for (uint32_t i = 0; i < nstep; ++i) {
      if (i < nstage) {
        float *slot = ring[i % kDmaSlots];
#pragma unroll
        for (int q = 0; q < kDmaPerWave; ++q) {
          const uint32_t g = q * Ring::kLoaders + lw;
          uint32_t row = i * TR + g * 4 + r;
          row = row < rows ? row : rows - 1;
          LoadDwordToLds(colp + static_cast<size_t>(row) * stride, slot + g * kWave);
        }
        WaitStageLanded<Ring>();
      } else {
        WaitAllLanded();
      }
      BareBarrier();
    }
  } else {
    const bool chain_lane = lane < static_cast<uint32_t>(CW) && x0 + lane < cols && wanted;
    for (uint32_t i = 0; i < nstep; ++i) {
      BareBarrier();
      if (i >= static_cast<uint32_t>(kDmaAhead) && chain_lane) {
        const uint32_t st = i - kDmaAhead;
        const uint32_t row0 = st * TR;
        const float *mine = ring[st % kDmaSlots] + lane * 4;
        const int count = (rows - row0 < (uint32_t)TR) ? static_cast<int>(rows - row0) : TR;
        int begin = 0;
        if (!BEGUN && st == 0) {  // the reference starts from src(0, x), not from an initial value
          res = mine[0];
          begin = 1;
        }
        ChainFold<Reducer, kWave>(res, mine, begin, count);
      }
    }
    if (chain_lane) done(res, lane);
  }
}
template <typename Saver, typename Reducer>
__global__ void __launch_bounds__(kDmaThreads)
    ReduceKeepLowestDmaKernel(float *dst, const float *src, uint32_t stride, uint32_t rows,
                              uint32_t cols, float scale) {
  __shared__ MSHADOW_ALIGNED(16) float ring[LowestRing::kSlots][LowestRing::kElems];
  const uint32_t x0 = StripOfBlock(blockIdx.x, gridDim.x) * kLowestCols;
  LowestDmaFold<Reducer, LowestRing, false>(
      ring, src, stride, rows, cols, x0, true, 0.0f,
      [=](float res, uint32_t lane) { Saver::template Save<float>(dst[x0 + lane], res * scale); });
}

/* ------------------------------------------------------------------ KeepLowest in strips
 * The same roles and ring, a slot holding ROWS rows as they lie in memory. A load instruction
 * covers one or more whole rows of the strip, so a strip of 64 floats fetches whole cache lines
 * where the kernel above fetches 64 bytes at a time, and every lane of the chain wave has a
 * column to add; a chain lane reads its column of one row after the other, neighbouring lanes
 * neighbouring words. The ring is small (16 to 64 KB), so that several workgroups share a CU and
 * a short reduction does not fetch rows it does not have.
 *
 * What bounds it, and hence the width of the strips: a CU's requests bring about 43 GB/s at most
 * and a chain step takes 4.2 to 5.9 ns, so as many CUs as possible must have a strip, and as few
 * as possible more than one round of them (LowestColumnsPerStrip). Measured, sums of floats,
 * before (16 columns per workgroup, 128 KB ring) and now: 8192 x 32000 299 -> 174 us (6.0 TB/s),
 * 2048 x 50257 215 -> 77 us (5.3 TB/s), 512 x 50000 78 -> 20 us, 128 x 128000 106 -> 13 us,
 * 16384 x 8192 149 -> 87 us, 1500 x 1000 12.5 -> 10 us, 128 x 10 3.8 -> 2.8 us (the kernel alone: calls that short wait for
 * their launches); binary16
 * (register-staged kernel of reduce.h before) 8192 x 32000 260 -> 81 us, 4096 x 9000 52 -> 25 us.
 * Sixteen bytes a lane instead of four fetch no faster (8192 x 32000: 174 us both). */

/*! \brief columns of a strip by the number of columns and of CUs: narrow strips until every CU
 *  has one (with 8192 x 6000 floats: 16 columns 52 us, 32 columns 43 us, 64 columns 52 us), wide
 *  ones - whole cache lines - from there on (8192 x 10000: 78, 71 and 59 us) */
inline int LowestColumnsPerStrip(uint32_t cols, uint32_t cus) {
  return cols <= 16 * cus ? 16 : cols <= 32 * cus ? 32 : 64;
}

/*! \brief PITCH elements of a row in LDS, ROWS rows a slot. SHIFTED (16-bit elements only): rows
 *  need not start at 4-byte borders. A load then brings the dwords that hold the strip, whose
 *  elements sit one place further in rows that start at an odd element, and a strip has two
 *  columns less than the pitch. */
template <typename DType, int PITCH, int ROWS, int SLOTS, int LOADERS, int PER_LANE, bool SHIFTED>
struct LowestStrip {
  typedef DType Type;
  static const bool kShifted = SHIFTED;
  static const int kPitch = PITCH;
  static const int kCols = SHIFTED ? PITCH - 2 : PITCH;
  static const int kRows = ROWS;
  static const int kSlots = SLOTS;
  static const int kAhead = SLOTS - 2;
  static const int kLoaders = LOADERS;
  static const int kThreads = (LOADERS + 1) * kWave;
  static const int kElemsPerDword = 4 / sizeof(DType);
  static const int kLanesPerRow = PITCH / kElemsPerDword;
  static const int kRowsPerLoad = kWave / kLanesPerRow;
  static const int kPerWave = ROWS / kRowsPerLoad / LOADERS;
  /*! \brief columns of a chain lane */
  static const int kPerLane = PER_LANE;
  static const int kChainLanes = kCols / PER_LANE;
  static_assert(kWave % kLanesPerRow == 0 && ROWS % (kRowsPerLoad * LOADERS) == 0, "whole loads");
  static_assert(kChainLanes <= kWave && kAhead >= 1 && kAhead * kPerWave < 64, "ring");
  static_assert(!SHIFTED || (sizeof(DType) == 2 && PER_LANE == 1 && LOADERS % 2 == 0), "shifted rows");
};
typedef LowestStrip<float, 16, 64, 4, 4, 1, false> LowestStrip16;
/*! \brief 2048 rows to where the kernel above is the faster one: longer stages, whose first LDS reads
 *  are waited for less often (4096 x 2000: 20.4 us, with 64 rows a stage 22.9 us, the kernel above
 *  22.1 us) */
typedef LowestStrip<float, 16, 256, 4, 8, 1, false> LowestStrip16Long;
typedef LowestStrip<float, 32, 64, 4, 4, 1, false> LowestStrip32;
typedef LowestStrip<float, 64, 64, 4, 8, 1, false> LowestStrip64;
/*! \brief up to 1024 rows and more than two strips per CU: half the ring, twice the workgroups on
 *  a CU (128 x 128000: 13 against 18 us; 4096 x 9000: 38 against 32 us) */
typedef LowestStrip<float, 64, 32, 4, 4, 1, false> LowestStrip64Short;
typedef LowestStrip<half::half_t, 32, 128, 4, 4, 1, false> LowestHalfStrip32;
typedef LowestStrip<half::half_t, 64, 64, 4, 4, 1, false> LowestHalfStrip64;
/*! \brief a packed add of two columns has a longer latency (5.7 ns against 4.9 ns a row) but makes
 *  strips of whole cache lines possible: 8192 x 32000 81 against 87 us */
typedef LowestStrip<half::half_t, 128, 32, 4, 4, 2, false> LowestHalfStrip128;
typedef LowestStrip<half::half_t, 32, 128, 4, 4, 1, true> LowestHalfStrip30;
typedef LowestStrip<half::half_t, 64, 64, 4, 4, 1, true> LowestHalfStrip62;

/*! \brief one step of the chains of a lane: N columns side by side */
template <typename Reducer, typename DType, int N>
struct ChainStep {
  static __device__ __forceinline__ void Run(expr::Pack<DType, N> &res, const expr::Pack<DType, N> &v) {
#pragma unroll
    for (int i = 0; i < N; ++i) Reducer::Reduce(res.v[i], v.v[i]);
  }
};
/*! \brief two binary16 sums: one packed add, which rounds each half as half_t's += does */
template <>
struct ChainStep<red::sum, half::half_t, 2> {
  typedef _Float16 Pair __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ void Run(expr::Pack<half::half_t, 2> &res,
                                             const expr::Pack<half::half_t, 2> &v) {
    Pair a, b;
    __builtin_memcpy(&a, &res, sizeof(a));
    __builtin_memcpy(&b, &v, sizeof(b));
    a += b;
    __builtin_memcpy(static_cast<void *>(&res), &a, sizeof(a));
  }
};

/*! \brief fold a lane's column(s) of a slot, `count` rows (FULL: the whole slot), in order; even
 *  rows from `even`, odd ones from `odd`. The slot is read block by block, one block ahead of the
 *  folds; everything is unrolled, so that the waits are for exactly the block in front. `first`:
 *  the chain starts from row 0's values, as the reference's does, not from an initial value. */
template <typename Reducer, typename Strip, bool FULL, typename P>
__device__ __forceinline__ void StripFold(P &res, const typename Strip::Type *even,
                                          const typename Strip::Type *odd, int count, bool first) {
  typedef typename Strip::Type DType;
  const int kBlk = 16, kBlocks = Strip::kRows / kBlk;
  static_assert(Strip::kRows % kBlk == 0, "whole blocks");
  P v[2][kBlk];
#pragma unroll
  for (int k = 0; k < kBlk; ++k) {
    v[0][k] = *reinterpret_cast<const P *>((k & 1 ? odd : even) + k * Strip::kPitch);
  }
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) {
    if (b + 1 < kBlocks) {
#pragma unroll
      for (int k = 0; k < kBlk; ++k) {
        v[(b + 1) & 1][k] = *reinterpret_cast<const P *>((k & 1 ? odd : even) +
                                                         ((b + 1) * kBlk + k) * Strip::kPitch);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!FULL && b * kBlk >= count) break;
#pragma unroll
    for (int k = 0; k < kBlk; ++k) {
      if (b == 0 && k == 0 && first) {
        res = v[0][0];
      } else if (FULL || b * kBlk + k < count) {
        ChainStep<Reducer, DType, Strip::kPerLane>::Run(res, v[b & 1][k]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename Saver, typename Reducer, typename Strip>
__global__ void __launch_bounds__(Strip::kThreads)
    ReduceKeepLowestStripKernel(typename Strip::Type *dst, const typename Strip::Type *src, uint32_t stride,
                                uint32_t rows, uint32_t cols, typename Strip::Type scale) {
  typedef typename Strip::Type DType;
  const int ROWS = Strip::kRows, kSlots = Strip::kSlots, kAhead = Strip::kAhead;
  const int kPerWave = Strip::kPerWave, N = Strip::kPerLane;
  typedef expr::Pack<DType, Strip::kPerLane> P;
  __shared__ MSHADOW_ALIGNED(16) DType ring[kSlots][ROWS * Strip::kPitch];

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t x0 = StripOfBlock(blockIdx.x, gridDim.x) * Strip::kCols;
  const uint32_t nstage = (rows + ROWS - 1) / ROWS;
  const uint32_t nstep = nstage + kAhead;
  /* workgroups that share a CU run their chains on different SIMDs (see the split kernel below) */
  const uint32_t chain_wave = (blockIdx.x ^ (blockIdx.x >> 8)) & 1u;
  if (wave != chain_wave) {
    const uint32_t lw = wave < chain_wave ? wave : wave - 1;
    /* This lane's place in a row of the strip. Out-of-range columns and rows re-read the last valid
       ones: never consumed. The rows of a lane's loads lie an even number of rows apart and so are
       shifted alike: one address, moved on by a constant. */
    const uint32_t at = lane % Strip::kLanesPerRow;
    auto place = [&](uint32_t row) -> const char * {
      const DType *from = src + static_cast<size_t>(row) * stride;
      if (Strip::kShifted) {
        const uintptr_t whole = ~static_cast<uintptr_t>(3);
        const uintptr_t mine = (reinterpret_cast<uintptr_t>(from + x0) & whole) + at * 4u;
        const uintptr_t last = reinterpret_cast<uintptr_t>(from + (cols - 1)) & whole;
        return reinterpret_cast<const char *>(mine < last ? mine : last);
      }
      const uint32_t x = x0 + at * Strip::kElemsPerDword;
      return reinterpret_cast<const char *>(from + (x < cols ? x : cols - Strip::kElemsPerDword));
    };
    const uint32_t row0 = lw * Strip::kRowsPerLoad + lane / Strip::kLanesPerRow;
    const uint32_t step_rows = Strip::kLoaders * Strip::kRowsPerLoad;
    const char *from = place(row0 < rows ? row0 : rows - 1);
    const size_t step = static_cast<size_t>(step_rows) * stride * sizeof(DType);
    for (uint32_t i = 0; i < nstep; ++i) {
      if (i < nstage) {
        DType *slot = ring[i % kSlots] + lw * Strip::kRowsPerLoad * Strip::kPitch;
        const bool whole_stage = (i + 1) * ROWS <= rows;
#pragma unroll
        for (int q = 0; q < kPerWave; ++q) {
          const char *p = from + q * step;
          if (!whole_stage) {
            const uint32_t row = i * ROWS + q * step_rows + row0;
            p = place(row < rows ? row : rows - 1);
          }
          LoadLaneToLds<4>(p, slot + q * step_rows * Strip::kPitch);
        }
        from += kPerWave * step;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAhead * kPerWave) : "memory");
      } else {
        WaitAllLanded();
      }
      BareBarrier();
    }
    return;
  }
  P res;
#pragma unroll
  for (int k = 0; k < N; ++k) res.v[k] = DType(0);
  const uint32_t chain_lane = lane < static_cast<uint32_t>(Strip::kChainLanes) ? lane : 0;
  uint32_t even = chain_lane * N, odd = even;
  if (Strip::kShifted) {  // a slot has an even number of rows: the same places in every slot
    const uint32_t first = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(src) / sizeof(DType)) + x0;
    even += first & 1u;
    odd += (first + stride) & 1u;
  }
  for (uint32_t i = 0; i < nstep; ++i) {
    BareBarrier();
    if (i < static_cast<uint32_t>(kAhead)) continue;
    const uint32_t st = i - kAhead;
    const DType *slot = ring[st % kSlots];
    const uint32_t left = rows - st * ROWS;
    if (left >= static_cast<uint32_t>(ROWS)) {
      StripFold<Reducer, Strip, true>(res, slot + even, slot + odd, ROWS, st == 0);
    } else {
      StripFold<Reducer, Strip, false>(res, slot + even, slot + odd, static_cast<int>(left), st == 0);
    }
  }
  const uint32_t x = x0 + lane * N;
  if (lane < static_cast<uint32_t>(Strip::kChainLanes)) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if (x + k < cols) Saver::template Save<DType>(dst[x + k], res.v[k] * scale);
    }
  }
}

/* ------------------------------------------------------------------ KeepHighDim
 * shape viewed as (n_out, n_keep, n_y, n_x); one workgroup per kept index c; SEGS inner
 * segments (n values) side by side in a slot, TL = 4096 / SEGS elements of each per
 * stage, one chain lane per segment. One load instruction fetches 64 consecutive
 * elements of one segment into their place in the slot. */
/* The element type is float or a 16-bit type: a load moves a dword per lane, i.e. one float or
 * two neighbouring 16-bit elements, which must then lie in one row of the source (n_x and the
 * pitch even, the base 4-byte aligned: the launcher's business). */
template <typename Saver, typename Reducer, typename DType, int SEGS>
__global__ void __launch_bounds__(kDmaThreads)
    ReduceKeepHighDimDmaKernel(DType *dst, const DType *src, uint32_t stride, uint32_t n_out,
                               uint32_t n_keep, uint32_t n_y, uint32_t n_x, FastDivU32 div_x,
                               DType scale) {
  typedef HighDimRing Ring;
  const int kDmaSlots = Ring::kSlots, kDmaAhead = Ring::kAhead, kDmaPerWave = Ring::kPerWave;
  const int EPD = 4 / sizeof(DType);       // elements per dword
  const int TL = Ring::kElems * EPD / SEGS;
  const int LD = TL + 16 / sizeof(DType);  // chain lanes read words LD elements apart: no bank conflicts
  static_assert(sizeof(DType) == 4 || sizeof(DType) == 2, "a dword holds one or two elements");
  static_assert(TL % (kWave * EPD) == 0, "an instruction stays inside one segment");
  __shared__ MSHADOW_ALIGNED(16) DType ring[Ring::kSlots][SEGS * LD];

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t c = blockIdx.x;
  const uint32_t seg_len = n_y * n_x;
  const uint32_t stages_per_group = (seg_len + TL - 1) / TL;
  const uint32_t groups = (n_out + SEGS - 1) / SEGS;
  const uint32_t nstage = groups * stages_per_group;
  const uint32_t nstep = nstage == 0 ? 0 : nstage + kDmaAhead;

  if (wave != 0) {
    const uint32_t lw = wave - 1;
    uint32_t g = 0, sg = 0;  // group and stage within it of the stage being loaded
    for (uint32_t i = 0; i < nstep; ++i) {
      if (i < nstage) {
        DType *slot = ring[i % kDmaSlots];
#pragma unroll
        for (int q = 0; q < kDmaPerWave; ++q) {
          const uint32_t f0 = (q * kDmaLoaders + lw) * kWave * EPD;  // first element of this instruction
          const uint32_t seg = f0 / TL, off = f0 % TL;
          uint32_t n = g * SEGS + seg;
          uint32_t e = sg * TL + off + lane * EPD;
          n = n < n_out ? n : n_out - 1;  // clamped, never consumed
          e = e < seg_len ? e : seg_len - EPD;
          const uint32_t y = div_x.Div(e);
          const size_t row = static_cast<size_t>(n * n_keep + c) * n_y + y;
          LoadDwordToLds(src + row * stride + (e - y * n_x), slot + seg * LD + off);
        }
        if (++sg == stages_per_group) {
          sg = 0;
          ++g;
        }
        WaitStageLanded<Ring>();
      } else {
        WaitAllLanded();
      }
      BareBarrier();
    }
  } else {
    DType res, tres;
    Reducer::SetInitValue(res);
    Reducer::SetInitValue(tres);
    uint32_t g = 0, sg = 0;  // of the stage being folded
    for (uint32_t i = 0; i < nstep; ++i) {
      BareBarrier();
      if (i < static_cast<uint32_t>(kDmaAhead)) continue;
      const uint32_t st = i - kDmaAhead;
      const DType *slot = ring[st % kDmaSlots];
      const uint32_t e0 = sg * TL;
      const uint32_t live = (n_out - g * SEGS < (uint32_t)SEGS) ? n_out - g * SEGS : SEGS;
      if (lane < live) {
        const int count = (seg_len - e0 < (uint32_t)TL) ? static_cast<int>(seg_len - e0) : TL;
        ChainFold<Reducer>(tres, slot + lane * LD, 0, count);
      }
      if (++sg == stages_per_group) {
        /* the group's inner results are final: merge them in n order, then restart */
        for (uint32_t k = 0; k < live; ++k) {
          const DType v = WaveBroadcast(tres, static_cast<int>(k));
          Reducer::Reduce(res, v);
        }
        Reducer::SetInitValue(tres);
        sg = 0;
        ++g;
      }
    }
    if (lane == 0) Saver::template Save<DType>(dst[c], res * scale);
  }
}

/* ------------------------------------------------------------------ KeepHighDim, split over n
 * The reference's order has two levels (mshadow/tensor_cpu-inl.h:230-268): an inner chain
 * per (n, c) segment, then a chain over n of the inner results. Only the second is tied to
 * the kept index c; the inner chains are independent of one another, so they are dealt out in
 * the order the segments lie in memory, SEGS neighbouring segments per workgroup (one chain
 * lane each), however few kept indices there are. The inner results go to a scratch array
 * `partial` of n_out * n_keep words; the workgroup that finishes last (counters in the
 * scratch memory, kSplitCounterWords words at `counter`, tell it so) folds them per kept index
 * in n order and saves the result; the counters are zero again when the launch ends. Launches that share a scratch array must not
 * overlap: the library hands one out per stream.
 *
 * A stage is one load instruction per segment: 64 lanes x 4 or 16 bytes of consecutive
 * elements, which land in LDS as they lie in memory, so a chain lane reads its operands four
 * at a time. 16-byte loads need rows of whole 16-byte packs (n_x, pitch, base); 4-byte loads
 * of 16-bit elements rows of whole pairs. */
template <int SEGS_, int LOADERS_, int SLOTS_, int WBYTES_>
struct SplitRing {
  static const int kSegs = SEGS_;
  static const int kLoaders = LOADERS_;
  static const int kSlots = SLOTS_;
  /*! \brief bytes a lane loads at a time: 4, or 16 where rows are whole 16-byte packs */
  static const int kLaneBytes = WBYTES_;
  static const int kAhead = SLOTS_ - 2;
  static const int kPerWave = SEGS_ / LOADERS_;
  static const int kThreads = (LOADERS_ + 1) * kWave;
  static_assert(SEGS_ % LOADERS_ == 0 && SEGS_ <= kWave, "one chain lane per segment");
  static_assert(kAhead >= 1 && kAhead * kPerWave < 64, "the wait-by-count immediate has 6 bits");
  static_assert(WBYTES_ == 4 || WBYTES_ == 16, "load width");
};
/*! \brief the configurations the library launches (measured on MI355X, sum over
 *  (64,64,112,112) / (256,16,112,112) floats: 54 / 71 us and 68 / 87 us, against 103 / 388 us
 *  with one workgroup per kept index): rows of whole 16-byte packs - 16 segments per
 *  workgroup, a kilobyte of each per stage; any rows - 32 segments, 256 bytes of each. */
typedef SplitRing<16, 8, 4, 16> HighDimSplitRingPacks;
/*! \brief ... and with more segments than 16 per CU: 32 per workgroup, one workgroup per CU
 *  (two workgroups of 16 on a CU ask for more than the CU's loads deliver: (128,64,112,112)
 *  took 105 us) */
typedef SplitRing<32, 8, 4, 16> HighDimSplitRingPacksWide;
typedef SplitRing<32, 8, 8, 4> HighDimSplitRing;

/*! \brief the counters of the split reduction: a root and kSplitLeaves leaves, each in a cache
 *  line of its own (kSplitCounterStride words apart), all zero between launches */
const int kSplitLeaves = 64;
const int kSplitCounterStride = 32;
const int kSplitCounterWords = (1 + kSplitLeaves) * kSplitCounterStride;

/*! \brief words of scratch memory a launch needs for its inner results */
inline size_t SplitPartialWords(uint32_t n_out, uint32_t n_keep) {
  return static_cast<size_t>(n_out) * n_keep;
}

template <typename Saver, typename Reducer, typename DType, typename Ring>
__global__ void __launch_bounds__(Ring::kThreads)
    ReduceKeepHighDimSplitKernel(DType *dst, const DType *src, uint32_t stride, uint32_t n_out,
                                 uint32_t n_keep, uint32_t n_y, uint32_t n_x, FastDivU32 div_x,
                                 DType scale, uint32_t *partial, uint32_t *counter) {
  const int SEGS = Ring::kSegs, kSlots = Ring::kSlots, kAhead = Ring::kAhead, kPerWave = Ring::kPerWave;
  const int EPL = Ring::kLaneBytes / sizeof(DType);  // elements per lane and load
  const int TL = kWave * EPL;          // elements of a segment per stage
  const int LD = TL + 16 / sizeof(DType);  // chain lanes read words LD elements apart: no bank conflicts
  static_assert(sizeof(DType) == 4 || sizeof(DType) == 2, "a word of scratch memory holds a result");
  __shared__ MSHADOW_ALIGNED(16) DType ring[kSlots][SEGS * LD];
  __shared__ uint32_t i_am_last;

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t nseg = n_out * n_keep;
  const uint32_t s0 = blockIdx.x * SEGS;
  const uint32_t live = (nseg - s0 < static_cast<uint32_t>(SEGS)) ? nseg - s0 : SEGS;
  const uint32_t seg_len = n_y * n_x;
  const uint32_t nstage = (seg_len + TL - 1) / TL;
  const uint32_t nstep = nstage == 0 ? 0 : nstage + kAhead;

  /* Which wave runs the chains: two workgroups share a CU where the ring is half the LDS, and
     two chain waves on one SIMD take turns (measured: 11.4 ns per add against 5.6 ns). The
     workgroups that meet on a CU differ in the lowest bit of their number or in bit 8. */
  const uint32_t chain_wave = (blockIdx.x ^ (blockIdx.x >> 8)) & 1u;
  if (wave != chain_wave) {
    const uint32_t lw = wave < chain_wave ? wave : wave - 1;
    for (uint32_t i = 0; i < nstep; ++i) {
      if (i < nstage) {
        DType *slot = ring[i % kSlots];
        uint32_t e = i * TL + lane * EPL;
        e = e < seg_len ? e : seg_len - EPL;  // clamped, never consumed
        const uint32_t y = div_x.Div(e);
        const size_t in_seg = static_cast<size_t>(y) * stride + (e - y * n_x);
#pragma unroll
        for (int q = 0; q < kPerWave; ++q) {
          const uint32_t seg = q * Ring::kLoaders + lw;
          const uint32_t sg = s0 + seg < nseg ? s0 + seg : nseg - 1;  // clamped likewise
          LoadLaneToLds<Ring::kLaneBytes>(src + static_cast<size_t>(sg) * n_y * stride + in_seg,
                                          slot + seg * LD);
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAhead * kPerWave) : "memory");
      } else {
        WaitAllLanded();
      }
      BareBarrier();
    }
  } else {
    DType tres;
    Reducer::SetInitValue(tres);
    for (uint32_t i = 0; i < nstep; ++i) {
      BareBarrier();
      if (i < static_cast<uint32_t>(kAhead)) continue;
      const uint32_t st = i - kAhead;
      const uint32_t e0 = st * TL;
      if (lane < live) {
        const int count = (seg_len - e0 < (uint32_t)TL) ? static_cast<int>(seg_len - e0) : TL;
        ChainFold<Reducer>(tres, ring[st % kSlots] + lane * LD, 0, count);
      }
    }
    if (lane < live) {
      uint32_t bits = 0;
      __builtin_memcpy(&bits, static_cast<const void *>(&tres), sizeof(DType));
      __hip_atomic_store(partial + s0 + lane, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    /* The inner results must have reached the memory side before a counter moves. They are
       written through by device-scope stores, whose completion is what the wait below waits
       for; a release fence would do, but it also writes back this L2's every dirty line,
       once per workgroup. The last workgroup reads them with device-scope loads.
       Counting is in two levels, because increments of one address are served one after the
       other (about 40 ns each, which a thousand workgroups finishing together would wait
       for): workgroup b counts on leaf b % kSplitLeaves, and whoever completes a leaf counts
       on the root; whoever completes the root is last. A completed counter is cleared by the
       workgroup that completed it. */
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0) {
      const uint32_t leaf = blockIdx.x % kSplitLeaves;
      const uint32_t in_leaf = (gridDim.x - leaf + kSplitLeaves - 1) / kSplitLeaves;
      const uint32_t leaves = gridDim.x < static_cast<uint32_t>(kSplitLeaves) ? gridDim.x : kSplitLeaves;
      uint32_t *leaf_counter = counter + (1 + leaf) * kSplitCounterStride;
      uint32_t last = 0u;
      if (__hip_atomic_fetch_add(leaf_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
          in_leaf - 1u) {
        __hip_atomic_store(leaf_counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
            leaves - 1u) {
          last = 1u;
        }
      }
      i_am_last = last;
    }
  }
  __syncthreads();
  if (i_am_last == 0u) return;
  /* The merge: dst[c] = fold over n of the inner results, in n order. The results come in by
     device-scope loads, a tile of kMergeCols kept indices x as many n as the ring's memory
     holds at a time, all of a tile's loads in flight together (one after the other they would
     cost a trip to memory each); then thread c folds its column of the tile from LDS. */
  const int kMergeCols = 256;
  static_assert(Ring::kThreads >= kMergeCols, "a thread per kept index of a tile");
  uint32_t *tile = reinterpret_cast<uint32_t *>(&ring[0][0]);
  const uint32_t tile_words = sizeof(ring) / sizeof(uint32_t);
  const uint32_t tile_n = tile_words / kMergeCols;
  for (uint32_t c0 = 0; c0 < n_keep; c0 += kMergeCols) {
    const uint32_t c = c0 + threadIdx.x;
    DType res;
    Reducer::SetInitValue(res);
    for (uint32_t n0 = 0; n0 < n_out; n0 += tile_n) {
      const uint32_t nn = (n_out - n0 < tile_n) ? n_out - n0 : tile_n;
      for (uint32_t i = threadIdx.x; i < nn * kMergeCols; i += Ring::kThreads) {
        const uint32_t cc = c0 + i % kMergeCols;
        if (cc < n_keep) {
          tile[i] = __hip_atomic_load(partial + static_cast<size_t>(n0 + i / kMergeCols) * n_keep + cc,
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      __syncthreads();
      if (threadIdx.x < static_cast<uint32_t>(kMergeCols) && c < n_keep) {
        for (uint32_t n = 0; n < nn; ++n) {
          const uint32_t bits = tile[n * kMergeCols + threadIdx.x];
          DType v;
          __builtin_memcpy(static_cast<void *>(&v), &bits, sizeof(DType));
          Reducer::Reduce(res, v);
        }
      }
      __syncthreads();
    }
    if (threadIdx.x < static_cast<uint32_t>(kMergeCols) && c < n_keep) {
      Saver::template Save<DType>(dst[c], res * scale);
    }
  }
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_REDUCE_DMA_H_
