/*
 * Softmax / SoftmaxGrad for element types other than float (half_t, double), written in the
 * element type's own arithmetic so that every intermediate rounds where the CPU path rounds
 * (mshadow/tensor_cpu-inl.h:270-302): the difference x - max, the exponential stored into
 * dst, the running sum after every add and the final quotient are all values of DType.
 * For half_t that matters: a sum kept in 16 bits stops growing once its ulp exceeds twice the
 * terms (4096 equal logits give 1/2048 each, not 1/4096), and only the left-to-right order
 * reproduces it.
 *
 * A workgroup of 256 threads takes kAnyRows = 8 rows, 32 threads per row, each thread four
 * packs of kAnyTile = 8 consecutive elements per step (128-bit accesses for half_t when rows are
 * aligned whole packs; a row is visited in contiguous stretches of 1024 elements). The maximum
 * is a reduction over the row's 32 threads (exact in any order). The rows then pass in tiles
 * of 1024 columns: every thread computes its packs of terms (the next tile's logits are
 * already on their way), stores them to dst and parks them in LDS; eight lanes of one wave
 * then each add one row's 1024 terms to that row's running sum, term by term, four packs
 * being added while the next four come from LDS, and while the other waves make the next
 * tile in the second LDS buffer. A wave instruction costs the same for one active lane as
 * for sixty-four, so the chains of the eight rows share their instructions (one wave per
 * row: 1457 us for 8192 x 32000 half_t; this kernel: 670 us, of which the five passes over
 * memory - logits twice, terms written, read back and written again - would take about 440
 * at the rate of a plain copy; four or sixteen rows per workgroup were slower, as was making
 * the terms a second time from the logits instead of storing them and reading them back).
 * A last pass divides the stored terms. A thread only ever reads back and writes the
 * elements it handled itself, so in-place calls (dst == src) are safe.
 *
 * The float versions are the fixed-function kernels of the library (csrc/softmax_kernels.h).
 */
#ifndef MSHADOW_HIP_KERNELS_SOFTMAX_ANY_H_
#define MSHADOW_HIP_KERNELS_SOFTMAX_ANY_H_

#include "../../core/fastdiv.h"
#include "../../half.h"
#include "./common.h"

namespace mshadow {
namespace hip {

const int kAnyBlock = 256;
/*! \brief rows per workgroup */
const int kAnyRows = 8;
/*! \brief consecutive elements of one thread per step */
const int kAnyTile = 8;
const int kAnyThreadsPerRow = kAnyBlock / kAnyRows;
/*! \brief packs of one thread per step: a row is visited in stretches of
 *  kAnyBatch * kAnyThreadsPerRow packs (2 KB of half_t), pack q of thread p being pack
 *  q * kAnyThreadsPerRow + p of the stretch, so that a wave's accesses stay contiguous */
const int kAnyBatch = 4;
const int kAnyStepCols = kAnyThreadsPerRow * kAnyTile;
const int kAnyTileCols = kAnyBatch * kAnyStepCols;
/*! \brief row pitch of the LDS tile: one pack more than it holds, so that the eight chain
 *  lanes read from different banks */
const int kAnyPitch = kAnyTileCols + kAnyTile;

template <typename DType>
struct alignas(16) AnyPack {
  DType v[kAnyTile];
};

/*! \brief what std::exp(DType) resolves to on the host: the float function for half_t
 *  (through its conversion to float) and float, the double function for double */
__device__ __forceinline__ float SoftmaxExp(half::half_t v) { return expf(static_cast<float>(v)); }
__device__ __forceinline__ float SoftmaxExp(float v) { return expf(v); }
__device__ __forceinline__ double SoftmaxExp(double v) { return exp(v); }

/*! \brief the type comparisons of DType are made in (exact widening) */
template <typename DType>
struct WideOf { typedef float Type; };
template <>
struct WideOf<double> { typedef double Type; };

/*! \brief static_cast<int>(label) as the host makes it: half_t goes through float */
__device__ __forceinline__ int LabelIndex(half::half_t v) { return static_cast<int>(static_cast<float>(v)); }
__device__ __forceinline__ int LabelIndex(float v) { return static_cast<int>(v); }
__device__ __forceinline__ int LabelIndex(double v) { return static_cast<int>(v); }

__device__ __forceinline__ float WaveShuffleXor(float v, int mask) { return __shfl_xor(v, mask); }
__device__ __forceinline__ double WaveShuffleXor(double v, int mask) { return __shfl_xor(v, mask); }

/*! \brief sum += t as DType does it. For half_t one 16-bit add: it rounds the exact sum once,
 *  which equals widening, adding in float and rounding back (24 >= 2 * 11 + 2 bits), and is a
 *  third of the dependent instructions. */
template <typename DType>
__device__ __forceinline__ void ChainAdd(DType &sum, const DType &t) { sum += t; }
__device__ __forceinline__ void ChainAdd(half::half_t &sum, const half::half_t &t) {
  const _Float16 a = __builtin_bit_cast(_Float16, sum.half_);
  const _Float16 b = __builtin_bit_cast(_Float16, t.half_);
  sum.half_ = __builtin_bit_cast(uint16_t, static_cast<_Float16>(a + b));
}

/*! \brief sixteen bytes at an address aligned only to a 16-bit element, which costs no more than the
 *  cache lines it touches */
typedef uint32_t AnyWords __attribute__((ext_vector_type(4)));
typedef AnyWords AnyLooseWords __attribute__((aligned(2)));
/*! \brief the pack moved down by `by` < 8 halves; what moves in is one of its halves */
__device__ __forceinline__ void MoveHalvesDown(AnyWords *w, uint32_t by) {
  AnyWords v = *w;
  if ((by & 4u) != 0u) v[0] = v[2], v[1] = v[3];
  if ((by & 2u) != 0u) v[0] = v[1], v[1] = v[2], v[2] = v[3];
  if ((by & 1u) != 0u) {
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = (v[k] >> 16) | (v[k + 1] << 16);
    v[3] >>= 16;
    v[3] |= v[3] << 16;
  }
  *w = v;
}
/*! \brief how a kernel moves a row: element by element (short code for short rows), as packs at any
 *  alignment, as whole aligned packs (cols % kAnyTile == 0 and every row starts 16-byte aligned) */
const int kAnyApart = 0, kAnyLoose = 1, kAnyWhole = 2;
/*! \brief elements [x, x + kAnyTile) of a row; what lies past the end of the row is `absent` or
 *  any of the row's elements. A row's last pack that is no whole one is taken element by element, of 16-bit elements as the row's last eight, moved down: one load whichever lane
 *  has it. Of 131072 x 127 half_t the Softmax took 115 us with every pack of such rows taken apart, 4096 x
 *  50257 the gradient 408 us; with whole packs and single elements side by side in a wave the Softmax
 *  takes 95 us there and 6.0 us of 200 x 10, now 90 and 5.85 (5.6 with every pack taken apart). */
template <typename DType, int HOW>
__device__ __forceinline__ void LoadAnyPack(AnyPack<DType> *p, const DType *row, uint32_t x,
                                            uint32_t cols, DType absent) {
  if (HOW == kAnyWhole) {
    *p = *reinterpret_cast<const AnyPack<DType> *>(row + x);
  } else if (HOW == kAnyLoose &&
             (x + kAnyTile <= cols || (sizeof(DType) == 2 && cols >= static_cast<uint32_t>(kAnyTile)))) {
    const uint32_t past = sizeof(DType) == 2 && x + kAnyTile > cols ? x + kAnyTile - cols : 0u;
    AnyWords w[sizeof(AnyPack<DType>) / sizeof(AnyWords)];
#pragma unroll
    for (unsigned i = 0; i < sizeof(w) / sizeof(w[0]); ++i) {
      w[i] = reinterpret_cast<const AnyLooseWords *>(row + x - past)[i];
    }
    if (sizeof(DType) == 2 && past != 0u) MoveHalvesDown(&w[0], past);
    __builtin_memcpy(static_cast<void *>(p), w, sizeof(w));
  } else {
#pragma unroll
    for (int i = 0; i < kAnyTile; ++i) p->v[i] = (x + i < cols) ? row[x + i] : absent;
  }
}
template <typename DType, int HOW>
__device__ __forceinline__ void StoreAnyPack(DType *row, uint32_t x, uint32_t cols,
                                             const AnyPack<DType> &p) {
  if (HOW == kAnyWhole) {
    *reinterpret_cast<AnyPack<DType> *>(row + x) = p;
  } else if (HOW == kAnyLoose && x + kAnyTile <= cols) {
    AnyWords w[sizeof(AnyPack<DType>) / sizeof(AnyWords)];
    __builtin_memcpy(w, &p, sizeof(w));
#pragma unroll
    for (unsigned i = 0; i < sizeof(w) / sizeof(w[0]); ++i) {
      reinterpret_cast<AnyLooseWords *>(row + x)[i] = w[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kAnyTile; ++i) {
      if (x + i < cols) row[x + i] = p.v[i];
    }
  }
}

template <typename DType, int HOW>
__global__ void __launch_bounds__(kAnyBlock)
    SoftmaxAnyKernel(DType *dst, uint32_t dstride, const DType *src, uint32_t sstride,
                     uint32_t rows, uint32_t cols) {
  typedef typename WideOf<DType>::Type Wide;
  __shared__ AnyPack<DType> tile_packs[2][kAnyRows][kAnyPitch / kAnyTile];
  __shared__ DType sums[kAnyRows];
  const uint32_t r = threadIdx.x / kAnyThreadsPerRow;
  const uint32_t p = threadIdx.x % kAnyThreadsPerRow;
  const uint32_t row = blockIdx.x * kAnyRows + r;
  /* threads without a row run along (the barriers are the workgroup's) and touch nothing */
  const bool live = row < rows;
  const DType *e = src + static_cast<size_t>(live ? row : 0) * sstride;
  DType *o = dst + static_cast<size_t>(live ? row : 0) * dstride;

  /* maximum: `if (mmax < e[x]) mmax = e[x]` from e[0] on, which is the largest value */
  const DType first = e[0];
  Wide m = static_cast<Wide>(first);
  if (live) {
    for (uint32_t x0 = 0; x0 < cols; x0 += kAnyTileCols) {
      AnyPack<DType> in[kAnyBatch];
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
        const uint32_t x = x0 + (q * kAnyThreadsPerRow + p) * kAnyTile;
        if (x < cols) {
          LoadAnyPack<DType, HOW>(&in[q], e, x, cols, first);
        } else {
#pragma unroll
          for (int i = 0; i < kAnyTile; ++i) in[q].v[i] = first;
        }
      }
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
#pragma unroll
        for (int i = 0; i < kAnyTile; ++i) {
          const Wide v = static_cast<Wide>(in[q].v[i]);
          m = (m < v) ? v : m;
        }
      }
    }
  }
#pragma unroll
  for (int d = 1; d < kAnyThreadsPerRow; d <<= 1) {  // the row's 32 threads are half a wave
    const Wide other = WaveShuffleXor(m, d);
    m = (m < other) ? other : m;
  }
  const DType mmax = static_cast<DType>(m);  // exact: m is one of the row's values

  /* chain lane c (lane c < kAnyRows of one wave) owns the running sum of row c. Which wave
     does it rotates with the workgroup number, so that the chains of the workgroups sharing
     a CU sit on different SIMDs */
  const uint32_t chain_wave = blockIdx.x % (kAnyBlock / kWave);
  const uint32_t c = threadIdx.x & (kWave - 1);
  const bool chain_slot = (threadIdx.x >> 6) == chain_wave && c < static_cast<uint32_t>(kAnyRows);
  const bool chain_lane = chain_slot && blockIdx.x * kAnyRows + c < rows;
  DType sum = DType(0.0f);
  /* the packs of the next tile are fetched before this tile's terms are computed and summed */
  AnyPack<DType> in[kAnyBatch];
#pragma unroll
  for (int q = 0; q < kAnyBatch; ++q) {
    const uint32_t x = (q * kAnyThreadsPerRow + p) * kAnyTile;
    if (live && x < cols) LoadAnyPack<DType, HOW>(&in[q], e, x, cols, mmax);
  }
  /* Tile i's terms are added while tile i + 1 is being made: in step i every thread makes its
     packs of tile i (LDS buffer i & 1), then the chain lanes add tile i - 1 from the other
     buffer, then all meet. One step more than there are tiles adds the last one. A buffer is
     written again two steps after it was written, one barrier after it was last read. */
  const uint32_t ntiles = (cols + kAnyTileCols - 1) / kAnyTileCols;
  for (uint32_t step = 0; step <= ntiles; ++step) {
    const uint32_t x0 = step * kAnyTileCols;
    if (step < ntiles) {
      AnyPack<DType> next[kAnyBatch];
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
        const uint32_t x = x0 + kAnyTileCols + (q * kAnyThreadsPerRow + p) * kAnyTile;
        if (live && x < cols) LoadAnyPack<DType, HOW>(&next[q], e, x, cols, mmax);
      }
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
        const uint32_t x = x0 + (q * kAnyThreadsPerRow + p) * kAnyTile;
        if (live && x < cols) {
          AnyPack<DType> t;
#pragma unroll
          for (int i = 0; i < kAnyTile; ++i) t.v[i] = DType(SoftmaxExp(in[q].v[i] - mmax));
          StoreAnyPack<DType, HOW>(o, x, cols, t);
          tile_packs[step & 1u][r][q * kAnyThreadsPerRow + p] = t;
        }
      }
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) in[q] = next[q];
    }
    if (chain_lane && step > 0) {
      const uint32_t done = x0 - kAnyTileCols;  // first column of the tile being added
      const uint32_t n = cols - done < static_cast<uint32_t>(kAnyTileCols) ? cols - done : kAnyTileCols;
      const AnyPack<DType> *mine = tile_packs[(step - 1u) & 1u][c];
      const uint32_t full = n / kAnyTile;  // whole packs
      uint32_t k = 0;
      if (full >= 4) {
        /* four packs are added while the next four are on their way from LDS */
        AnyPack<DType> a[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = mine[q];
        for (; k + 8 <= full; k += 4) {
          AnyPack<DType> b[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) b[q] = mine[k + 4 + q];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int i = 0; i < kAnyTile; ++i) ChainAdd(sum, a[q].v[i]);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) a[q] = b[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int i = 0; i < kAnyTile; ++i) ChainAdd(sum, a[q].v[i]);
        }
        k += 4;
      }
      for (; k < full; ++k) {
        const AnyPack<DType> t = mine[k];
#pragma unroll
        for (int i = 0; i < kAnyTile; ++i) ChainAdd(sum, t.v[i]);
      }
      if (k * kAnyTile < n) {
        const AnyPack<DType> t = mine[k];
#pragma unroll
        for (int i = 0; i < kAnyTile; ++i) {  // unrolled: a run-time index would put t in scratch memory
          if (k * kAnyTile + i < n) ChainAdd(sum, t.v[i]);
        }
      }
    }
    __syncthreads();
  }
  if (chain_slot) sums[c] = sum;
  __syncthreads();
  sum = sums[r];

  /* every thread reads back only what it stored itself */
  if (live) {
    for (uint32_t x0 = 0; x0 < cols; x0 += kAnyTileCols) {
      AnyPack<DType> t[kAnyBatch];
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
        const uint32_t x = x0 + (q * kAnyThreadsPerRow + p) * kAnyTile;
        if (x < cols) LoadAnyPack<DType, HOW>(&t[q], o, x, cols, sum);
      }
#pragma unroll
      for (int q = 0; q < kAnyBatch; ++q) {
        const uint32_t x = x0 + (q * kAnyThreadsPerRow + p) * kAnyTile;
        if (x < cols) {
#pragma unroll
          for (int i = 0; i < kAnyTile; ++i) t[q].v[i] /= sum;
          StoreAnyPack<DType, HOW>(o, x, cols, t[q]);
        }
      }
    }
  }
}

/*! \brief which gradient: bit 0 label smoothing, bit 1 an ignored label (the values of
 *  MSHADOW_HIP_GRAD_SMOOTH / MSHADOW_HIP_GRAD_IGNORE) */
const int kAnyGradSmooth = 1;
const int kAnyGradIgnore = 2;

/*! \brief one element of SoftmaxGrad / SmoothSoftmaxGrad (mshadow/tensor_cpu-inl.h:286-455)
 *  with the host's expressions in the host's types: `p - 1.0f + alpha` and `p - smooth`
 *  round after every operation for half_t (its operators return half_t), are double
 *  arithmetic for double, and `smooth` = alpha / (classes - 1) is a float for every type */
template <typename DType, int FLAGS>
__device__ __forceinline__ DType GradElement(const DType &p, bool at_label, bool ignored,
                                             float alpha, float smooth) {
  if ((FLAGS & kAnyGradIgnore) && ignored) return DType(0.0f);
  if (FLAGS & kAnyGradSmooth) {
    if (at_label) return DType(p - 1.0f + alpha);
    return DType(p - smooth);
  }
  if (at_label) return DType(p - 1.0f);
  return p;
}

/*! \brief a pack of the gradient FLAGS selects for probabilities src and the row's label k; a label
 *  outside the row marks no column */
template <typename DType, int FLAGS>
__device__ __forceinline__ void GradPack(DType *o, const DType *s, uint32_t x, uint32_t cols, int k,
                                         int ignore_k, float alpha, float smooth) {
  AnyPack<DType> v;
  LoadAnyPack<DType, kAnyLoose>(&v, s, x, cols, DType(0.0f));
  const bool ignored = (FLAGS & kAnyGradIgnore) && k == ignore_k;
  const uint32_t off = static_cast<uint32_t>(k) - x;  // wraps for k < x
  const bool label_here = k >= 0 && off < static_cast<uint32_t>(kAnyTile);
  if (FLAGS != 0 || label_here) {
#pragma unroll
    for (int i = 0; i < kAnyTile; ++i) {
      v.v[i] = GradElement<DType, FLAGS>(v.v[i], label_here && static_cast<uint32_t>(i) == off,
                                         ignored, alpha, smooth);
    }
  }
  StoreAnyPack<DType, kAnyLoose>(o, x, cols, v);
}
/*! \brief blockIdx.x = row, blockIdx.y = stretch of columns; a thread moves packs of kAnyTile */
template <typename DType, int FLAGS>
__global__ void __launch_bounds__(kAnyBlock)
    SoftmaxGradAnyKernel(DType *dst, uint32_t dstride, const DType *src, uint32_t sstride,
                         const DType *label, uint32_t cols, int ignore_k, float alpha,
                         float smooth) {
  const uint32_t row = blockIdx.x;
  const int k = LabelIndex(label[row]);
  const DType *s = src + static_cast<size_t>(row) * sstride;
  DType *o = dst + static_cast<size_t>(row) * dstride;
  const uint32_t step = gridDim.y * kAnyBlock * kAnyTile;
  for (uint32_t x = (blockIdx.y * kAnyBlock + threadIdx.x) * kAnyTile; x < cols; x += step) {
    GradPack<DType, FLAGS>(o, s, x, cols, k, ignore_k, alpha, smooth);
  }
}
/*! \brief the same for rows of up to kAnyGradShort columns, where a workgroup per row leaves most of
 *  its threads idle: a workgroup takes kAnyBlock / packs consecutive rows of `packs` = ceil(cols /
 *  kAnyTile) packs each (`div_packs` divides by it), a thread one pack */
const uint32_t kAnyGradShort = 1024;
template <typename DType, int FLAGS>
__global__ void __launch_bounds__(kAnyBlock)
    SoftmaxGradAnyShortKernel(DType *dst, uint32_t dstride, const DType *src, uint32_t sstride,
                              const DType *label, uint32_t cols, int ignore_k, float alpha, float smooth,
                              uint32_t rows, uint32_t rows_per_block, FastDivU32 div_packs) {
  const uint32_t r = div_packs.Div(threadIdx.x);
  const uint32_t row = blockIdx.x * rows_per_block + r;
  if (r >= rows_per_block || row >= rows) return;
  const uint32_t x = (threadIdx.x - r * div_packs.div) * kAnyTile;
  GradPack<DType, FLAGS>(dst + static_cast<size_t>(row) * dstride, src + static_cast<size_t>(row) * sstride,
                         x, cols, LabelIndex(label[row]), ignore_k, alpha, smooth);
}

/* ---- tensors of three dimensions (d0, d1, d2): the softmax runs over the middle one
 * (mshadow/tensor_cpu-inl.h:466-488). Element (y, x, n) is at (y * d1 + x) * stride + n. */
const int kAny3dBlock = 256;

/*! \brief one thread per (y, n), neighbouring threads neighbouring n (coalesced): the
 *  thread walks x three times, exactly as the host loop does - maximum, terms stored and
 *  summed left to right in DType, quotients. In place (dst == src) is safe: a thread reads
 *  and writes its own column only. */
template <typename DType>
__global__ void __launch_bounds__(kAny3dBlock)
    Softmax3dAnyKernel(DType *dst, uint32_t dstride, const DType *src, uint32_t sstride,
                       uint32_t d0, uint32_t d1, uint32_t d2) {
  const size_t idx = static_cast<size_t>(blockIdx.x) * kAny3dBlock + threadIdx.x;
  if (idx >= static_cast<size_t>(d0) * d2) return;
  const uint32_t y = static_cast<uint32_t>(idx / d2);
  const uint32_t n = static_cast<uint32_t>(idx - static_cast<size_t>(y) * d2);
  const DType *s = src + static_cast<size_t>(y) * d1 * sstride + n;
  DType *o = dst + static_cast<size_t>(y) * d1 * dstride + n;
  DType mmax = s[0];
  for (uint32_t x = 1; x < d1; ++x) {
    const DType e = s[static_cast<size_t>(x) * sstride];
    if (mmax < e) mmax = e;
  }
  DType sum = DType(0.0f);
  for (uint32_t x = 0; x < d1; ++x) {
    const DType t = DType(SoftmaxExp(DType(s[static_cast<size_t>(x) * sstride] - mmax)));
    o[static_cast<size_t>(x) * dstride] = t;
    ChainAdd(sum, t);
  }
  for (uint32_t x = 0; x < d1; ++x) {
    DType t = o[static_cast<size_t>(x) * dstride];
    t /= sum;
    o[static_cast<size_t>(x) * dstride] = t;
  }
}

/*! \brief one thread per element; label (y, n) at y * lstride + n */
template <typename DType, int FLAGS>
__global__ void __launch_bounds__(kAny3dBlock)
    SoftmaxGrad3dAnyKernel(DType *dst, uint32_t dstride, const DType *src, uint32_t sstride,
                           const DType *label, uint32_t lstride, uint32_t d0, uint32_t d1,
                           uint32_t d2, int ignore_k, float alpha, float smooth) {
  const size_t total = static_cast<size_t>(d0) * d1 * d2;
  for (size_t idx = static_cast<size_t>(blockIdx.x) * kAny3dBlock + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * kAny3dBlock) {
    const size_t row = idx / d2;  // y * d1 + x
    const uint32_t n = static_cast<uint32_t>(idx - row * d2);
    const uint32_t y = static_cast<uint32_t>(row / d1);
    const uint32_t x = static_cast<uint32_t>(row - static_cast<size_t>(y) * d1);
    const int k = LabelIndex(label[static_cast<size_t>(y) * lstride + n]);
    const bool ignored = (FLAGS & kAnyGradIgnore) && k == ignore_k;
    dst[row * dstride + n] = GradElement<DType, FLAGS>(src[row * sstride + n],
                                                       static_cast<int>(x) == k, ignored, alpha,
                                                       smooth);
  }
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_SOFTMAX_ANY_H_
