/*
 * pool<Reducer>(half_t tensor, K, K, S, S) for windows of 2, 3 or 5 elements a side that move by one
 * or two, every window whole (mshadow/extension/spatial_pool.h:20-149 of the reference with DType =
 * half_t; other windows take the map kernel, which fetches every element of every window).
 *
 * A thread makes four adjacent outputs of up to kPoolHalfRows (S = 1) or half as many rows one below
 * the other (fewer where that leaves the chip short of waves), with the K input rows of a window in
 * registers: an input element is fetched (rows + K - 1) / rows times and in 16-byte pieces wherever it lies. The last thread of an output row
 * is moved back to end with the row (it makes some outputs a second time, with the same result).
 *
 * Two outputs share a register and an instruction. A sum is K * K packed adds in the window's order,
 * each rounded as half_t's += does. For maximum and minimum any order of the elements gives the same
 * number, so rows are combined first; `if (dst < src) dst = src` differs from that only in which zero
 * it keeps and in ignoring NaN, so a thread that meets a negative zero or a NaN goes on with the
 * reducer itself, window by window.
 *
 * Bound by memory with a step of two, by its loads and stores of half a cache line with a step of
 * one. Maximum on (128,64,112,112), before (map kernel) and now: 3x3 step 2 192 -> 48 us (5.3 TB/s),
 * 2x2 step 2 102 -> 45 us, 3x3 step 1 499 -> 98 us (4.1 TB/s), 5x5 step 1 1612 -> 97 us; (64,96,55,55)
 * 3x3 step 2 34 -> 11 us; (168,298,10,16) 5x5 step 1 83 -> 7 us.
 */
#ifndef MSHADOW_HIP_KERNELS_POOL_HALF_H_
#define MSHADOW_HIP_KERNELS_POOL_HALF_H_

#include "../../core/fastdiv.h"
#include "../../half.h"
#include "./common.h"

namespace mshadow {
namespace hip {

const int kPoolHalfBlock = 256;
const int kPoolHalfRows = 8;

/*! \brief one packed step of a reduction, and whether it may take elements in any order */
template <typename Reducer>
struct PoolHalfOp;  // sum, maximum, minimum
template <>
struct PoolHalfOp<red::sum> {
  static const bool kAnyOrder = false;
  static __device__ __forceinline__ uint32_t Do(uint32_t a, uint32_t b) {
    typedef _Float16 Pair __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(Pair, a) + __builtin_bit_cast(Pair, b));
  }
};
template <>
struct PoolHalfOp<red::maximum> {
  static const bool kAnyOrder = true;
  static __device__ __forceinline__ uint32_t Do(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
  }
};
template <>
struct PoolHalfOp<red::minimum> {
  static const bool kAnyOrder = true;
  static __device__ __forceinline__ uint32_t Do(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
  }
};

struct PoolHalfGeom {
  uint32_t h, w, ph, pw;
  uint32_t rows;                   //!< rows of outputs to a strip
  uint32_t groups, strips, total;  //!< threads to a row, strips of rows to a plane, threads in all
  FastDivU32 div_groups, div_strips;
};

/*! \brief N halves from a 2-byte aligned address into words; a half that fills no word stands in
 *  the low part of one */
template <int N>
__device__ __forceinline__ void LoadHalves(uint32_t (&w)[(N + 1) / 2], const uint16_t *p) {
  typedef uint32_t W4 __attribute__((ext_vector_type(4)));
  typedef uint32_t W2 __attribute__((ext_vector_type(2)));
  typedef W4 Loose4 __attribute__((aligned(2)));
  typedef W2 Loose2 __attribute__((aligned(2)));
  typedef uint32_t Loose1 __attribute__((aligned(2)));
  int at = 0;
  if (N >= 8) {
    const W4 q = *reinterpret_cast<const Loose4 *>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = q[i];
    at = 4;
  }
  if (N % 8 >= 4) {
    const W2 q = *reinterpret_cast<const Loose2 *>(p + 2 * at);
    w[at] = q[0];
    w[at + 1] = q[1];
    at += 2;
  }
  if (N % 4 >= 2) {
    w[at] = *reinterpret_cast<const Loose1 *>(p + 2 * at);
    at += 1;
  }
  if (N % 2 != 0) w[at] = p[2 * at];
}
/*! \brief halves I and I + STEP of a row of words as one word */
template <int I, int STEP, int WORDS>
__device__ __forceinline__ uint32_t PairOf(const uint32_t (&w)[WORDS]) {
  const int J = I + STEP;
  if (STEP == 1 && I % 2 == 0) return w[I / 2];
  const uint32_t lo = I % 2 == 0 ? w[I / 2] & 0xffffu : w[I / 2] >> 16;
  const uint32_t hi = J % 2 == 0 ? w[J / 2] << 16 : w[J / 2] & 0xffff0000u;
  return lo | hi;
}

/*! \brief res (two outputs, of which the left one's window begins at half FIRST) reduced with the K
 *  elements of a row, in order */
template <typename Op, int FIRST, int K, int S, int X, int WORDS>
struct PoolHalfRow {
  static __device__ __forceinline__ void Run(uint32_t *res, const uint32_t (&w)[WORDS]) {
    *res = Op::Do(*res, PairOf<FIRST + X, S>(w));
    PoolHalfRow<Op, FIRST, K, S, X + 1, WORDS>::Run(res, w);
  }
};
template <typename Op, int FIRST, int K, int S, int WORDS>
struct PoolHalfRow<Op, FIRST, K, S, K, WORDS> {
  static __device__ __forceinline__ void Run(uint32_t *, const uint32_t (&)[WORDS]) {}
};

template <typename Reducer, int K, int S>
__global__ void __launch_bounds__(kPoolHalfBlock)
    PoolHalfKernel(half::half_t *dst, uint32_t dstride, const half::half_t *src, uint32_t sstride,
                   PoolHalfGeom g) {
  typedef PoolHalfOp<Reducer> Op;
  const int N = 3 * S + K, WORDS = (N + 1) / 2, ROWS = kPoolHalfRows / S;
  const uint32_t idx = blockIdx.x * kPoolHalfBlock + threadIdx.x;
  if (idx >= g.total) return;
  const uint32_t strip = g.div_groups.Div(idx);
  const uint32_t plane = g.div_strips.Div(strip);
  const uint32_t py0 = (strip - plane * g.strips) * g.rows;
  const uint32_t nrows = g.rows < g.ph - py0 ? g.rows : g.ph - py0;
  const uint32_t group = idx - strip * g.groups;
  const uint32_t px0 = group * 4 + 4 <= g.pw ? group * 4 : g.pw - 4;
  const uint16_t *in = reinterpret_cast<const uint16_t *>(src) + static_cast<size_t>(plane) * g.h * sstride + px0 * S;
  uint16_t *out = reinterpret_cast<uint16_t *>(dst) + (static_cast<size_t>(plane) * g.ph + py0) * dstride + px0;
  half::half_t start;
  Reducer::SetInitValue(start);
  const uint32_t init = start.half_ * 0x10001u;

  uint32_t ring[K][WORDS];  // row y of the plane in ring row y % K of the unrolled loop
  uint32_t most = 0u, top = 0x80008000u, least = 0x7fff7fffu;  // of all halves: unsigned, signed, signed
#define MSHADOW_POOL_ROW(SLOT, Y)                                                               \
  {                                                                                             \
    const uint32_t y = (Y) < g.h ? (Y) : g.h - 1u; /* behind the last output: never used */     \
    LoadHalves<N>(ring[SLOT], in + static_cast<size_t>(y) * sstride);                           \
    if (Op::kAnyOrder) {                                                                        \
      _Pragma("unroll") for (int i = 0; i < WORDS; ++i) {                                       \
        asm("v_pk_max_u16 %0, %0, %1" : "+v"(most) : "v"(ring[SLOT][i]));                       \
        asm("v_pk_max_i16 %0, %0, %1" : "+v"(top) : "v"(ring[SLOT][i]));                        \
        asm("v_pk_min_i16 %0, %0, %1" : "+v"(least) : "v"(ring[SLOT][i]));                      \
      }                                                                                         \
    }                                                                                           \
  }
#pragma unroll
  for (int k = 0; k < K - S; ++k) MSHADOW_POOL_ROW(k, py0 * S + k)
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if (static_cast<uint32_t>(r) >= nrows) break;
#pragma unroll
    for (int k = K - S; k < K; ++k) MSHADOW_POOL_ROW((r * S + k) % K, (py0 + r) * S + k)
    uint32_t left = init, right = init;
    bool plain = true;
    if (Op::kAnyOrder) {
      /* no negative zero (the least signed number), no NaN (above infinity with either sign) */
      plain = (least & 0xffffu) != 0x8000u && (least >> 16) != 0x8000u &&
              (most & 0xffffu) <= 0xfc00u && (most >> 16) <= 0xfc00u &&
              static_cast<int16_t>(top & 0xffffu) <= 0x7c00 && static_cast<int16_t>(top >> 16) <= 0x7c00;
      uint32_t rows[WORDS];
#pragma unroll
      for (int i = 0; i < WORDS; ++i) {
        rows[i] = ring[0][i];
#pragma unroll
        for (int k = 1; k < K; ++k) rows[i] = Op::Do(rows[i], ring[k][i]);
      }
      PoolHalfRow<Op, 0, K, S, 0, WORDS>::Run(&left, rows);
      PoolHalfRow<Op, 2 * S, K, S, 0, WORDS>::Run(&right, rows);
    } else {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        PoolHalfRow<Op, 0, K, S, 0, WORDS>::Run(&left, ring[(r * S + k) % K]);
        PoolHalfRow<Op, 2 * S, K, S, 0, WORDS>::Run(&right, ring[(r * S + k) % K]);
      }
    }
    if (!plain) {
      uint32_t four[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        half::half_t res = start;
        for (uint32_t k = 0; k < static_cast<uint32_t>(K); ++k) {
          const uint16_t *row = in + static_cast<size_t>((py0 + r) * S + k) * sstride + e * S;
          for (int x = 0; x < K; ++x) Reducer::Reduce(res, half::half_t::Binary(row[x]));
        }
        four[e] = res.half_;
      }
      left = four[0] | (four[1] << 16);
      right = four[2] | (four[3] << 16);
    }
    typedef uint32_t W2 __attribute__((ext_vector_type(2)));
    typedef W2 Loose2 __attribute__((aligned(2)));
    *reinterpret_cast<Loose2 *>(out + static_cast<size_t>(r) * dstride) = W2{left, right};
  }
#undef MSHADOW_POOL_ROW
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_POOL_HALF_H_
