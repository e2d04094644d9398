/*
 * sumall_except_dim<1> and its kin over dense planes, a wave to itself with eight or sixteen of them.
 *
 * The order is that of the other kernels (one chain per (n, c) plane, then one over n of their results:
 * mshadow/tensor_cpu-inl.h:230-268). A workgroup owns a few neighbouring kept indices c with all their
 * planes, a wave LANES planes, a lane the chain of one. The wave fetches 16 bytes a lane, PACKS lanes
 * next to one another in a plane, two slices ahead in registers, and passes each slice through its own
 * piece of LDS to the lanes that add; waves meet only once, for the chains over n. No ring that fills a
 * CU, no scratch memory, and every wave adds, where the kernels of reduce_dma.h have one that does.
 */
#ifndef MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_
#define MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_

#include "../../core/fastdiv.h"
#include "./common.h"
#include "./reduce.h"
#include "./segments_plan.h"

namespace mshadow {
namespace hip {

template <typename DType, int LANES>
struct SegSlice {
  static const int kPerPack = 16 / sizeof(DType);
  static const int kPacks = 256 / LANES;               //!< packs of a plane in a slice: four a lane in all
  static const int kElems = kPacks * kPerPack;         //!< elements of a plane in a slice
  static const int kPitch = kElems + kPerPack;         //!< no bank conflicts; the place in front of a plane is free
  static const int kWaveElems = kPerPack + LANES * kPitch;
  /*! \brief dynamic LDS of a workgroup of `waves` waves with `planes` planes */
  static size_t LdsBytes(uint32_t waves, uint32_t planes) { return (waves * kWaveElems + planes) * sizeof(DType); }
};

/*! \brief what may be reduced in the place of a value behind the end of a plane: kPadNegZero, which no sum notices
 *  (x + -0 is x for every x), kPadItself, the result so far, or, of a reducer that is not known, nothing. The last
 *  values of a plane are then read a few packs at a time; one by one each waited for LDS. */
enum SegmentPad { kPadNothing, kPadNegZero, kPadItself };
template <typename Reducer>
struct PadOf {
  static const SegmentPad value = kPadNothing;
};
template <>
struct PadOf<red::sum> {
  static const SegmentPad value = kPadNegZero;
};
template <>
struct PadOf<red::maximum> {
  static const SegmentPad value = kPadItself;
};
template <>
struct PadOf<red::minimum> {
  static const SegmentPad value = kPadItself;
};

template <typename Saver, typename Reducer, typename DType, int LANES>
__global__ void __launch_bounds__(kSegMostWaves * kWave)
    ReduceSegmentsKernel(DType *dst, const DType *src, uint32_t seg_len, uint32_t n_out, uint32_t n_keep, uint32_t kept,
                         FastDivU32 div_kept, DType scale) {
  typedef SegSlice<DType, LANES> Slice;
  static_assert(LANES == 8 || LANES == 16, "a slice is 16 or 32 packs of a plane");
  const int EPP = Slice::kPerPack, PACKS = Slice::kPacks, ELEMS = Slice::kElems, AHEAD = 2;
  const SegmentPad kPad = PadOf<Reducer>::value;
  typedef uint32_t Pack __attribute__((ext_vector_type(4)));
  typedef Pack LoosePack __attribute__((aligned(2)));  // wherever a plane begins
  extern __shared__ __attribute__((aligned(16))) unsigned char segment_lds[];
  const uint32_t waves = blockDim.x / kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
  DType *tile = reinterpret_cast<DType *>(segment_lds) + wave * Slice::kWaveElems + EPP;
  DType *part = reinterpret_cast<DType *>(segment_lds) + waves * Slice::kWaveElems;
  const uint32_t c0 = blockIdx.x * kept, planes = kept * n_out;
  const uint32_t pack = lane % PACKS;
  const uint32_t slices = (seg_len + ELEMS - 1) / ELEMS;
  for (uint32_t p0 = wave * LANES; p0 < planes; p0 += waves * LANES) {
    /* the planes that this lane fetches pack `lane % PACKS` of a slice of; one that is not there is another one again */
    uint32_t from[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t p = p0 + (q * kWave + lane) / PACKS;
      p = p < planes ? p : planes - 1;
      const uint32_t n = div_kept.Div(p), c = c0 + (p - n * kept);
      from[q] = n * n_keep + (c < n_keep ? c : n_keep - 1);
    }
    Pack v[AHEAD][4];
    /* ordinary, not streaming, loads: the next slice has the rest of a cache line ((248,552,7,40) 43 -> 41 us) */
    auto fetch = [&](Pack (&to)[4], uint32_t slice) {
      const uint32_t e = slice * ELEMS + pack * EPP;
      const uint32_t at = e + EPP <= seg_len ? e : seg_len - EPP;  // the plane's end: its last pack
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        to[q] = *reinterpret_cast<const LoosePack *>(src + static_cast<size_t>(from[q]) * seg_len + at);
      }
    };
    DType res;
    Reducer::SetInitValue(res);
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      if (a < static_cast<int>(slices)) fetch(v[a], a);
    }
    for (uint32_t s0 = 0; s0 < slices; s0 += AHEAD) {
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        const uint32_t s = s0 + a;
        if (s >= slices) break;
        const uint32_t left = seg_len - s * ELEMS;
        const bool whole = left >= static_cast<uint32_t>(ELEMS);
        if (whole) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            *reinterpret_cast<Pack *>(tile + ((q * kWave + lane) / PACKS) * Slice::kPitch + pack * EPP) = v[a][q];
          }
        } else {  // the last pack of a plane ends with it, wherever that is (behind it again and again)
          const int at = static_cast<int>(pack * EPP) + EPP <= static_cast<int>(left) ? static_cast<int>(pack * EPP)
                                                                                       : static_cast<int>(left) - EPP;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            DType *to = tile + ((q * kWave + lane) / PACKS) * Slice::kPitch + at;
            DType e[EPP];
            __builtin_memcpy(static_cast<void *>(e), &v[a][q], sizeof(Pack));
#pragma unroll
            for (int i = 0; i < EPP; ++i) to[i] = e[i];
          }
        }
        if (s + AHEAD < slices) fetch(v[a], s + AHEAD);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the lanes' stores before one another's loads
        if (lane < static_cast<uint32_t>(LANES)) {
          const DType *mine = tile + lane * Slice::kPitch;
          if (whole) {
            const int GROUP = 8;
#pragma unroll
            for (int p = 0; p < PACKS; p += GROUP) {
              Pack e[GROUP];
#pragma unroll
              for (int k = 0; k < GROUP; ++k) e[k] = *reinterpret_cast<const Pack *>(mine + (p + k) * EPP);
              DType w[GROUP * EPP];
              __builtin_memcpy(static_cast<void *>(w), e, sizeof(w));
#pragma unroll
              for (int i = 0; i < GROUP * EPP; ++i) Reducer::Reduce(res, w[i]);
            }
          } else if (kPad != kPadNothing && sizeof(DType) == 4) {
            const int END = 2;
            for (uint32_t i = 0; i < left; i += END * EPP) {
              Pack e[END];
#pragma unroll
              for (int k = 0; k < END; ++k) e[k] = *reinterpret_cast<const Pack *>(mine + i + k * EPP);
              DType w[END * EPP];
              __builtin_memcpy(static_cast<void *>(w), e, sizeof(w));
#pragma unroll
              for (int k = 0; k < END * EPP; ++k) {
                const DType none = kPad == kPadNegZero ? -DType(0.0f) : res;
                Reducer::Reduce(res, i + k < left ? w[k] : none);
              }
            }
          } else {
            /* halves: whole packs, then one by one. Selecting 32 of them costs more than it saves ((7,1488,690) 11.2 and
               17 us), -0 stored behind a plane's end the registers of a wave ((22,1625,640) 12 and 14 us). */
            uint32_t i = 0;
            for (; i + EPP <= left; i += EPP) {
              const Pack e = *reinterpret_cast<const Pack *>(mine + i);
              DType w[EPP];
              __builtin_memcpy(static_cast<void *>(w), &e, sizeof(w));
#pragma unroll
              for (int k = 0; k < EPP; ++k) Reducer::Reduce(res, w[k]);
            }
            for (; i < left; ++i) Reducer::Reduce(res, mine[i]);
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    if (lane < static_cast<uint32_t>(LANES) && p0 + lane < planes) part[p0 + lane] = res;
  }
  __syncthreads();
  const uint32_t c = c0 + threadIdx.x;
  if (threadIdx.x < kept && c < n_keep) {
    DType sum;
    Reducer::SetInitValue(sum);
#pragma unroll 8
    for (uint32_t n = 0; n < n_out; ++n) Reducer::Reduce(sum, part[n * kept + threadIdx.x]);
    Saver::template Save<DType>(dst[c], sum * scale);
  }
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_
