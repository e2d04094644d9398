/*
 * sumall_except_dim<1> and its kin over dense planes, a wave to itself with up to 64 of them.
 *
 * The order is that of the other kernels (one chain per (n, c) plane, then one over n of their results:
 * mshadow/tensor_cpu-inl.h:230-268). A workgroup owns a few neighbouring kept indices c with all their
 * planes, a wave LANES planes, a lane the chain of one. The wave fetches 16 bytes a lane, PACKS lanes
 * next to one another in a plane, three slices ahead in registers, and passes each slice through its own
 * piece of LDS to the lanes that add; waves meet only once, for the chains over n. No ring that fills a
 * CU, no scratch memory, and every wave adds, where the kernels of reduce_dma.h have one that does.
 */
#ifndef MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_
#define MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_

#include "../../core/fastdiv.h"
#include "./common.h"
#include "./reduce.h"

namespace mshadow {
namespace hip {

const uint32_t kSegMostWaves = 16;

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

template <typename Saver, typename Reducer, typename DType, int LANES>
__global__ void __launch_bounds__(kSegMostWaves * kWave)
    ReduceSegmentsKernel(DType *dst, const DType *src, uint32_t seg_len, uint32_t n_out, uint32_t n_keep, uint32_t kept,
                         FastDivU32 div_kept, DType scale) {
  typedef SegSlice<DType, LANES> Slice;
  const int EPP = Slice::kPerPack, PACKS = Slice::kPacks, ELEMS = Slice::kElems, AHEAD = 2;
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
        if (LANES == kWave || lane < static_cast<uint32_t>(LANES)) {
          const DType *mine = tile + lane * Slice::kPitch;
          if (whole) {
            const int GROUP = PACKS < 8 ? PACKS : 8;
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
          } else {
            for (uint32_t i = 0; i < left; ++i) Reducer::Reduce(res, mine[i]);
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    if ((LANES == kWave || lane < static_cast<uint32_t>(LANES)) && p0 + lane < planes) part[p0 + lane] = res;
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

/*! \brief how (n, c) planes of `len` elements are dealt out */
struct SegmentsPlan {
  bool use;        //!< false: the kernels of reduce_dma.h and reduce.h are the sooner ones
  int lanes;       //!< planes of a wave
  uint32_t kept, waves;  //!< kept indices and waves of a workgroup
};
/*! \brief Measured on (n, c, len), us, the other kernels and this one; floats, binary16 gains as much. It wants planes
 *  enough for a wave of sixteen on every SIMD or nearly, and wins by what the others leave idle.
 *  Few kept indices (workgroups that share out the planes otherwise, and merge in the last of them): short planes
 *  (200,100,400) 38 and 17, (213,58,312) 28 and 15, (60,190,1500) 30 and 21, but (160,40,2296) 27 and 45,
 *  (64,64,12544) 52 and 78. A workgroup per kept index that fills a CU: (248,552,280) 70 and 42, (30,600,2500) 74
 *  and 44, (19,304,5760) 93 and 35, (5,1144,8320) 115 and 49, where chain lanes (n up to the next 64, 16 or 4) and
 *  the last round of workgroups are idle for more than three tenths; (64,256,3136) 35.6 and 40, (64,512,1600) 43 and 41.
 *  A workgroup of four waves per kept index, for fewer than 65536 values of each: (17,896,260) 11.7 and 7.2,
 *  (39,957,384) 14.9 and 11.9, but (8,573,240) 5.1 and 6.3, (256,500,100) 19.8 and 22.3. One plane per kept index,
 *  which is one lane there: (1,2048,3136) 46 and 20. */
inline SegmentsPlan PlanSegments(uint32_t n_out, uint32_t n_keep, uint64_t len, uint32_t cus, int least_len) {
  SegmentsPlan p = {false, 16, 1, 1};
  const uint64_t planes = static_cast<uint64_t>(n_out) * n_keep;
  /* 32-bit numbers of planes, fewer than 2^32 threads */
  if (len < static_cast<uint64_t>(least_len) || n_out < 1 || n_out > 2048 || n_keep > 1u << 21 || len >= 1ull << 31 ||
      planes >= 1ull << 31) {
    return p;
  }
  const bool few_kept = static_cast<uint64_t>(n_keep) * 4 < 3ull * cus;
  const bool middling = n_out >= 5 && n_out <= 16;
  const uint32_t side = n_out > 16 ? 64 : n_out > 4 ? 16 : n_out > 1 ? 4 : 1;
  const uint64_t lanes = (n_out + side - 1) / side * side, turns = (n_keep + cus - 1) / cus * cus;
  if (few_kept) {
    p.use = !middling && ((len <= 1100 && planes >= 2048) || (len <= 2048 && planes >= 8192));
  } else if (n_out == 1) {
    p.use = n_keep >= 2 * cus && len <= 4096 && planes * len >= 800000;
  } else if (n_out * len >= 1u << 16) {
    p.use = planes >= 2048 && lanes * turns * 100 > planes * 130;
  } else {
    p.use = !middling && ((len <= 1100 && planes >= 2048) || planes >= 4096) && (n_out <= 4 || lanes * 100 > n_out * 102ull);
  }
  if (!p.use) return p;
  if (len >= 512 && planes / 16 < 4 * cus) p.lanes = 8;  // more waves: (32,512,784) 12.4, with sixteen 13.3
  /* workgroups of four waves or so where planes are few per kept index, but one for every CU */
  while (p.kept * n_out < 4u * p.lanes && n_keep / (p.kept + 1) >= cus) ++p.kept;
  const uint32_t all = (p.kept * n_out + p.lanes - 1) / p.lanes;
  /* a CU holds 20 waves of this kernel: where there are more of them, small workgroups that go round again fill it */
  const uint32_t most = planes / p.lanes >= 20ull * cus ? 4 : kSegMostWaves;
  const uint32_t rounds = (all + most - 1) / most;
  p.waves = (all + rounds - 1) / rounds;
  return p;
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_REDUCE_SEGMENTS_H_
