/*
 * Softmax on binary16 rows that are kept on chip: one row per workgroup, up to 131072 columns, read
 * once into registers and written once. Every intermediate is the half_t value
 * the CPU path has (mshadow/tensor_cpu-inl.h:270-285 with DType = half_t), bit for bit.
 *
 * Terms. x - max is one packed 16-bit subtraction. exp of a binary16 number d <= 0 rounded to
 * binary16 is exp2 of the once-rounded product d * log2(e) by the hardware's exp2, rounded: all
 * 31745 such d (every finite one, -0 and -infinity) give the correctly rounded value, and with
 * it what the library's expf gives, at a third of its instructions.
 *
 * Quotients. t / sum goes through the float reciprocal of the row's sum as two floats, high +
 * low: t * high + t * low is the float quotient bit for bit (a quotient of two 11-bit
 * significands is nowhere near half way between two floats), so rounding it to binary16 gives
 * what the division would. All 173,041,665 pairs of a term in [0, 1] and a sum in [1, 2048] agree.
 * The rounding has to be a step of its own: v_fma_mixlo_f16 rounds once, and 1398 of them differ
 * (tests/host/half_quotient_check.cc).
 *
 * The sum. `sum += t` on half_t is one 16-bit add, and their order decides the result: the
 * sum stands still once its ulp exceeds twice the terms. While it stays in one binade
 * [2^k, 2^(k+1)) with ulp u and S = m u, an add moves it by rne(t / u) ulps whatever m is, but for
 * a tie, where the parity of m decides. So what a lane's eight terms do to the sum is two numbers,
 * its increments from an even and from an odd m, and two sums started at the binade's bottom, one
 * ulp apart - the two halves of a packed add - find both. A run is the 64 x 8 = 512 terms of
 * one load of a wave. Where no term of a run is a tie its total is the plain sum of the lanes'
 * increments, and it is applied whole if the sum is in the binade assumed and stays there.
 *   - Every wave holds up to PACKS runs of neighbouring columns, guesses their binade
 *     from float sums of the terms (the sum in 16 bits is the smaller one: the binade below the
 *     guess is prepared too) and files each run's total for both.
 *   - The waves then walk their runs in row order, one wave after the other, the sum handed on
 *     through LDS. One scan over their totals finds the first run that cannot be applied
 *     - a power of two crossed, a tie, another binade - and that one is walked by itself
 *     (HalfRunSum): lane prefixes, the parity rule for ties, real adds by the lane in which a
 *     power of two is crossed, then on from there in the next binade. N(0, 9) logits of 32000
 *     columns cross 14 powers of two and have ties in 4 or 5 runs of 63. A guess is never
 *     trusted: a wrong one costs time.
 *
 * What bounds it: memory where several rows share a CU (8192 x 32000: 230 us, 4.6 TB/s; 204 us with
 * N(0, 0.01) logits, whose sum soon stands still), the latency of a row's steps where it has the CU to
 * itself (2048 x 128000: 329 us), the walk on short rows (65536 x 1000: 97 us). Before - the terms that
 * may change the sum listed and added one by one, 49 instructions an element; a tile kernel for the
 * other lengths, five passes over memory - these took 540, 1519, 1585 and 157 us, 16384 x 8192 481
 * (now 115) and 4096 x 50257 1209 (235).
 */
#ifndef MSHADOW_HIP_KERNELS_SOFTMAX_HALF_H_
#define MSHADOW_HIP_KERNELS_SOFTMAX_HALF_H_

#include "../../half.h"
#include "./common.h"
#include "./half_prune.h"

namespace mshadow {
namespace hip {

/*! \brief columns of a lane's pack and of a run, the packs of a wave */
const int kHalfPack = 8;
const int kHalfRun = kWave * kHalfPack;
/*! \brief lanes of a row's first run whose terms are added one by one */
const uint32_t kHalfPlainLanes = 16;

/*! \brief eight binary16 values as four 32-bit words */
typedef uint32_t HalfWords __attribute__((ext_vector_type(4)));
typedef _Float16 HalfPair __attribute__((ext_vector_type(2)));
typedef float FloatPair __attribute__((ext_vector_type(2)));

__device__ __forceinline__ HalfPair AsHalfPair(uint32_t w) { return __builtin_bit_cast(HalfPair, w); }
__device__ __forceinline__ uint32_t AsWord(HalfPair p) { return __builtin_bit_cast(uint32_t, p); }

/*! \brief value i of a pack, and its replacement */
__device__ __forceinline__ uint16_t HalfBits(const HalfWords &p, int i) {
  return static_cast<uint16_t>(p[i >> 1] >> ((i & 1) * 16));
}
__device__ __forceinline__ void SetHalfBits(HalfWords *p, int i, uint32_t bits) {
  const uint32_t keep = (i & 1) ? 0x0000ffffu : 0xffff0000u;
  (*p)[i >> 1] = ((*p)[i >> 1] & keep) | (bits << ((i & 1) * 16));
}

/*! \brief the larger of two pairs, half by half (one instruction; NaN operands are ignored) */
__device__ __forceinline__ uint32_t MaxHalfPair(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
/*! \brief ... as unsigned 16-bit integers */
__device__ __forceinline__ uint32_t MaxU16Pair(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_max_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

/*! \brief pack `at` (uniform) of the registers: a binary tree of uniform branches */
template <int PACKS, int LO, int HI>
struct HalfPackPicker {
  static __device__ __forceinline__ HalfWords Pick(const HalfWords (&v)[PACKS], int at) {
    const int MID = (LO + HI) / 2;
    return at < MID ? HalfPackPicker<PACKS, LO, MID>::Pick(v, at) : HalfPackPicker<PACKS, MID, HI>::Pick(v, at);
  }
};
template <int PACKS, int LO>
struct HalfPackPicker<PACKS, LO, LO + 1> {
  static __device__ __forceinline__ HalfWords Pick(const HalfWords (&v)[PACKS], int) {
    HalfWords t = v[LO];
    /* keeps the tree a tree: folded into one indexed access, the row would move from registers
       to scratch memory */
    asm volatile("" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]));
    return t;
  }
};

/*! \brief two binary16 sums started one ulp apart at the bottom of binade `base` (a bit
 *  pattern with no fraction), behind the eight terms: the even one in the low half */
__device__ __forceinline__ uint32_t HalfDualSum(const HalfWords &t, uint32_t base) {
  HalfPair acc = AsHalfPair(base | ((base + 1u) << 16));
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const HalfPair p = AsHalfPair(t[k]);
    acc += HalfPair{p.x, p.x};
    acc += HalfPair{p.y, p.y};
  }
  return AsWord(acc);
}

/*! \brief inclusive scan over the lanes of the maps "parity of the sum -> increment": *even and
 *  *odd are what a lane adds to an even / odd sum, and become what lanes 0 .. l add together */
__device__ __forceinline__ void HalfScanMaps(uint32_t *even, uint32_t *odd) {
#define MSHADOW_MAP_STEP(CTRL, MASK)                                    \
  {                                                                     \
    const uint32_t e = DppU32<CTRL, MASK>(0u, *even);                   \
    const uint32_t o = DppU32<CTRL, MASK>(0u, *odd);                    \
    const uint32_t behind_even = e + ((e & 1u) != 0u ? *odd : *even);   \
    const uint32_t behind_odd = o + ((o & 1u) != 0u ? *even : *odd);    \
    *even = behind_even;                                                \
    *odd = behind_odd;                                                  \
  }
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_SHR(1), 0xf)
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_SHR(2), 0xf)
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_SHR(4), 0xf)
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_SHR(8), 0xf)
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_BCAST15, 0xa)
  MSHADOW_MAP_STEP(MSHADOW_DPP_ROW_BCAST31, 0xc)
#undef MSHADOW_MAP_STEP
}

/*! \brief bits of the sum s (uniform) behind the terms of lane `from`: every lane adds its own,
 *  one result is taken */
__device__ __forceinline__ uint32_t HalfLaneSum(const HalfWords &t, uint32_t s, int from) {
  HalfPair sum = AsHalfPair(s);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const HalfPair p = AsHalfPair(t[k]);
    sum.x += p.x;
    sum.x += p.y;
  }
  return ReadLaneU32(AsWord(sum) & 0xffffu, from);
}

/*! \brief bits of the sum `s` (uniform) behind the wave's 512 terms, lane by lane, eight to a
 *  lane, each add rounded. Terms are non-negative or NaN, and at most 1, so s is finite or NaN. */
__device__ __forceinline__ uint32_t HalfRunSum(const HalfWords &t, uint32_t s) {
  const uint32_t lane = LaneId();
  /* a run of which no term can change the sum (half_prune.h) */
  const uint32_t peaks = MaxU16Pair(MaxU16Pair(t[0], t[1]), MaxU16Pair(t[2], t[3]));
  const uint32_t peak = (peaks & 0xffffu) > (peaks >> 16) ? peaks & 0xffffu : peaks >> 16;
  if (__ballot(peak >= HalfSignificantFrom(s)) == 0ull) return s;
  uint32_t start = 0u;  // lanes in front of it are in s already
  if (s == 0u) {
    /* a sum that starts doubles within a few lanes, again and again: those are added plainly
       (65536 x 1000: 164 us without, 140 us with eight lanes) */
#pragma unroll 1
    for (; start < kHalfPlainLanes; ++start) s = HalfLaneSum(t, s, static_cast<int>(start));
  }
  while ((s >> 10) < 31u) {  // nothing changes a NaN
    const uint32_t base = s & 0x7c00u, m = s & 0x3ffu;
    const uint32_t acc = HalfDualSum(t, base);
    uint32_t even = (acc & 0xffffu) - base, odd = (acc >> 16) - base - 1u;
    if (lane < start) even = odd = 0u;
    uint32_t incl;
    if (__ballot(even != odd) == 0ull) {
      incl = WaveInclusiveScanU32(even);
    } else {
      HalfScanMaps(&even, &odd);
      incl = (m & 1u) != 0u ? odd : even;
    }
    /* a lane that leaves the binade by itself has an increment of 1024 and more (from an odd m,
       of 1023), so the first lane found here is the one in which the binade ends; what the scan
       holds for lanes behind it does not matter */
    const unsigned long long leaving = __ballot(m + incl >= 1024u);
    if (leaving == 0ull) return s + ReadLaneU32(incl, kWave - 1);
    const int first = __ffsll(leaving) - 1;
    if (first > 0) s += ReadLaneU32(incl, first - 1);
    s = HalfLaneSum(t, s, first);
    start = static_cast<uint32_t>(first) + 1u;
    if (start == static_cast<uint32_t>(kWave)) break;
  }
  return s;
}

/*! \brief increments of all runs of a wave in the binades of `guess` (lane q: biased exponent
 *  for run q), lane l the total of run l % PACKS; *ties gets a bit per run that holds a
 *  tie or a NaN */
template <int PACKS>
__device__ __forceinline__ uint32_t HalfRunTotals(const HalfWords (&v)[PACKS], uint32_t runs,
                                                  uint32_t guess, uint32_t *ties) {
  uint32_t part[PACKS];
  uint32_t tied = 0u;
#pragma unroll
  for (int q = 0; q < PACKS; ++q) {
    part[q] = 0u;
    if (static_cast<uint32_t>(q) < runs) {
      const uint32_t base = ReadLaneU32(guess, q) << 10;
      const uint32_t acc = HalfDualSum(v[q], base);
      part[q] = (acc & 0xffffu) - base;
      tied |= __ballot((acc >> 16) - (acc & 0xffffu) != 1u) != 0ull ? 1u << q : 0u;
    }
  }
  *ties = tied;
  return WaveReduceMany<WaveOpSum, uint32_t, PACKS>(part);
}

/*! \brief one row of more than 16 columns, and at most WAVES * PACKS runs, per workgroup of WAVES
 *  waves (seven columns fewer where rows of src do not all start 16-byte aligned). In place (dst == src) is safe: the
 *  row is read whole before any of it is written.
 *
 *  The row is cut where src is 16-byte aligned, up to seven columns before its start: loads that
 *  straddle cache lines cost a sixth of the kernel (8192 x 31999: 270 us with packs counted from the
 *  row's start, 8192 x 32000: 231 us). The columns that the first and the last pack lack are
 *  -infinity, i.e. zero terms, and those packs' own columns come and go one by one. */
template <int WAVES, int PACKS>
__global__ void __launch_bounds__(WAVES * kWave, PACKS <= 4 ? 8 : PACKS <= 8 ? 5 : 4)
    SoftmaxHalfRowKernel(half::half_t *dst, uint32_t dstride, const half::half_t *src, uint32_t sstride,
                         uint32_t cols) {
  typedef HalfWords Loose __attribute__((aligned(2)));
  const float kLog2E = 1.44269504088896340736f;
  __shared__ float wave_max[WAVES];
  __shared__ float wave_total[WAVES];
  __shared__ uint32_t row_sum;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint16_t *e = reinterpret_cast<const uint16_t *>(src) + static_cast<size_t>(blockIdx.x) * sstride;
  uint16_t *o = reinterpret_cast<uint16_t *>(dst) + static_cast<size_t>(blockIdx.x) * dstride;
  const uint32_t skew = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(e) / sizeof(uint16_t)) % kHalfPack;
  e -= skew;
  o -= skew;
  /* the row is columns skew .. end of what e and o point to; whole packs [whole_from, whole_to) */
  const uint32_t end = skew + cols;
  const uint32_t whole_from = skew != 0u ? kHalfPack : 0u;
  const uint32_t whole_to = end - end % kHalfPack;

  /* this wave's runs: neighbouring ones, so that the sum passes from wave to wave once */
  const uint32_t all_runs = (end + kHalfRun - 1) / kHalfRun;
  const uint32_t per_wave = (all_runs + WAVES - 1) / WAVES;
  const uint32_t first_run = wave * per_wave;
  const uint32_t runs = first_run >= all_runs ? 0u
                        : all_runs - first_run < per_wave ? all_runs - first_run : per_wave;
  const uint32_t x_of_lane = first_run * kHalfRun + lane * kHalfPack;
  const uint32_t tail_run = whole_to / kHalfRun - first_run;  // of this wave, if below `runs`
  const bool tail_lane = (whole_to - x_of_lane) % kHalfRun == 0u;

  HalfWords v[PACKS];
#pragma unroll
  for (int q = 0; q < PACKS; ++q) {
    v[q] = HalfWords{0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u};
    const uint32_t x = x_of_lane + q * kHalfRun;
    if (static_cast<uint32_t>(q) < runs && x >= whole_from && x < whole_to) {
      v[q] = *reinterpret_cast<const HalfWords *>(e + x);
    }
  }
  HalfWords edge = {0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u, 0xfc00fc00u};
  /* The columns of the edges: their loads all under way together, those of columns that are not the row's from
     one that is. Loaded where each is wanted they came one after the other: 8192 x 31999 241 us that way and
     232 now, 1064 x 28245 51 and 47.5, 4096 x 50257 235 and 230, 20000 x 777 36.5 and 35.3. */
  if (wave == 0u && skew != 0u && lane == 0u) {
    uint32_t t[kHalfPack];
#pragma unroll
    for (int i = 1; i < kHalfPack; ++i) t[i] = e[static_cast<uint32_t>(i) >= skew ? i : skew];
#pragma unroll
    for (int i = 1; i < kHalfPack; ++i) asm volatile("" : "+v"(t[i]));
#pragma unroll
    for (int i = 1; i < kHalfPack; ++i) {
      if (static_cast<uint32_t>(i) >= skew) SetHalfBits(&v[0], i, t[i]);
    }
  }
  if (end != whole_to && tail_run < runs && tail_lane) {
    uint32_t t[kHalfPack];
#pragma unroll
    for (int i = 0; i < kHalfPack - 1; ++i) t[i] = e[whole_to + i < end ? whole_to + i : end - 1u];
#pragma unroll
    for (int i = 0; i < kHalfPack - 1; ++i) asm volatile("" : "+v"(t[i]));
#pragma unroll
    for (int i = 0; i < kHalfPack - 1; ++i) {
      if (whole_to + i < end) SetHalfBits(&edge, i, t[i]);
    }
#pragma unroll
    for (int q = 0; q < PACKS; ++q) {
      if (static_cast<uint32_t>(q) == tail_run) v[q] = edge;
    }
  }

  /* its maximum: `if (mmax < e[x]) mmax = e[x]` from e[0] on, which is the largest value. With a
     NaN in the row every result is NaN, whatever maximum is found. */
  uint32_t most = 0xfc00fc00u;
#pragma unroll
  for (int q = 0; q < PACKS; ++q) {
    if (static_cast<uint32_t>(q) < runs) {
      most = MaxHalfPair(most, MaxHalfPair(MaxHalfPair(v[q][0], v[q][1]), MaxHalfPair(v[q][2], v[q][3])));
    }
  }
  const HalfPair two = AsHalfPair(most);
  const float low_half = static_cast<float>(two.x), high_half = static_cast<float>(two.y);
  float m = WaveMaxF32(low_half < high_half ? high_half : low_half);
  if (WAVES > 1) {
    if (lane == 0) wave_max[wave] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float other = wave_max[w];
      m = m < other ? other : m;
    }
  }
  const _Float16 mh = static_cast<_Float16>(m);  // exact: m is one of the row's values
  const HalfPair mmax = {mh, mh};

  /* the terms, in place of the logits, and float sums of every run */
  float sums[PACKS];
#pragma unroll
  for (int q = 0; q < PACKS; ++q) {
    sums[q] = 0.0f;
    if (static_cast<uint32_t>(q) < runs) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const HalfPair d = AsHalfPair(v[q][k]) - mmax;
        FloatPair t;
        t.x = __builtin_amdgcn_exp2f(__builtin_fmaf(static_cast<float>(d.x), kLog2E, 0.0f));
        t.y = __builtin_amdgcn_exp2f(__builtin_fmaf(static_cast<float>(d.y), kLog2E, 0.0f));
        const HalfPair h = __builtin_convertvector(t, HalfPair);
        v[q][k] = AsWord(h);
        sums[q] = __builtin_amdgcn_fdot2(h, HalfPair{1.0f, 1.0f}, sums[q], false);
      }
      /* one pack after the other, and only its packed words kept: 128 floats would spill */
      asm volatile("" : "+v"(v[q][0]), "+v"(v[q][1]), "+v"(v[q][2]), "+v"(v[q][3]), "+v"(sums[q]));
    }
  }

  /* binades guessed from the sums, and every run's increments in them and the ones below */
  const float own = WaveSumMany<PACKS>(sums);  // lane l: run l % PACKS
  const float own_incl = WaveInclusiveScanF32(lane < static_cast<uint32_t>(PACKS) ? own : 0.0f);
  float in_front = 0.0f;
  if (WAVES > 1) {
    if (lane == 0) wave_total[wave] = ReadLaneF32(own_incl, PACKS - 1);
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) in_front += wave_total[w];
  }
  /* the sum of terms of at most 1 does not pass 2048 in 16 bits; a NaN becomes that as well */
  const float about = in_front + own_incl;
  const _Float16 guessed = static_cast<_Float16>(about < 2048.0f ? about : 2048.0f);
  const uint32_t guess = static_cast<uint32_t>(__builtin_bit_cast(uint16_t, guessed)) >> 10;
  const uint32_t below = guess > 0u ? guess - 1u : 0u;
  uint32_t ties, ties_below;
  const uint32_t total = HalfRunTotals(v, runs, guess, &ties);
  const uint32_t total_below = HalfRunTotals(v, runs, below, &ties_below);

  /* the walk, wave after wave */
  uint32_t s = 0u;
  for (uint32_t w = 0; w < static_cast<uint32_t>(WAVES); ++w) {
    if (w == wave) {
      __builtin_amdgcn_s_setprio(3);  // the row waits for it
      if (WAVES > 1 && wave != 0u) s = __builtin_amdgcn_readfirstlane(row_sum);
      uint32_t done = 0u;
      while (done < runs && (s >> 10) < 31u) {
        const uint32_t binade = s >> 10;
        uint32_t step = guess == binade ? ((ties >> (lane & 31u)) & 1u ? 1024u : total)
                        : below == binade ? ((ties_below >> (lane & 31u)) & 1u ? 1024u : total_below)
                                          : 1024u;
        const bool mine = lane >= done && lane < runs;
        if (!mine) step = 0u;
        const uint32_t incl = WaveInclusiveScanU32(step);
        const unsigned long long stop = __ballot(mine && (s & 0x3ffu) + incl >= 1024u);
        const int at = stop == 0ull ? static_cast<int>(runs) : __ffsll(stop) - 1;
        if (at > 0) s += ReadLaneU32(incl, at - 1);
        if (stop == 0ull) break;
        s = __builtin_amdgcn_readfirstlane(
            HalfRunSum(HalfPackPicker<PACKS, 0, PACKS>::Pick(v, at), s));
        done = static_cast<uint32_t>(at) + 1u;
      }
      if (WAVES > 1 && lane == 0) row_sum = s;
      __builtin_amdgcn_s_setprio(0);
    }
    if (WAVES > 1) __syncthreads();
  }
  if (WAVES > 1) s = row_sum;

  const float sum = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(s)));
  const float high = 1.0f / sum;
  const float low = __builtin_fmaf(-sum, high, 1.0f) * high;
#pragma unroll
  for (int q = 0; q < PACKS; ++q) {
    if (static_cast<uint32_t>(q) < runs) {
      const uint32_t x = x_of_lane + q * kHalfRun;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const HalfPair t = AsHalfPair(v[q][k]);
        FloatPair p;
        p.x = __builtin_fmaf(static_cast<float>(t.x), high, __builtin_fmaf(static_cast<float>(t.x), low, 0.0f));
        p.y = __builtin_fmaf(static_cast<float>(t.y), high, __builtin_fmaf(static_cast<float>(t.y), low, 0.0f));
        asm volatile("" : "+v"(p.x), "+v"(p.y));  // the rounding to binary16 is a step of its own
        v[q][k] = AsWord(__builtin_convertvector(p, HalfPair));
      }
      if (x >= whole_from && x < whole_to) {
        __builtin_nontemporal_store(v[q], reinterpret_cast<Loose *>(o + x));
      } else if (x == whole_to) {
        edge = v[q];
      }
    }
  }
  if (wave == 0u && skew != 0u && lane == 0u) {
#pragma unroll
    for (int i = 1; i < kHalfPack; ++i) {
      if (static_cast<uint32_t>(i) >= skew) o[i] = HalfBits(v[0], i);
    }
  }
  if (end != whole_to && tail_run < runs && tail_lane) {
#pragma unroll
    for (int i = 0; i < kHalfPack - 1; ++i) {
      if (whole_to + i < end) o[whole_to + i] = HalfBits(edge, i);
    }
  }
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_SOFTMAX_HALF_H_
