/*
 * Parallel evaluation of a strictly left-to-right float32 sum of non-negative terms.
 *
 * The CPU softmax of the reference adds exp(x - max) into one float accumulator in
 * column order (mshadow/tensor_cpu-inl.h:277-281). With 32000 terms that running sum
 * sits 2.6e-5 (relative) below the exact sum, more than the 1e-5 the results must
 * agree to, so an accurate tree sum does not reproduce it. This file reproduces it
 * bit for bit, in parallel, from one observation:
 *
 *   while the accumulator S stays inside one binade [2^k, 2^(k+1)), its ulp
 *   u = 2^(k-23) is constant and S = m*u with integer m. For a term t >= 0 with
 *   S + t < 2^(k+1),   fl(S + t) = u * (m + rne(t / u))   unless t/u lies exactly
 *   half way between two integers (then the tie-break depends on the parity of m).
 *
 * So inside a binade the float adds are exact INTEGER adds of q = rne(t/u), which are
 * associative. What a lane's few consecutive terms add together is found by ordinary float
 * additions, to two sums that start at the bottom of the binade, one ulp apart: they end one
 * ulp apart exactly when no term was a tie, and the lower one has moved by the lane's total.
 * A wave adds the lanes' totals in unsigned integers and takes the sum as far as it stays in
 * the binade; the lane in which it leaves, or which holds a tie, performs its float additions
 * one by one, and the lanes behind it are measured against the new binade. A row of N(0,3)
 * logits crosses about twenty binades, nearly all of them within its first few hundred terms.
 *
 * The per-lane arithmetic below is plain C++ so that a host program can exercise it lane by
 * lane; the wave / block collectives live in softmax_kernels.h.
 */
#ifndef MSHADOW_AMD_CSRC_ORDERED_SUM_H_
#define MSHADOW_AMD_CSRC_ORDERED_SUM_H_

#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define OSUM_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define OSUM_HD inline __attribute__((always_inline))
#endif

namespace ordered_sum {

OSUM_HD uint32_t BitsOf(float f) {
  uint32_t u;
  memcpy(&u, &f, sizeof(u));
  return u;
}
OSUM_HD float FloatOf(uint32_t u) {
  float f;
  memcpy(&f, &u, sizeof(f));
  return f;
}

/*! \brief the real thing: N float additions in order */
template <int N>
OSUM_HD float TrueAdd(float s, const float (&t)[N]) {
  for (int i = 0; i < N; ++i) s = s + t[i];
  return s;
}

/* ---- the row as a list of addends -------------------------------------------------------
 * The planned row sum of softmax_kernels.h turns a row into a short ordered list of float
 * addends whose plain serial sum IS the left-to-right sum of all terms: a lane (N consecutive
 * terms) whose running sum provably stays in one binade joins a run of such lanes, and the
 * run enters the list as ONE addend, its integer total times the binade's ulp; any other lane
 * (next to a power of two, or holding a tie) enters with its N terms themselves. Adding a
 * run's addend is exact when the sum is in the run's binade before and after it, which is
 * checked on the sums actually obtained (RunHolds): a wrong plan is noticed, never used - it
 * costs time, not a bit. The plan comes from approximate prefix sums (PlanLowBound,
 * PlanHighBound): they say, before any exact work, which pieces of the row - the terms a wave
 * holds in one register slab, then the lanes of the others - the sum traverses in one binade. */

/*! \brief quantisation of one lane's N non-negative terms against the binade with biased
 *  exponent e (0 = the subnormal range, where sums are exact): two accumulators start at
 *  the bottom of the binade, one ulp apart, and take the terms by ordinary float additions.
 *  While both stay in the binade each addition moves them by rne(t / ulp) ulps; a term that
 *  lies half way between two multiples of the ulp moves the even one down and the odd one
 *  up, so the accumulators end one ulp apart exactly when no term was a tie. */
struct LaneQuantum {
  uint32_t q;  //!< sum of rne(t / ulp) over the lane's terms
  bool ok;     //!< no tie, no NaN, and the lane alone does not leave the binade
};
template <int N>
OSUM_HD LaneQuantum LaneDualQuant(const float (&t)[N], uint32_t e) {
  const uint32_t base = e << 23;
  float lo = FloatOf(base), hi = FloatOf(base + 1u);
  for (int i = 0; i < N; ++i) {
    lo = lo + t[i];
    hi = hi + t[i];
  }
  const uint32_t blo = BitsOf(lo), bhi = BitsOf(hi);
  LaneQuantum r;
  r.ok = (bhi - blo == 1u) && blo >= base && bhi < base + (1u << 23);
  r.q = blo - base;
  return r;
}

/*! \brief how many ulps of a sum in the binade that begins at bit pattern `base` (sign and
 *  fraction zero) one lane's N terms add to it: at least 2^23, which leaves any binade, where
 *  that cannot be said - a tie, a NaN, an infinite or (SIGNED) a negative term, no finite binade.
 *  The two sums never come together or part by rounding in the next binade unnoticed: one ulp
 *  apart at the end and the lower one inside the binade, they were so all along. */
template <bool SIGNED, int N>
OSUM_HD uint32_t LaneUlps(const float (&t)[N], uint32_t base) {
  const uint32_t kNone = 1u << 24;
  float lo = FloatOf(base), hi = FloatOf(base + 1u);
  uint32_t signs = 0u;
  for (int i = 0; i < N; ++i) {
    lo = lo + t[i];
    hi = hi + t[i];
    if (SIGNED) signs |= BitsOf(t[i]);
  }
  const uint32_t q = BitsOf(lo) - base;
  const bool ok = BitsOf(hi) - BitsOf(lo) == 1u && q < kNone && (!SIGNED || (signs >> 31) == 0u);
  return ok && base < 0x7f800000u ? q : kNone;
}

/*! \brief bounds on the sequential sum from an accurate sum `approx` of the same terms:
 *  every addition rounds by at most half an ulp, so after n terms the sequential sum sits
 *  within n * 2^-24 of it (relative); sums of softmax terms stay well inside a quarter of
 *  that below and almost nothing above. The bounds only steer the plan. */
OSUM_HD float PlanLowBound(float approx, float terms_in_front) {
  return approx * (1.0f - (terms_in_front * 1.4901161193847656e-08f + 8.0e-6f));  // n * 2^-26
}
OSUM_HD float PlanHighBound(float approx) { return approx * (1.0f + 8.0e-6f); }

/*! \brief the binade a piece stays in if the sum is at least `low` in front of it and at
 *  most `high` behind it; -1 if those lie in different binades (or are not finite) */
OSUM_HD int PlanBinade(float low, float high) {
  const uint32_t blo = BitsOf(low), bhi = BitsOf(high);
  const uint32_t elo = (blo >> 23) & 0xffu, ehi = (bhi >> 23) & 0xffu;
  const bool ok = elo == ehi && ehi < 255u && ((blo | bhi) >> 31) == 0u;
  return ok ? static_cast<int>(elo) : -1;
}

/*! \brief the addend of a run with integer total r in binade e. A total that cannot fit
 *  (the sum itself takes at least 2^23 ulps) becomes an addend that carries any sum out
 *  of the binade, so that RunHolds fails. */
OSUM_HD float RunAddend(uint32_t e, uint32_t r) {
  const uint32_t base = e << 23;
  return r < (1u << 23) ? FloatOf(base + r) - FloatOf(base) : FloatOf(base + (1u << 23));
}

/*! \brief was adding a run of binade e exact? (the sum before and after lies in it) */
OSUM_HD bool RunHolds(float before, float after, uint32_t e) {
  const uint32_t bb = BitsOf(before), ba = BitsOf(after);
  return (bb >> 23) == e && (ba >> 23) == e;  // sign bits are part of the comparison
}

}  // namespace ordered_sum
#endif  // MSHADOW_AMD_CSRC_ORDERED_SUM_H_
