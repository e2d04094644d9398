/*
 * Strictly left-to-right float32 sums of signed terms, a chunk of 128 terms at a time.
 *
 * The reference adds a column top to bottom into one float (mshadow/tensor_cpu-inl.h:203-228). A
 * chunk of terms maps the sum S in front of it to the sum behind it, f(S) = fl(...fl(fl(S + t0) + t1)
 * ...), and that map is regular: it is monotone, and if two sums differ by a multiple of 2 U, where U
 * is the largest ulp of any sum on the way, and the two ways pass through the same binades, every
 * rounding on the one is the same rounding on the other (ties included, for 2 U keeps the parity of a
 * sum's last bit) and the results differ by what the sums differed by. So if S is known nearly - A,
 * from ordinary sums in any order - then f is known on a window around A from eight chains:
 *
 *   u = ulp(A); chains start at A - W, A + u, A + 2u, ..., A + 6u, A + 7u + W, W a multiple of 8u.
 *   The outermost two bound every chain in between (f is monotone), so if they share sign and binade
 *   after every add, all starts in the window do; if moreover no sum's ulp exceeds 4u, sums that
 *   differ by a multiple of 8u are translated. Then for S = A + q u inside the window
 *   f(S) = f(A + (q mod 8) u) + (q - q mod 8) u, exactly.
 *
 * Two more chains bound a window eight times as wide, and two one as wide as the sum in front can be away from
 * the expected one; the widest that holds is the one that counts: how far S is from A is not known, and a
 * window is lost where the sum passes zero or a power of two at a distance below its width. Roundings
 * at random leave S within the first or the second. Where they all go one way (a column of 0.1, a mean's
 * gradient, dropped-out ones) S drifts away from A by up to half an ulp a row, and only the third has it.
 *
 * The chains of all chunks run at once; what is left in sequence is one look-up per chunk (Apply,
 * about ten instructions for 128 dependent adds), which checks that S lies in the window. Chunks
 * whose map is not known this way - the sum grows fourfold from next to nothing, or passes a power of two
 * or zero too near - are added term by term: 3 to 4 % of the chunks of 16384 to 65536 N(0, 1) terms or a
 * classifier's gradients (up to 13 % in single columns, whose sum stays near such a value), 7 and 23 % with
 * one window; of columns of equal terms 3 to 8 %, 40 to 100 % without the third.
 *
 * Plain C++, so that a host program can run the same functions against a serial loop.
 */
#ifndef MSHADOW_AMD_CSRC_COLUMN_CHUNKS_H_
#define MSHADOW_AMD_CSRC_COLUMN_CHUNKS_H_

#include "ordered_sum.h"

namespace column_chunks {

using ordered_sum::BitsOf;
using ordered_sum::FloatOf;

const int kRows = 128;     // terms of a chunk
const int kClasses = 8;    // chains of a chunk
const uint32_t kMinWindow = 3, kMaxWindow = 14;  // of the second window: 8u * 2^j to either side
const uint32_t kNarrower = 3;                     // j of the second less that of the first
const uint32_t kMaxWidest = 16;                   // of the third: a sixteenth of a binade

/*! \brief what a chunk does to the sum in front of it */
struct Map {
  float a;         // the sum expected in front of it
  float e0;        // f(a)
  uint32_t shift;  // four bits a class b: (b u - (f(a + b u) - f(a))) / u, from -8 to 7; where there is no map
                   // whether all terms are finite
  uint32_t how;    // the window's exponent j (W = 8u * 2^j), kByTerms where there is no map, where the terms are
};
const uint32_t kByTerms = 0x80000000u;
/*! \brief where: in the matrix; nowhere, there is nothing to add (all are -0), or zeros that turn a sum of -0 into
 *  +0; or kKept + the place of a copy */
const uint32_t kInMatrix = 0, kNothing = 1, kPlusZero = 2, kKept = 3;
OSUM_HD uint32_t How(bool by_terms, uint32_t j, uint32_t where) { return (by_terms ? kByTerms : 0u) | where << 5 | j; }
OSUM_HD bool IsByTerms(uint32_t how) { return (how & kByTerms) != 0u; }
OSUM_HD uint32_t WindowOf(uint32_t how) { return how & 31u; }
OSUM_HD uint32_t WhereOf(uint32_t how) { return (how & ~kByTerms) >> 5; }

OSUM_HD uint32_t Exponent(float f) { return (BitsOf(f) >> 23) & 0xffu; }
OSUM_HD float Magnitude(float f) { return FloatOf(BitsOf(f) & 0x7fffffffu); }
/*! \brief chunks that start from sums of these exponents have a grid u whose reciprocal is a float too */
OSUM_HD bool StartsOnGrid(float a) { return Exponent(a) >= 40u && Exponent(a) <= 250u; }
OSUM_HD float Grid(float a) { return FloatOf((Exponent(a) - 23u) << 23); }
OSUM_HD float GridInverse(float a) { return FloatOf((277u - Exponent(a)) << 23); }
/*! \brief half the window, 8u * 2^j */
OSUM_HD float Window(float a, uint32_t j) { return FloatOf((Exponent(a) - 20u + j) << 23); }

/*! \brief j for the second window: the sum in front of the chunk has been rounded `rows` times at an ulp of at most
 *  ulp(most), so it is about 0.3 sqrt(rows) of those from the exact sum where roundings are at random, and more
 *  where small terms vanish in a large sum; the window is at least 4 sqrt(rows) of 2^-23 most. May exceed
 *  kMaxWindow: the chunk is then added term by term. */
OSUM_HD uint32_t WindowFor(float a, float most, float sqrt_rows) {
  const float want = most * sqrt_rows * FloatOf((127u - 21u) << 23);
  const uint32_t have = Exponent(a) - 20u, need = Exponent(want) + 1u;
  return need > have + kMinWindow ? need - have : kMinWindow;
}

/*! \brief j for the third: the sum in front of the chunk is off by half an ulp of `most` a row at worst */
OSUM_HD uint32_t WidestFor(float a, float most, float rows, uint32_t j) {
  const float want = most * rows * FloatOf((127u - 24u) << 23);
  const uint32_t have = Exponent(a) - 20u, need = Exponent(want) + 1u;
  const uint32_t widest = need > have + j ? need - have : j;
  return widest < kMaxWidest ? widest : kMaxWidest;
}

/*! \brief the windows a chunk's chains are started for: j of the second and third */
struct Windows {
  uint32_t second, third;
};
OSUM_HD Windows WindowsFor(float a, float most, float rows, float sqrt_rows) {
  Windows w;
  w.second = WindowFor(a, most, sqrt_rows);
  w.third = WidestFor(a, most, rows, w.second);
  return w;
}

struct Chains {
  float s[kClasses], low, high, lowest, highest;  // these bound the second and the third window
  uint32_t differ, far, farthest;  // the bits in which the outermost sums of the three windows ever differed
  float most;            // largest magnitude of a sum

  OSUM_HD void Start(float a, Windows j) {
    const float u = Grid(a), w = Window(a, j.second - kNarrower), wide = Window(a, j.second), widest = Window(a, j.third);
    for (int b = 0; b < kClasses; ++b) s[b] = a + static_cast<float>(b) * u;
    low = a - wide;
    high = s[kClasses - 1] + wide;
    lowest = a - widest;
    highest = s[kClasses - 1] + widest;
    s[0] = a - w;
    s[kClasses - 1] = s[kClasses - 1] + w;
    differ = BitsOf(s[0]) ^ BitsOf(s[kClasses - 1]);
    far = BitsOf(low) ^ BitsOf(high);
    farthest = BitsOf(lowest) ^ BitsOf(highest);
    most = 0.0f;
  }
  OSUM_HD void Add(float t) {
    for (int b = 0; b < kClasses; ++b) s[b] = s[b] + t;
    low = low + t;
    high = high + t;
    lowest = lowest + t;
    highest = highest + t;
    differ |= BitsOf(s[0]) ^ BitsOf(s[kClasses - 1]);
    far |= BitsOf(low) ^ BitsOf(high);
    farthest |= BitsOf(lowest) ^ BitsOf(highest);
    most = __builtin_fmaxf(most, __builtin_fabsf(s[0]));
  }
  /*! \brief the map, and whether it is one (Start was from a sum on a grid, j within bounds), and whether with the
   *  second or third window. Infinities and NaNs stay in a sum once they are in it, so the last sums show them. */
  OSUM_HD bool Finish(float a, Windows j, Map *m, bool *wide) const {
    const bool known = (differ & 0xff800000u) == 0u && Exponent(most) <= Exponent(a) + 2u &&
                       Exponent(s[0]) < 254u && Exponent(s[kClasses - 1]) < 254u;
    const bool widest = (farthest & 0xff800000u) == 0u && Exponent(lowest) < 254u && Exponent(highest) < 254u;
    *wide = widest || ((far & 0xff800000u) == 0u && Exponent(low) < 254u && Exponent(high) < 254u);
    const float w = Window(a, j.second - kNarrower), inverse = GridInverse(a);
    m->a = a;
    m->e0 = s[0] + w;
    m->shift = 0u;
    for (int b = 1; b < kClasses; ++b) {
      const float e = b < kClasses - 1 ? s[b] : s[b] - w;
      const int places = known ? b - static_cast<int>((e - m->e0) * inverse) : 0;
      m->shift |= (static_cast<uint32_t>(places) & 15u) << (4 * b);
    }
    m->how = How(!known, widest ? j.third : *wide ? j.second : j.second - kNarrower, kInMatrix);
    return known;
  }
};

/*! \brief a Map as the walk down a column reads it */
struct Step {
  float a, inverse, e0, grid;
  uint32_t shift;
  float window;  // -1: not a map
};
OSUM_HD Step StepOf(const Map &m) {
  Step s;
  const bool ok = !IsByTerms(m.how);
  s.a = m.a;
  s.inverse = ok ? GridInverse(m.a) : 0.0f;
  s.e0 = m.e0;
  s.grid = ok ? Grid(m.a) : 0.0f;
  s.shift = m.shift;
  s.window = ok ? Window(m.a, WindowOf(m.how)) : -1.0f;
  return s;
}
/*! \brief the sum behind the chunk into *next; false (and nothing of use there) where S is outside the window */
OSUM_HD bool Apply(const Step &m, float s, float *next) {
  const float d = s - m.a;  // exact inside the window: s and a share their binade
  /* d / u in the low bits of a float of 2^23 and a half */
  const uint32_t q = BitsOf(__builtin_fmaf(d, m.inverse, 12582912.0f));
#if defined(__HIP_DEVICE_COMPILE__)
  const int places = __builtin_amdgcn_sbfe(m.shift, q << 2, 4u);  // takes the place modulo 32
#else
  const int places = static_cast<int>(m.shift << (28u - ((q << 2) & 28u))) >> 28;
#endif
  *next = m.e0 + __builtin_fmaf(-static_cast<float>(places), m.grid, d);
  return __builtin_fabsf(d) <= m.window;
}

}  // namespace column_chunks

#endif  // MSHADOW_AMD_CSRC_COLUMN_CHUNKS_H_
