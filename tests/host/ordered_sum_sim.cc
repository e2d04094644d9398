// Host check of the order-faithful sum of one wave (WaveResolve and PartWaveResolve of
// mshadow_amd/csrc/softmax_kernels.h).
//
// Takes a row slab after slab - LANES lanes x N terms - with the decisions the device code takes:
// the first PLAIN lanes added as they are, then every lane's ulps in the binade of the sum
// (LaneUlps, the very function the device calls), their unsigned prefix sums, the first lane in
// which the binade ends, real float adds for that one, and on from there. The result must be a
// plain serial float loop's bit for bit, on rows built to hit every branch: softmax-like terms,
// ties, sums that double, negative terms, leading zeros, subnormals, infinities and NaN.
// Prints "OK <cases> cases, <n> lanes added as they are" and exits 0 on success.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../mshadow_amd/csrc/ordered_sum.h"

using namespace ordered_sum;

static float Serial(const std::vector<float> &t) {
  volatile float s = 0.0f;
  for (float v : t) s = s + v;
  return s;
}

static long lanes_walked = 0;

// SIGNED, PLAIN and N as on the device; LANES = 64, or 16 / 32 for rows side by side in a wave
template <bool SIGNED, int PLAIN, int LANES, int N>
static float ResolveSim(float s, const float (*t)[N]) {  // t[LANES][N]
  int start = 0;
  for (; start < PLAIN; ++start) s = TrueAdd<N>(s, t[start]);
  while (true) {
    const uint32_t bits = BitsOf(s);
    uint32_t incl[LANES], run = 0u;
    int first = -1;
    for (int l = 0; l < LANES; ++l) {
      run += l >= start ? LaneUlps<SIGNED, N>(t[l], bits & 0xff800000u) : 0u;
      incl[l] = run;
      if (l >= start && first < 0 && (bits & 0x7fffffu) + run >= (1u << 23)) first = l;
    }
    if (first < 0) return FloatOf(bits + incl[LANES - 1]);
    if (first > 0) s = FloatOf(bits + incl[first - 1]);
    s = TrueAdd<N>(s, t[first]);
    ++lanes_walked;
    start = first + 1;
    if (start == LANES) return s;
  }
}

// the first slab of a row with its plain lanes, the others without
template <bool SIGNED, int PLAIN, int LANES, int N>
static bool Check(const std::vector<float> &row, float want, const char *name) {
  std::vector<float> padded(row);
  while (padded.size() % (LANES * N)) padded.push_back(0.0f);
  const float(*t)[N] = reinterpret_cast<const float(*)[N]>(padded.data());
  float s = ResolveSim<SIGNED, PLAIN, LANES, N>(0.0f, t);
  for (size_t l = LANES; l * N < padded.size(); l += LANES) s = ResolveSim<SIGNED, 0, LANES, N>(s, t + l);
  if (BitsOf(s) != BitsOf(want) && !(std::isnan(s) && std::isnan(want))) {
    fprintf(stderr, "MISMATCH %s signed=%d plain=%d lanes=%d N=%d n=%zu got %a want %a\n", name, SIGNED, PLAIN, LANES, N,
            row.size(), s, want);
    return false;
  }
  return true;
}

template <bool SIGNED>
static bool CheckShapes(const std::vector<float> &row, float want, const char *name) {
  return Check<SIGNED, 16, 64, 4>(row, want, name) && Check<SIGNED, 0, 64, 4>(row, want, name) &&
         Check<SIGNED, 0, 64, 1>(row, want, name) && Check<SIGNED, 2, 16, 4>(row, want, name) &&
         Check<SIGNED, 2, 16, 8>(row, want, name) && Check<SIGNED, 2, 32, 8>(row, want, name);
}

// terms that are not negative, by both forms
static bool CheckAll(const std::vector<float> &row, const char *name) {
  const float want = Serial(row);
  return CheckShapes<false>(row, want, name) && CheckShapes<true>(row, want, name);
}

int main() {
  std::mt19937 rng(1234);
  std::normal_distribution<float> normal(0.0f, 1.0f);
  std::uniform_real_distribution<float> uni(0.0f, 1.0f);
  long cases = 0;
  bool ok = true;
  // 1. softmax-like rows: exp(x - max), x ~ N(0, sigma)
  for (float sigma : {0.1f, 1.0f, 3.0f, 10.0f, 40.0f}) {
    for (int n : {1, 3, 64, 257, 1000, 4096, 32000}) {
      for (int rep = 0; rep < 6; ++rep) {
        std::vector<float> x(n);
        float mx = -INFINITY;
        for (auto &v : x) { v = normal(rng) * sigma; mx = std::fmax(mx, v); }
        for (auto &v : x) v = expf(v - mx);
        ok = CheckAll(x, "softmax") && ok;
        ++cases;
      }
    }
  }
  // 2. grids that produce exact ties: multiples of 2^-k around a sum near powers of two
  for (int rep = 0; rep < 200; ++rep) {
    int n = 1 + rng() % 3000;
    std::vector<float> x(n);
    for (auto &v : x) v = std::ldexp(static_cast<float>(rng() % 64), -static_cast<int>(rng() % 30));
    ok = CheckAll(x, "ties") && ok;
    ++cases;
  }
  // 3. all equal (sum of ones is exact below 2^24, then sticks), and constants
  for (float c : {1.0f, 0.5f, 3.0f, 1e-3f, 0.1f}) {
    std::vector<float> x(40000, c);
    ok = CheckAll(x, "const") && ok;
    ++cases;
  }
  // 4. leading zeros / subnormals / tiny then large; ascending and descending magnitudes
  for (int rep = 0; rep < 60; ++rep) {
    int n = 500 + rng() % 5000;
    std::vector<float> x(n);
    for (int i = 0; i < n; ++i) {
      float e = -140.0f + 150.0f * i / n;  // 2^-140 .. 2^10
      x[i] = std::ldexp(1.0f + uni(rng), static_cast<int>(e));
      if (rng() % 7 == 0) x[i] = 0.0f;
    }
    if (rep % 3 == 1) std::reverse(x.begin(), x.end());
    if (rep % 3 == 2) std::shuffle(x.begin(), x.end(), rng);
    ok = CheckAll(x, "range") && ok;
    ++cases;
  }
  {
    std::vector<float> x(3000, 0.0f);
    ok = CheckAll(x, "zeros") && ok;
    x[2999] = 1e-40f;
    ok = CheckAll(x, "zeros+denorm") && ok;
    x[10] = 3e-42f;
    ok = CheckAll(x, "denorms") && ok;
    x[1500] = INFINITY;
    ok = CheckAll(x, "inf") && ok;
    x[100] = NAN;
    ok = CheckAll(x, "nan") && ok;
    x.assign(5000, 3.0e38f);  // overflow to inf on the way
    ok = CheckAll(x, "overflow") && ok;
    cases += 6;
  }
  // 5. uniform magnitudes (binade crossings spread over the whole row)
  for (int rep = 0; rep < 40; ++rep) {
    int n = 20000 + rng() % 20000;
    std::vector<float> x(n);
    for (auto &v : x) v = uni(rng);
    ok = CheckAll(x, "uniform") && ok;
    ++cases;
  }
  // 6. terms of either sign, by the form that allows them; in every third row sums that end a binade
  //    exactly, in every third few bits and hence ties
  for (int rep = 0; rep < 300; ++rep) {
    int n = 1 + rng() % 4000;
    std::vector<float> x(n);
    for (auto &v : x) {
      v = rep % 3 == 0 ? normal(rng) : std::ldexp(1.0f, -static_cast<int>(rng() % (rep % 3 == 1 ? 4 : 30)));
      if (rng() % 64 == 0) v = -std::fabs(v);
      if (rng() % 512 == 0) v = -0.0f;
    }
    if (rep % 10 == 9) x[n / 2] = rep % 20 == 9 ? INFINITY : NAN;
    ok = CheckShapes<true>(x, Serial(x), "signed") && ok;
    ++cases;
  }
  // 7. one lane at the top of a binade: from every sum just below a power of two, terms of half an
  //    ulp, one ulp and their neighbours, so that the upper of the two sums leaves and the lower stays
  for (uint32_t top : {1u, 0x00800000u, 0x01000000u, 0x3f800000u, 0x4b800000u, 0x7f000000u, 0x7f800000u}) {
    for (int rep = 0; rep < 400; ++rep) {
      const float from = FloatOf(top - 1u - (top > 8u ? rng() % 8 : 0u));
      const float ulp = FloatOf(top) - FloatOf(top - 1u);  // of the binade below; infinite at the last one
      std::vector<float> x(1, from);
      for (int i = 0; i < 300; ++i) x.push_back(std::isinf(ulp) ? 1.0141204801825835e31f : ulp * 0.25f * (rng() % 6));
      ok = CheckAll(x, "top") && ok;
      ++cases;
    }
  }
  if (!ok) return 1;
  printf("OK %ld cases, %ld lanes added as they are\n", cases, lanes_walked);
  return 0;
}
