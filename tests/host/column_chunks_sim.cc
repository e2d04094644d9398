// The column sums by chunks (csrc/column_chunks.h) on the host: the functions of the device code, walked down
// columns as the kernels walk them - approximate sums in front of every chunk, twelve chains a chunk, one
// look-up a chunk or 128 additions - against the reference's serial loop, bit for bit. Prints, per kind of
// column, the share of the chunks that were added term by term.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <string>
#include <vector>

#include "../../mshadow_amd/csrc/column_chunks.h"

using namespace column_chunks;

static float Serial(const std::vector<float> &t) {
  volatile float s = t[0];
  for (size_t i = 1; i < t.size(); ++i) s = s + t[i];
  return s;
}

// windows: how far beside the exact sum the expected sums are, in units of the window
static float Walk(const std::vector<float> &t, double beside, long *chunks, long *by_terms) {
  const size_t n = t.size(), count = (n + kRows - 1) / kRows;
  float sum = -0.0f, before = 0.0f, most = 0.0f;
  for (size_t c = 0; c < count; ++c) {
    float term[kRows];
    for (int i = 0; i < kRows; ++i) term[i] = c * kRows + i < n ? t[c * kRows + i] : -0.0f;
    float a = before;
    most = std::fmax(most, std::fabs(a));
    bool known = false, wide;
    Map m;
    if (StartsOnGrid(a)) {
      const float rows = static_cast<float>(c * kRows);
      const Windows j = WindowsFor(a, most, rows, std::sqrt(rows));
      if (j.second <= kMaxWindow) {
        if (beside != 0) a += static_cast<float>(beside) * Window(a, j.second);
        if (StartsOnGrid(a)) {
          Chains chains;
          chains.Start(a, j);
          for (int i = 0; i < kRows; ++i) chains.Add(term[i]);
          known = chains.Finish(a, j, &m, &wide);
        }
      }
    }
    if (!known) m.how = How(true, 0, kInMatrix), m.a = a, m.e0 = 0, m.shift = 0;
    const Step st = StepOf(m);
    float next;
    ++*chunks;
    if (Apply(st, sum, &next)) {
      sum = next;
    } else {
      ++*by_terms;
      volatile float s = sum;
      for (int i = 0; i < kRows; ++i) s = s + term[i];
      sum = s;
    }
    float part = 0.0f;
    for (int i = 0; i < kRows; ++i) part += term[i];
    before += part;
  }
  return sum;
}

int main() {
  std::mt19937 gen(5);
  std::normal_distribution<float> normal(0.0f, 1.0f);
  std::uniform_real_distribution<float> unit(0.0f, 1.0f);
  const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
  struct Kind {
    const char *name;
    int rows;
    double most;  // the largest share of chunks by terms that is no fault
  };
  const Kind kinds[] = {{"normal", 16384, 0.06}, {"normal", 65537, 0.06}, {"gradient", 65536, 0.05},
                        {"gradient100", 30000, 0.08}, {"positive", 30001, 0.05}, {"small", 16384, 0.06},
                        {"halves", 20000, 1}, {"integers", 20000, 1}, {"constant", 20000, 0.1}, {"constant", 65536, 0.06}, {"mean", 65536, 0.06},
                        {"kept", 65536, 0.06}, {"then constant", 65536, 0.06}, {"constant first", 65536, 0.06}, {"alternating", 9000, 1},
                        {"subnormal", 9000, 1}, {"wide", 9000, 1}, {"huge", 9000, 1}, {"infinity", 9000, 1},
                        {"nan", 9000, 1}, {"zeros", 9000, 1}, {"minus zeros", 9000, 1}, {"cancelling", 9000, 1},
                        {"one", 1, 1}, {"short", 127, 1}, {"chunk", 128, 1}, {"odd", 129, 1}};
  for (const Kind &kind : kinds) {
    const std::string name = kind.name;
    long chunks = 0, by_terms = 0;
    for (int column = 0; column < 24; ++column) {
      std::vector<float> t(kind.rows);
      const int classes = name == "gradient" ? 1000 : 100;
      for (int i = 0; i < kind.rows; ++i) {
        float v = normal(gen);
        if (name == "gradient" || name == "gradient100") {
          // p of a softmax over N(0, 9) logits: their sum is near classes * exp(4.5)
          const float p = std::exp(3.0f * v) / (classes * 90.0f);
          v = (p < 1 ? p : 1) - (unit(gen) * classes < 1 ? 1.0f : 0.0f);
        }
        if (name == "positive") v = unit(gen);
        if (name == "small") v *= 1e-20f;
        if (name == "halves") v = std::round(v * 64) / 64;
        if (name == "integers") v = std::round(v * 1000) * 4099;
        if (name == "constant") v = 0.1f * (column + 1);
        if (name == "mean") v = 1.0f / (65536.0f * (97 + column));
        if (name == "kept") v = unit(gen) < 0.1f + 0.03f * column ? 1.0f / (0.1f + 0.03f * column) : 0.0f;
        if (name == "then constant" && i > 30000) v = 0.03f * (column + 1);
        if (name == "constant first" && i < 30000) v = 0.03f * (column + 1);
        if (name == "alternating") v = (i & 1 ? -1.0f : 1.0f) * (1 + column);
        if (name == "subnormal") v *= 1e-42f;
        if (name == "wide") v *= std::exp2(std::floor(unit(gen) * 60) - 30);
        if (name == "huge") v = std::fabs(v) * 3e34f * (column + 1);
        if (name == "infinity" && i == 400 * (column + 1) / 2) v = column & 1 ? inf : -inf;
        if (name == "nan" && i == 350 * column) v = nan;
        if (name == "zeros") v = i == 300 * column ? -0.0f : 0.0f;
        if (name == "minus zeros") v = column & 1 && i == 8000 ? 0.0f : -0.0f;
        if (name == "cancelling" && i % 700 == 699) {
          volatile float s = 0;
          for (int k = 0; k < i; ++k) s = s + t[k];
          v = -s * (column & 1 ? 1.0f : 1.0000001f);
        }
        t[i] = v;
      }
      const float want = Serial(t);
      for (double beside : {0.0, 0.45, -0.9, 1.7}) {
        long n = 0, k = 0;
        const float got = Walk(t, beside, &n, &k);
        if (beside == 0) chunks += n, by_terms += k;
        if (BitsOf(got) != BitsOf(want) && !(got != got && want != want)) {
          std::printf("FAIL %s column %d beside %g: %a, not %a\n", kind.name, column, beside, got, want);
          return 1;
        }
      }
    }
    const double share = static_cast<double>(by_terms) / chunks;
    std::printf("%s %d: %.3f by terms\n", kind.name, kind.rows, share);
    if (share > kind.most) {
      std::printf("FAIL %s: too many\n", kind.name);
      return 1;
    }
  }
  std::printf("OK\n");
  return 0;
}
