// Could the column sums of sum_rows (signed terms) be built from runs the way the softmax row
// sum is? While the running sum S of a left-to-right float sum stays in one binade and keeps
// its sign, every step fl(S + t) equals S + rne(t / ulp) * ulp (ties aside): integer adds, so a
// run of such steps is ONE addend. This program measures the best any plan of that kind can do
// by cutting each column into runs with full knowledge of the true running sums, at several
// granularities (a block of g terms is either wholly inside one run or handed to the chain term
// by term), rebuilding the sum from the runs and checking it bit for bit against the serial loop.
// Two kinds of columns: 16384 terms drawn N(0, 1), as the benchmark has them, and the gradients of
// a classifier, p - 1 at the label and p elsewhere, for the softmax p of rows of 1000 N(0, 3^2)
// logits with labels drawn at random, 65536 rows. It prints, per kind, the share of the adds that
// leave the binade or change the sign, the share that are ties, and per granularity the share of a
// column's dependent adds that is left for the chain and the share of blocks that hold.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

static uint32_t Bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}
static int Binade(float s) { return static_cast<int>((Bits(s) >> 23) & 0xff); }  // 0 for zero / subnormal
static bool Negative(float s) { return (Bits(s) >> 31) != 0; }

// One step inside a run: S and the result are normal, same sign, same binade, and t is no tie
// on that binade's grid. Then fl(S + t) - S is the multiple of ulp nearest t.
static bool StepStaysInRun(float s, float t, float r) {
  if (Binade(s) == 0 || Binade(s) == 255 || Binade(r) != Binade(s) || Negative(r) != Negative(s)) return false;
  const double ulp = std::ldexp(1.0, Binade(s) - 127 - 23);
  const double q = static_cast<double>(t) / ulp;
  const double frac = q - std::floor(q);
  return frac != 0.5;
}

const int kGrains[] = {1, 4, 16, 64, 256};
const int kNumGrains = 5;

struct Shares {
  double crossings = 0, ties = 0, left[kNumGrains] = {0}, hold[kNumGrains] = {0};
};

// false: a sum rebuilt from runs is not the serial loop's
static bool AddColumn(const std::vector<float> &t, Shares *shares) {
  const int rows = static_cast<int>(t.size());
  std::vector<float> s(rows + 1);
  std::vector<char> clean(rows);
  // the reference's loop (tensor_cpu-inl.h:221-227): res = src(0, x); res += src(y, x)
  volatile float acc = t[0];
  s[0] = 0.0f;
  s[1] = acc;
  clean[0] = 0;
  for (int y = 1; y < rows; ++y) {
    const float before = acc;
    acc = acc + t[y];
    const float after = acc;
    s[y + 1] = after;
    clean[y] = StepStaysInRun(before, t[y], after) ? 1 : 0;
    const bool crosses = Binade(after) != Binade(before) || Negative(after) != Negative(before);
    shares->crossings += crosses ? 1.0 / rows : 0.0;
    shares->ties += !crosses && !clean[y] ? 1.0 / rows : 0.0;
  }
  for (int gi = 0; gi < kNumGrains; ++gi) {
    const int g = kGrains[gi];
    // a block is clean if every step in it stays in the run that the step before the
    // block was in (first step included: it continues the run)
    size_t addends = 0, holding = 0;
    bool in_run = false;
    int run_binade = -1;
    // rebuild the sum from the plan and compare
    float sum = 0.0f;
    int64_t run_q = 0;
    double run_ulp = 0.0;
    auto close_run = [&]() {
      if (in_run) {
        sum = static_cast<float>(static_cast<double>(sum) + static_cast<double>(run_q) * run_ulp);
        in_run = false;
      }
    };
    for (int b = 0; b < rows; b += g) {
      bool ok = true;
      for (int y = b; y < b + g && y < rows; ++y) ok = ok && clean[y];
      if (ok && in_run && Binade(s[b]) != run_binade) ok = false;
      if (ok) {
        if (!in_run) {
          in_run = true;
          run_binade = Binade(s[b]);
          run_q = 0;
          run_ulp = std::ldexp(1.0, run_binade - 127 - 23);
          ++addends;
        }
        ++holding;
        for (int y = b; y < b + g && y < rows; ++y) {
          run_q += static_cast<int64_t>(std::nearbyint(static_cast<double>(t[y]) / run_ulp));
        }
      } else {
        close_run();
        for (int y = b; y < b + g && y < rows; ++y) {
          volatile float v = sum;
          v = v + t[y];
          sum = v;
          ++addends;
        }
      }
    }
    close_run();
    if (Bits(sum) != Bits(s[rows])) {
      std::printf("MISMATCH grain %d: %a vs %a\n", g, sum, s[rows]);
      return false;
    }
    shares->left[gi] += static_cast<double>(addends) / rows;
    shares->hold[gi] += static_cast<double>(holding) * g / rows;
  }
  return true;
}

static void Report(const char *kind, int columns, int rows, const Shares &s) {
  std::printf("%s: %d columns of %d terms; crossings %.4f ties %.4f; share of the dependent adds left for the chain:",
              kind, columns, rows, s.crossings / columns, s.ties / columns);
  for (int gi = 0; gi < kNumGrains; ++gi) std::printf(" grain %d: %.3f", kGrains[gi], s.left[gi] / columns);
  std::printf("; share of blocks that hold:");
  for (int gi = 0; gi < kNumGrains; ++gi) std::printf(" of %d: %.3f", kGrains[gi], s.hold[gi] / columns);
  std::printf("\n");
}

int main(int argc, char **argv) {
  const int columns = argc > 1 ? std::atoi(argv[1]) : 256;
  std::mt19937 gen(6);
  std::normal_distribution<float> normal(0.0f, 1.0f);
  Shares drawn, gradients;
  {
    std::vector<float> t(16384);
    for (int c = 0; c < columns; ++c) {
      for (float &v : t) v = normal(gen);
      if (!AddColumn(t, &drawn)) return 1;
    }
  }
  const int rows = 65536, classes = 1000, kept = columns < classes ? columns : classes;
  {
    std::vector<std::vector<float>> t(kept, std::vector<float>(rows));
    std::vector<float> p(classes);
    for (int y = 0; y < rows; ++y) {
      float most = -1e30f, sum = 0.0f;
      for (float &v : p) {
        v = 3.0f * normal(gen);
        most = v > most ? v : most;
      }
      for (float &v : p) sum += v = std::exp(v - most);
      const int label = static_cast<int>(gen() % classes);
      for (int c = 0; c < kept; ++c) t[c][y] = c == label ? p[c] / sum - 1.0f : p[c] / sum;
    }
    for (int c = 0; c < kept; ++c) {
      if (!AddColumn(t[c], &gradients)) return 1;
    }
  }
  std::printf("OK ");
  Report("N(0, 1)", columns, 16384, drawn);
  Report("gradients", kept, rows, gradients);
  return 0;
}
