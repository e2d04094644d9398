// Which sums over dense planes go to the kernel that gives a workgroup all planes of a kept index
// (mshadow/hip/kernels/segments_plan.h): the measured shapes, (n, c, len), of either side, and what the kernel relies on
// of every plan.
#include <cstdio>
#include <random>

#include <mshadow/hip/kernels/segments_plan.h>

using mshadow::hip::PlanSegments;
using mshadow::hip::SegmentsPlan;

static const uint32_t kCus = 256;
static int g_wrong = 0;

static void Expect(uint32_t n, uint32_t c, uint64_t len, int least_len, bool use) {
  if (PlanSegments(n, c, len, kCus, least_len).use == use) return;
  ++g_wrong;
  printf("(%u,%u,%llu) %s: expected %d\n", n, c, static_cast<unsigned long long>(len), least_len == 8 ? "half" : "float", use);
}

int main() {
  const int kFloat = 4, kHalf = 8;
  // few kept indices: the split kernel deals their planes out, a workgroup an index would leave the chip idle
  const uint32_t split[][3] = {{512, 16, 784}, {2048, 1, 784}, {2048, 2, 784}, {2048, 4, 784}, {2048, 8, 784}, {2048, 4, 2048}, {1024, 8, 2048},
                               {512, 16, 1500}, {512, 24, 2025}, {1024, 16, 1500}, {2048, 16, 1500}, {256, 32, 1500}, {592, 17, 1521},
                               {950, 13, 1225}, {826, 31, 1936}, {160, 40, 2296}, {64, 64, 12544}};
  for (const auto &s : split) Expect(s[0], s[1], s[2], kFloat, false);
  Expect(2048, 4, 2048, kHalf, false);
  Expect(64, 48, 100, kFloat, false);
  Expect(40, 60, 255, kHalf, false);
  Expect(44, 174, 460, kHalf, true);
  // ... but short planes, or few of them, are done sooner
  const uint32_t own[][3] = {{256, 16, 1024}, {128, 16, 1024}, {256, 32, 1024}, {250, 64, 784}, {1024, 8, 1024}, {2048, 16, 1024}, {2048, 32, 784},
                             {200, 100, 400}, {213, 58, 312}, {60, 190, 1500}, {1024, 8, 196}, {2048, 4, 100}, {32, 64, 196}, {128, 16, 196},
                             {1718, 39, 35}, {1618, 41, 100}, {1024, 128, 100}, {40, 60, 255}};
  for (const auto &s : own) Expect(s[0], s[1], s[2], kFloat, true);
  const uint32_t own_half[][3] = {{512, 16, 784}, {2048, 1, 784}, {826, 31, 1936}, {64, 128, 2048}, {48, 180, 2016}, {512, 16, 2025}, {512, 16, 1500}};
  for (const auto &s : own_half) Expect(s[0], s[1], s[2], kHalf, true);
  // up to a kept index a CU: one round of workgroups with either kernel
  const uint32_t ring[][3] = {{64, 192, 3136}, {64, 192, 1640}, {64, 224, 3136}, {60, 196, 3136}, {48, 240, 3136}, {48, 255, 1640}, {64, 256, 3136}};
  for (const auto &s : ring) {
    Expect(s[0], s[1], s[2], kFloat, false);
    Expect(s[0], s[1], s[2], kHalf, false);
  }
  Expect(48, 192, 3136, kFloat, true);
  Expect(48, 192, 3136, kHalf, false);
  Expect(32, 192, 3136, kFloat, true);
  Expect(32, 192, 3136, kHalf, true);
  // a plane a kept index: the other kernel's waves hide more of a long plane's reads, up to four workgroups a CU
  const uint32_t single[][3] = {{512, 50000, 0}, {512, 40000, 0}, {640, 50000, 0}, {1000, 40000, 0}, {1000, 65500, 0}, {1024, 65535, 0},
                                {512, 32768, 1}, {1000, 32768, 1}, {1024, 24000, 1}, {1100, 50000, 1}, {2048, 50000, 1}, {512, 65536, 1},
                                {700, 400000, 1}, {768, 300, 1}};
  for (const auto &s : single) Expect(1, s[0], s[1], kFloat, s[2] != 0);
  for (const auto &s : single) Expect(1, s[0], s[1], kHalf, true);
  for (const uint32_t c : {64u, 150u, 191u}) Expect(1, c, 200000, kHalf, true);
  // half_t, few kept indices: one round of the split kernel's workgroups is sooner done than long chains ...
  const uint32_t half_split[][3] = {{64, 46, 5000}, {64, 64, 8000}, {40, 46, 3000}, {40, 8, 2048}, {48, 80, 6384}, {81, 50, 6384}, {81, 46, 5000},
                                    {10, 46, 40001}, {16, 64, 31251}, {16, 8, 20001}, {10, 8, 26215}};
  for (const auto &s : half_split) Expect(s[0], s[1], s[2], kHalf, false);
  // ... short ones and two rounds are not
  const uint32_t half_own[][3] = {{64, 46, 1400}, {64, 80, 5000}, {72, 46, 3000}, {81, 64, 8000}, {32, 100, 2048}, {32, 180, 6384}, {128, 46, 8000},
                                  {8, 46, 40001}, {16, 46, 10001}, {16, 180, 20001}, {17, 46, 40001}};
  for (const auto &s : half_own) Expect(s[0], s[1], s[2], kHalf, true);
  // up to sixteen planes of many kept indices
  const uint32_t middling[][4] = {{3, 220, 1000, 0}, {4, 256, 6119, 0}, {3, 280, 1000, 1}, {14, 600, 161, 0}, {9, 600, 161, 0}, {14, 600, 250, 0}, {14, 600, 257, 1}, {8, 600, 250, 1},
                                  {14, 1400, 161, 1}, {15, 8000, 2385, 0}, {13, 4000, 4000, 0}, {14, 2947, 1500, 1}, {10, 12000, 4000, 1}, {15, 906, 881, 1}};
  for (const auto &s : middling) Expect(s[0], s[1], s[2], kFloat, s[3] != 0);
  const uint32_t middling_half[][4] = {{15, 1400, 133, 0}, {9, 1400, 161, 0}, {16, 2947, 250, 0}, {15, 1400, 257, 1}, {5, 600, 400, 1}};
  for (const auto &s : middling_half) Expect(s[0], s[1], s[2], kHalf, s[3] != 0);
  // ... and how they are dealt out: no CU has more waves than need be
  if (PlanSegments(14, 906, 881, kCus, kFloat).kept != 2 || PlanSegments(9, 1024, 2385, kCus, kFloat).kept != 4) ++g_wrong, printf("kept\n");
  // short reductions of many kept indices: ends of planes
  Expect(46, 409, 120, kFloat, false);
  Expect(95, 745, 50, kFloat, false);
  Expect(65, 208, 117, kFloat, true);
  Expect(4, 667, 756, kFloat, false);
  Expect(4, 1928, 637, kFloat, true);
  Expect(38, 1675, 55, kHalf, false);
  Expect(20, 346, 231, kHalf, false);
  Expect(2, 1439, 1005, kHalf, false);
  Expect(112, 335, 56, kHalf, true);
  Expect(22, 422, 198, kHalf, true);
  Expect(43, 835, 1275, kHalf, true);

  std::mt19937 rng(3);
  for (int i = 0; i < 2000000; ++i) {
    const uint32_t n = 1 + (rng() >> (21 + rng() % 11)), c = 1 + (rng() >> (16 + rng() % 16));
    const uint64_t len = 1 + (rng() >> (8 + rng() % 24));
    const int least = i % 2 ? kFloat : kHalf;
    const SegmentsPlan p = PlanSegments(n, c, len, kCus, least);
    if (!p.use) continue;
    const uint32_t size = 16 / least, per_wave = (16 + p.lanes * (4096 / p.lanes + 16)) / size;
    const bool fits = (p.lanes == 8 || p.lanes == 16) && p.waves >= 1 && p.waves <= mshadow::hip::kSegMostWaves &&
                      p.kept >= 1 && p.kept <= p.waves * 64 && n <= 2048 && len >= static_cast<uint64_t>(least) &&
                      (static_cast<uint64_t>(p.waves) * per_wave + static_cast<uint64_t>(p.kept) * n) * size <= 80 * 1024 &&
                      static_cast<uint64_t>((c + p.kept - 1) / p.kept) * p.waves * 64 < (1ull << 32);
    if (!fits && ++g_wrong < 10) printf("plan of (%u,%u,%llu) does not fit the kernel\n", n, c, static_cast<unsigned long long>(len));
  }
  if (g_wrong) return 1;
  printf("OK\n");
  return 0;
}
