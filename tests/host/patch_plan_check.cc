// Which im2col kernel takes patch rows shorter than a pack (csrc/patch_plan.h): a matrix of more workgroups than one
// launch has must be left to the kernel that stages bands of an image.
#include <cstdio>

#include "../../mshadow_amd/csrc/patch_plan.h"

using namespace mshadow_hipk;

static int g_wrong = 0;

static void Fits(int64_t rows, int64_t cols, int ept, bool fits) {
  if (Im2ColPacksFit(rows, cols, ept) == fits) return;
  ++g_wrong;
  printf("%lld x %lld, packs of %d: expected %d\n", static_cast<long long>(rows), static_cast<long long>(cols), ept, fits);
}

int main() {
  const int kFloat = 4, kHalf = 8;
  // 2^24 workgroups of 256 threads are 2^32 threads: a row of the matrix each, and several
  Fits((1 << 24) - 1, 49, kHalf, true);
  Fits(1 << 24, 49, kHalf, false);
  Fits(1900000ll * 9, 49, kHalf, false);
  Fits((1 << 23) - 1, 2049, kHalf, true);
  Fits(1 << 23, 2048, kHalf, true);
  Fits(1 << 23, 2049, kHalf, false);
  Fits(1 << 23, 1024, kFloat, true);
  Fits(1 << 23, 1025, kFloat, false);
  Fits(9, (1ll << 31) - 1, kHalf, true);
  Fits(9, 1ll << 31, kHalf, false);
  if (g_wrong == 0) printf("OK\n");
  return g_wrong != 0;
}
