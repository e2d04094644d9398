/*
 * C ABI, group 3: fixed-function operations on plain (pointer, pitch, shape) arguments.
 * Each entry validates its arguments on the host (a kernel is never launched on shapes
 * it does not cover), picks the kernel variant from shape and alignment, queues it on
 * the caller's stream and reports launch errors. See include/mshadow_hip.h.
 */
#include "abi_common.h"

#include <climits>
#include <mutex>
#include <type_traits>

#include <mshadow/hip/kernels/reduce.h>
#include <mshadow/hip/kernels/reduce_dma.h>
#include <mshadow/hip/kernels/reduce_segments.h>

#include "column_chunk_kernels.h"
#include "patch_kernels.h"
#include "pool_kernels.h"
#include "row_kernels.h"
#include "scratch_slots.h"
#include "softmax_kernels.h"

using namespace mshadow_abi;
using namespace mshadow_hipk;

namespace {

/* minimal evaluators with the Plan interface the kernel templates expect */
template <typename T>
struct RawPlan2D {
  T *p;
  int stride;
  __device__ T &REval(unsigned y, unsigned x) { return p[static_cast<size_t>(y) * stride + x]; }
  __device__ const T &Eval(unsigned y, unsigned x) const {
    return p[static_cast<size_t>(y) * stride + x];
  }
};
template <typename T>
struct RawPlan1D {
  T *p;
  __device__ T &REval(unsigned, unsigned x) { return p[x]; }
  __device__ const T &Eval(unsigned, unsigned x) const { return p[x]; }
};

inline bool Aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <typename F>
int DispatchSaver(int saver, F f) {
  switch (saver) {
    case MSHADOW_HIP_SAVETO: return f(mshadow::sv::saveto());
    case MSHADOW_HIP_PLUSTO: return f(mshadow::sv::plusto());
    case MSHADOW_HIP_MINUSTO: return f(mshadow::sv::minusto());
    case MSHADOW_HIP_MULTO: return f(mshadow::sv::multo());
    case MSHADOW_HIP_DIVTO: return f(mshadow::sv::divto());
    default: return Fail(MSHADOW_HIP_ERR_ARGUMENT, "unknown saver");
  }
}
template <typename F>
int DispatchReducer(int reducer, F f) {
  switch (reducer) {
    case MSHADOW_HIP_SUM: return f(mshadow::red::sum());
    case MSHADOW_HIP_MAX: return f(mshadow::red::maximum());
    case MSHADOW_HIP_MIN: return f(mshadow::red::minimum());
    default: return Fail(MSHADOW_HIP_ERR_ARGUMENT, "unknown reducer");
  }
}

}  // namespace

namespace {
const size_t kPatchLdsBudget = 24 * 1024;  // per workgroup (col2im: every tap's patch rows of a band)
/* input rows staged per workgroup: small bands, many workgroups in different phases per CU
   ((16,64,224,224) 3x3 stride 2: 117 us against 150 us with 40 KB) */
const size_t kIm2ColLdsBudget = 16 * 1024;
/* reductions long enough to fill the LDS ring of the direct-to-LDS kernels that hold a whole
   CU's LDS; shorter ones run kernels of which several share a CU */
const int kDmaMinRows = 6144;
const long long kDmaMinPerKept = 1ll << 16;

int MakePatchGeom(PatchGeom *g, int n, int c, int h, int w, int ky, int kx, int sy, int sx,
                  int dy, int dx, int pad_y, int pad_x) {
  if (n < 0 || c < 0 || h < 0 || w < 0) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "negative shape");
  if (ky < 1 || kx < 1 || sy < 1 || sx < 1 || dy < 1 || dx < 1 || pad_y < 0 || pad_x < 0) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "kernel, stride, dilation must be >= 1, pad >= 0");
  }
  const int hp = h + 2 * pad_y, wp = w + 2 * pad_x;
  if (hp < ky || wp < kx || hp < dy * (ky - 1) + 1 || wp < dx * (kx - 1) + 1) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "image shape smaller than patch size");
  }
  g->n = n; g->c = c; g->h = h; g->w = w;
  g->ky = ky; g->kx = kx; g->sy = sy; g->sx = sx; g->dy = dy; g->dx = dx;
  g->pad_y = pad_y; g->pad_x = pad_x; g->hp = hp; g->wp = wp;
  g->oh = (hp - (dy * (ky - 1) + 1)) / sy + 1;
  g->ow = (wp - (dx * (kx - 1) + 1)) / sx + 1;
  const long long rows = static_cast<long long>(ky) * kx * c;
  const long long cols = static_cast<long long>(n) * g->oh * g->ow;
  if (rows >= (1ll << 31) || cols >= (1ll << 31) ||
      static_cast<long long>(n) * c * h >= (1ll << 31) ||
      static_cast<long long>(n) * c * h * w >= (1ll << 32)) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "too large for 32-bit indices");
  }
  return MSHADOW_HIP_OK;
}

template <typename T>
int Im2Col(T *col, int cstride, const T *img, int istride, const PatchGeom &g, void *stream) {
  const long long rows = static_cast<long long>(g.ky) * g.kx * g.c;
  const long long cols = static_cast<long long>(g.n) * g.oh * g.ow;
  if (rows == 0 || cols == 0) return MSHADOW_HIP_OK;
  if (col == NULL || img == NULL) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "im2col: NULL tensor");
  if (cstride < cols || istride < g.w) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "im2col: pitch smaller than the row");
  }
  const int EPT = 16 / sizeof(T);
  const bool unit_steps = g.sy == 1 && g.sx == 1 && g.dy == 1 && g.dx == 1;
  /* the binary16 3-tap kernel without staging (below) serves this case better */
  const bool three_taps_direct = unit_steps && g.kx == 3 && g.pad_x == 1 && g.ow == g.w &&
                                 g.w % EPT == 0 && istride == g.w && cstride % EPT == 0 &&
                                 Aligned16(col) && Aligned16(img) && cols < (1ll << 31);
  if (three_taps_direct) {
    const uint32_t places = static_cast<uint32_t>(cols / EPT);
    const uint32_t per_block = kPatchBlock * kIm2ColDirectPer;
    const uint32_t chunks = (places + per_block - 1) / per_block;
    const long long pieces = (static_cast<long long>(g.c) * chunks + 7) / 8 * 8;
    const long long direct_blocks = pieces * g.ky;
    if (direct_blocks < (1ll << 31)) {
      LaunchKernelIfFits((Im2ColRow3DirectKernel<T, kIm2ColDirectPer>),
                         dim3(static_cast<unsigned>(direct_blocks)), dim3(kPatchBlock), 0,
                         AsStream(stream), col, cstride, img, g,
                         mshadow::FastDivU32(static_cast<uint32_t>(g.ow / EPT)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.oh)), chunks,
                         mshadow::FastDivU32(chunks));
      return AfterLaunch("im2col");
    }
  }
  /* 3, 5 or 7 taps a row next to one another (4 with a step of two), a step of one or two between patches, patch rows of
     a pack or more: all taps of a tap row from one fetch of the image under them (3x3 stride 2 on
     (32,256,56,56) binary16: 27 us against 41 us with a fetch per tap; 5x5 stride 1 on (32,128,28,28):
     29 against 40 us. Three taps with a step of one keep a fetch per tap: 96 against 100 us on
     (32,256,56,56) without padding) */
  if (g.dx == 1 && (g.sx == 2 || (g.sx == 1 && g.kx >= 5)) &&
      (g.kx == 3 || g.kx == 5 || g.kx == 7 || (g.kx == 4 && g.sx == 2)) && g.ow >= EPT) {
    const long long ppr = (g.ow + EPT - 1) / EPT;
    const long long places = static_cast<long long>(g.n) * g.oh * ppr;
    const uint32_t chunks = static_cast<uint32_t>((places + kPatchBlock - 1) / kPatchBlock);
    const long long pieces = (static_cast<long long>(g.c) * chunks + 7) / 8 * 8;
    const long long blocks = pieces * g.ky;
    if (places + kPatchBlock < (1ll << 31) && blocks < (1ll << 31)) {
#define IM2COL_ROW_TAPS(KX, SX)                                                                       \
  LaunchKernelIfFits((Im2ColRowTapsKernel<T, KX, SX>), dim3(static_cast<unsigned>(blocks)),           \
                     dim3(kPatchBlock), 0, AsStream(stream), col, cstride, img, istride, g,           \
                     mshadow::FastDivU32(static_cast<uint32_t>(ppr)),                                 \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.oh)), chunks,                        \
                     mshadow::FastDivU32(chunks), static_cast<uint32_t>(places))
      if (g.sx == 1) {
        if (g.kx == 5) IM2COL_ROW_TAPS(5, 1);
        else IM2COL_ROW_TAPS(7, 1);
      } else {
        if (g.kx == 3) IM2COL_ROW_TAPS(3, 2);
        else if (g.kx == 4) IM2COL_ROW_TAPS(4, 2);
        else if (g.kx == 5) IM2COL_ROW_TAPS(5, 2);
        else IM2COL_ROW_TAPS(7, 2);
      }
#undef IM2COL_ROW_TAPS
      return AfterLaunch("im2col");
    }
  }
  /* stride 1, dilation 1, patch rows of a pack or more: pack by pack, no staging */
  if (unit_steps && g.ow >= EPT) {
    const long long ppr = (g.ow + EPT - 1) / EPT;
    const long long places = static_cast<long long>(g.n) * g.oh * ppr;
    const uint32_t chunks = static_cast<uint32_t>((places + kPatchBlock - 1) / kPatchBlock);
    const long long pieces = (static_cast<long long>(g.c) * chunks + 7) / 8 * 8;
    const long long blocks = pieces * g.ky * g.kx;
    if (places + kPatchBlock < (1ll << 31) && blocks < (1ll << 31)) {
      LaunchKernelIfFits((Im2ColDirectS1Kernel<T>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kPatchBlock), 0, AsStream(stream), col, cstride, img, istride, g,
                         mshadow::FastDivU32(static_cast<uint32_t>(ppr)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.oh)), chunks,
                         mshadow::FastDivU32(chunks), static_cast<uint32_t>(places));
      return AfterLaunch("im2col");
    }
  }
  /* a step of two between patches (the usual strided convolution): the same, every pack made of
     every second element of two fetched packs (3x3 stride 2 on (32,256,56,56) binary16: 42 us
     against 64 us for the staged kernel below) */
  if (g.sx == 2 && g.ow >= EPT) {
    const long long ppr = (g.ow + EPT - 1) / EPT;
    const long long places = static_cast<long long>(g.n) * g.oh * ppr;
    const uint32_t chunks = static_cast<uint32_t>((places + kPatchBlock - 1) / kPatchBlock);
    const long long pieces = (static_cast<long long>(g.c) * chunks + 7) / 8 * 8;
    const long long blocks = pieces * g.ky * g.kx;
    if (places + kPatchBlock < (1ll << 31) && blocks < (1ll << 31)) {
      LaunchKernelIfFits((Im2ColDirectS2Kernel<T>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kPatchBlock), 0, AsStream(stream), col, cstride, img, istride, g,
                         mshadow::FastDivU32(static_cast<uint32_t>(ppr)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.oh)), chunks,
                         mshadow::FastDivU32(chunks), static_cast<uint32_t>(places));
      return AfterLaunch("im2col");
    }
  }
  /* tiled: padded input rows of a band of patch rows must fit the LDS budget */
  const size_t row_bytes = static_cast<size_t>(g.wp) * sizeof(T);
  const long long max_rows = static_cast<long long>(kIm2ColLdsBudget / row_bytes);
  const long long halo = static_cast<long long>(g.ky - 1) * g.dy + 1;
  long long band = max_rows >= halo ? (max_rows - halo) / g.sy + 1 : 0;
  if (band > g.oh) band = g.oh;
  const long long planes = static_cast<long long>(g.n) * g.c;
  while (band > 8 && planes * ((g.oh + band - 1) / band) < 1024) band = (band + 1) / 2;
  /* patch rows shorter than a pack would be written element by element there */
  const bool short_rows = g.ow < EPT && Im2ColPacksFit(rows, cols, EPT);
  if (band >= 1 && !short_rows) {
    const long long nb = (g.oh + band - 1) / band;
    band = (g.oh + nb - 1) / nb;
    PatchTile t;
    t.band = static_cast<int>(band);
    t.bands = static_cast<int>(nb);
    t.rows_max = static_cast<int>((band - 1) * g.sy + halo);
    t.pitch = g.wp;
    const long long blocks = planes * nb;
    if (blocks >= (1ll << 31)) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "im2col: too many workgroups");
    const size_t lds = static_cast<size_t>(t.rows_max) * row_bytes;
    LaunchKernelIfFits((Im2ColTiledKernel<T, EPT>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kPatchBlock), lds, AsStream(stream), col, cstride, img, istride, g, t);
  } else {
    const long long chunks = (cols + kPatchBlock * EPT - 1) / (kPatchBlock * EPT);
    const long long blocks = Im2ColPackBlocks(rows, cols, EPT);
    if (blocks >= (1ll << 31)) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "im2col: too many workgroups");
    LaunchKernelIfFits((Im2ColKernel<T, EPT>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kPatchBlock), 0, AsStream(stream), col, cstride, img, istride, g,
                       static_cast<unsigned>(chunks), mshadow::FastDivU32(static_cast<uint32_t>(chunks)),
                       mshadow::FastDivU32(static_cast<uint32_t>(g.ow)), mshadow::FastDivU32(static_cast<uint32_t>(g.oh)));
  }
  return AfterLaunch("im2col");
}

template <typename T>
int Col2Im(T *img, int istride, const T *col, int cstride, const PatchGeom &g, void *stream) {
  const long long cols = static_cast<long long>(g.n) * g.oh * g.ow;
  const long long total = static_cast<long long>(g.n) * g.c * g.h * g.w;
  if (total == 0) return MSHADOW_HIP_OK;
  if (col == NULL || img == NULL) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "col2im: NULL tensor");
  if (cstride < cols || istride < g.w) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "col2im: pitch smaller than the row");
  }
  const int EPT = 16 / sizeof(T);
  /* the convolution-backward case on rows of whole aligned packs: nine shifted streams */
  if (sizeof(T) == 2 && g.ky == 3 && g.kx == 3 && g.sy == 1 && g.sx == 1 && g.dy == 1 && g.dx == 1 &&
      g.pad_y == 1 && g.pad_x == 1 && g.w % 8 == 0 && g.w <= 512 && istride % 8 == 0 &&
      cstride % 8 == 0 && Aligned16(img) && Aligned16(col) && total < (1ll << 31) &&
      static_cast<long long>(g.c) * 9 * cstride < (1ll << 40)) {
    RowsGeom rg;
    rg.total_rows = static_cast<uint32_t>(static_cast<long long>(g.n) * g.c * g.h);
    rg.groups = static_cast<uint32_t>(g.w / 8);
    rg.rows_per_wave = 64u / rg.groups;
    rg.div_groups = mshadow::FastDivU32(rg.groups);
    rg.div_h = mshadow::FastDivU32(static_cast<uint32_t>(g.h));
    rg.div_c = mshadow::FastDivU32(static_cast<uint32_t>(g.c));
    const uint32_t waves = (rg.total_rows + rg.rows_per_wave - 1) / rg.rows_per_wave;
    const uint32_t blocks = (waves + kPatchBlock / 64 - 1) / (kPatchBlock / 64);
    LaunchKernelIfFits(Col2ImHalfRows3x3Kernel, dim3(blocks), dim3(kPatchBlock), 0, AsStream(stream),
                       reinterpret_cast<uint16_t *>(img), istride,
                       reinterpret_cast<const uint16_t *>(col), cstride, g, rg);
    return AfterLaunch("col2im");
  }
  /* stride 1, dilation 1, image rows of a pack or more: pack by pack, no staging */
  if (g.sy == 1 && g.sx == 1 && g.dy == 1 && g.dx == 1 && g.w >= EPT) {
    const long long wpk = (g.w + EPT - 1) / EPT;
    const long long packs = static_cast<long long>(g.n) * g.c * g.h * wpk;
    if (packs + kPatchBlock < (1ll << 31) && cols < (1ll << 31)) {
      const unsigned blocks = static_cast<unsigned>((packs + kPatchBlock - 1) / kPatchBlock);
      LaunchKernelIfFits((Col2ImDirectS1Kernel<T>), dim3(blocks), dim3(kPatchBlock), 0, AsStream(stream),
                         img, istride, col, cstride, g, mshadow::FastDivU32(static_cast<uint32_t>(wpk)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.h)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.c)), static_cast<uint32_t>(packs));
      return AfterLaunch("col2im");
    }
  }
  /* strides above 1, image rows of a pack or more: a pixel has few patches, gathered directly */
  if ((g.sy > 1 || g.sx > 1) && g.w >= EPT) {
    const long long wpk = (g.w + EPT - 1) / EPT;
    const long long packs = static_cast<long long>(g.n) * g.c * g.h * wpk;
    if (packs + kPatchBlock < (1ll << 31) && cols < (1ll << 31)) {
      const unsigned blocks = static_cast<unsigned>((packs + kPatchBlock - 1) / kPatchBlock);
      const PatchDivs dv = {mshadow::FastDivU32(static_cast<uint32_t>(g.sy)),
                            mshadow::FastDivU32(static_cast<uint32_t>(g.sx)),
                            mshadow::FastDivU32(static_cast<uint32_t>(g.dy)),
                            mshadow::FastDivU32(static_cast<uint32_t>(g.dx))};
      /* dilation 1 and few patches over a pixel: every load of a thread under way at once */
      const int over_y = (g.ky + g.sy - 1) / g.sy, over_x = (g.kx + g.sx - 1) / g.sx;
      const int over = over_y > over_x ? over_y : over_x;
      if (g.dy == 1 && g.dx == 1 && over <= 4) {
#define COL2IM_FLAT(TY, TX)                                                                                  \
  LaunchKernelIfFits((Col2ImGatherFlatKernel<T, TY, TX>), dim3(blocks), dim3(kPatchBlock), 0, AsStream(stream), \
                     img, istride, col, cstride, g, dv, mshadow::FastDivU32(static_cast<uint32_t>(wpk)),       \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.h)),                                          \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.c)), static_cast<uint32_t>(packs))
        /* a step of two along x: the patches of every second pixel are neighbours in the matrix */
        if (g.sx == 2 && g.ow >= EPT / 2 && over >= 2) {
#define COL2IM_S2(TY, TX)                                                                                    \
  LaunchKernelIfFits((Col2ImGatherS2Kernel<T, TY, TX>), dim3(blocks), dim3(kPatchBlock), 0, AsStream(stream), \
                     img, istride, col, cstride, g, dv, mshadow::FastDivU32(static_cast<uint32_t>(wpk)),       \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.h)),                                          \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.c)), static_cast<uint32_t>(packs))
          if (over == 2) COL2IM_S2(2, 2);
          else if (over == 3) COL2IM_S2(3, 3);
          else COL2IM_S2(4, 4);
#undef COL2IM_S2
          return AfterLaunch("col2im");
        }
        if (over <= 1) COL2IM_FLAT(1, 1);
        else if (over == 2) COL2IM_FLAT(2, 2);
        else if (over == 3) COL2IM_FLAT(3, 3);
        else COL2IM_FLAT(4, 4);
#undef COL2IM_FLAT
        return AfterLaunch("col2im");
      }
      LaunchKernelIfFits((Col2ImGatherKernel<T>), dim3(blocks), dim3(kPatchBlock), 0, AsStream(stream),
                         img, istride, col, cstride, g, dv, mshadow::FastDivU32(static_cast<uint32_t>(wpk)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.h)),
                         mshadow::FastDivU32(static_cast<uint32_t>(g.c)), static_cast<uint32_t>(packs));
      return AfterLaunch("col2im");
    }
  }
  /* image rows shorter than a pack: pixel by pixel (3x3 on (128,256,7,7) binary16 236 us staged) */
  {
    const int over_y = (g.ky + g.sy - 1) / g.sy, over_x = (g.kx + g.sx - 1) / g.sx;
    const int over = over_y > over_x ? over_y : over_x;
    if (g.w < EPT && g.dy == 1 && g.dx == 1 && over <= 5 && total + kPatchBlock < (1ll << 31) && cols < (1ll << 31)) {
      const PatchDivs dv = {mshadow::FastDivU32(static_cast<uint32_t>(g.sy)),
                            mshadow::FastDivU32(static_cast<uint32_t>(g.sx)), mshadow::FastDivU32(1u),
                            mshadow::FastDivU32(1u)};
#define COL2IM_PIXEL(TY, TX)                                                                                       \
  LaunchKernelIfFits((Col2ImPixelKernel<T, TY, TX>),                                                               \
                     dim3(static_cast<unsigned>((total + kPatchBlock - 1) / kPatchBlock)), dim3(kPatchBlock), 0,   \
                     AsStream(stream), img, istride, col, cstride, g, dv,                                          \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.w)), mshadow::FastDivU32(static_cast<uint32_t>(g.h)), \
                     mshadow::FastDivU32(static_cast<uint32_t>(g.n)), static_cast<uint32_t>(total))
      if (over <= 1) COL2IM_PIXEL(1, 1);
      else if (over == 2) COL2IM_PIXEL(2, 2);
      else if (over == 3) COL2IM_PIXEL(3, 3);
      else if (over == 4) COL2IM_PIXEL(4, 4);
      else COL2IM_PIXEL(5, 5);
#undef COL2IM_PIXEL
      return AfterLaunch("col2im");
    }
  }
  /* tiled: per tap, the patch rows a band of image rows touches; all taps must fit */
  const long long taps = static_cast<long long>(g.ky) * g.kx;
  const size_t prow_bytes = static_cast<size_t>(taps) * g.ow * sizeof(T);
  const long long max_prows = static_cast<long long>(kPatchLdsBudget / prow_bytes);
  /* an image band of b rows touches at most (b + span_y - 2) / sy + 2 patch rows */
  const long long span_y = static_cast<long long>(g.dy) * (g.ky - 1) + 1;
  long long band = (max_prows - 2) * g.sy - span_y + 2;
  if (band > g.h) band = g.h;
  const long long planes = static_cast<long long>(g.n) * g.c;
  while (band > 8 && planes * ((g.h + band - 1) / band) < 1024) band = (band + 1) / 2;
  if (band >= 1 && max_prows >= 3) {
    const long long nb = (g.h + band - 1) / band;
    band = (g.h + nb - 1) / nb;
    PatchTile t;
    t.band = static_cast<int>(band);
    t.bands = static_cast<int>(nb);
    t.rows_max = static_cast<int>((band + span_y - 2) / g.sy + 2);
    t.pitch = (t.rows_max * g.ow + EPT - 1) / EPT * EPT;
    const size_t lds = static_cast<size_t>(taps) * t.pitch * sizeof(T);
    const long long blocks = planes * nb;
    if (blocks >= (1ll << 31)) return Fail(MSHADOW_HIP_ERR_ARGUMENT, "col2im: too many workgroups");
    if (g.dy == 1 && g.dx == 1 && g.sy == 1 && g.sx == 1) {
      LaunchKernelIfFits((Col2ImTiledKernel<T, EPT, true>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kPatchBlock), lds, AsStream(stream), img, istride, col, cstride, g, t);
    } else {
      LaunchKernelIfFits((Col2ImTiledKernel<T, EPT, false>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kPatchBlock), lds, AsStream(stream), img, istride, col, cstride, g, t);
    }
  } else {
    unsigned grid = 0;
    int st = mshadow_hip_suggest_grid(static_cast<size_t>(total), kPatchBlock, 8, &grid);
    if (st != MSHADOW_HIP_OK) return st;
    LaunchKernelIfFits((Col2ImKernel<T>), dim3(grid), dim3(kPatchBlock), 0, AsStream(stream), img,
                       istride, col, cstride, g, static_cast<unsigned>(total));
  }
  return AfterLaunch("col2im");
}
struct UnpoolArgs {
  float *dst; int dstride; const float *src; int sstride; const float *pooled; int pstride;
  const float *grad; int gstride; PoolGeom g; int prow_max; unsigned blocks; size_t lds;
  hipStream_t s;
};
#define UNPOOL_ARGS(a) a.dst, a.dstride, a.src, a.sstride, a.pooled, a.pstride, a.grad, a.gstride, a.g, a.prow_max
template <int KY, int KX, int SY, int SX, bool VEC>
void LaunchUnpoolBlock(int reducer, const UnpoolArgs &a, const mshadow::FastDivU32 &div_bw) {
  switch (reducer) {
    case MSHADOW_HIP_SUM:
      LaunchKernelIfFits((UnpoolBlockKernel<MSHADOW_HIP_SUM, KY, KX, SY, SX, VEC>), dim3(a.blocks),
                         dim3(kPoolBlock), a.lds, a.s, UNPOOL_ARGS(a), div_bw);
      break;
    case MSHADOW_HIP_MAX:
      LaunchKernelIfFits((UnpoolBlockKernel<MSHADOW_HIP_MAX, KY, KX, SY, SX, VEC>), dim3(a.blocks),
                         dim3(kPoolBlock), a.lds, a.s, UNPOOL_ARGS(a), div_bw);
      break;
    default:
      LaunchKernelIfFits((UnpoolBlockKernel<MSHADOW_HIP_MIN, KY, KX, SY, SX, VEC>), dim3(a.blocks),
                         dim3(kPoolBlock), a.lds, a.s, UNPOOL_ARGS(a), div_bw);
      break;
  }
}
void LaunchUnpoolGeneric(int reducer, const UnpoolArgs &a) {
  switch (reducer) {
    case MSHADOW_HIP_SUM:
      LaunchKernelIfFits((UnpoolKernel<MSHADOW_HIP_SUM, 0, 0, 0, 0>), dim3(a.blocks), dim3(kPoolBlock),
                         a.lds, a.s, UNPOOL_ARGS(a));
      break;
    case MSHADOW_HIP_MAX:
      LaunchKernelIfFits((UnpoolKernel<MSHADOW_HIP_MAX, 0, 0, 0, 0>), dim3(a.blocks), dim3(kPoolBlock),
                         a.lds, a.s, UNPOOL_ARGS(a));
      break;
    default:
      LaunchKernelIfFits((UnpoolKernel<MSHADOW_HIP_MIN, 0, 0, 0, 0>), dim3(a.blocks), dim3(kPoolBlock),
                         a.lds, a.s, UNPOOL_ARGS(a));
      break;
  }
}
#undef UNPOOL_ARGS


struct GradLaunch {
  float *dst; int dstride; const float *src; int sstride; const float *label; int cols;
  unsigned chunks; GradParams gp; unsigned blocks; hipStream_t s;
};
template <bool VEC>
void LaunchGrad(int flags, const GradLaunch &g) {
#define GRAD2D(FLAGS)                                                                         \
  LaunchKernelIfFits((SoftmaxGradKernel<VEC, FLAGS>), dim3(g.blocks), dim3(kGradBlock), 0, g.s, \
                     g.dst, g.dstride, g.src, g.sstride, g.label, g.cols, g.chunks, g.gp)
  switch (flags) {
    case 0: GRAD2D(0); break;
    case 1: GRAD2D(1); break;
    case 2: GRAD2D(2); break;
    default: GRAD2D(3); break;
  }
#undef GRAD2D
}


}  // namespace


template <int OP>
static int LaunchRowsByIndex(float *dst, int dstride, int k_rows, const void *rows_of,
                             const void *from_of, int index_is_int, int n_index, const float *src,
                             int sstride, int cols, void *stream, const char *what) {
  unsigned grid = 0;
  int rows_per_wave = 0;
  mshadow::hip::RowsByIndexGrid(k_rows, &grid, &rows_per_wave);
  const bool vec = Aligned16(dst) && Aligned16(src) && dstride % 4 == 0 && sstride % 4 == 0 &&
                   cols % 4 == 0;
  hipStream_t s = AsStream(stream);
#define ROWS_LAUNCH(ITYPE, VEC)                                                               \
  LaunchKernelIfFits((RowsByIndexKernel<ITYPE, float, OP, VEC>), dim3(grid), dim3(kTakeBlock), 0, \
                     s, dst, dstride, k_rows, rows_per_wave, static_cast<const ITYPE *>(rows_of), \
                     static_cast<const ITYPE *>(from_of), n_index, src, sstride, cols)
  if (index_is_int) {
    if (vec) ROWS_LAUNCH(int32_t, true); else ROWS_LAUNCH(int32_t, false);
  } else {
    if (vec) ROWS_LAUNCH(float, true); else ROWS_LAUNCH(float, false);
  }
#undef ROWS_LAUNCH
  return AfterLaunch(what);
}

namespace {
/*! \brief rows (or kept indices) of one launch that gives each `threads` threads at most: with 2^32
 *  threads or more along an axis workgroups are dropped, and no error says so */
int RowsOfLaunch(unsigned threads) {
  const unsigned long long most = (0xffffffffull - 1024u) / threads;  // the last workgroup may not be full
  return most < static_cast<unsigned long long>(INT_MAX) ? static_cast<int>(most) : INT_MAX;
}
/*! \brief threads a row of the kernels below takes, where there are many rows */
unsigned SoftmaxThreadsPerRow(int cols) { return cols <= 32 ? 1u : cols <= 256 ? 32u : cols <= 3072 ? 64u : 1024u; }

/*! \brief rows that a thread, a part of a wave or a wave takes; false: longer ones, which take a
 *  workgroup */
template <bool TERMS_GIVEN>
bool LaunchShortSoftmax(float *dst, int dstride, const float *src, int sstride, int rows, int cols,
                        hipStream_t s) {
#define SHORT_THREAD(CMAX) \
  LaunchKernelIfFits((SoftmaxThreadRowKernel<CMAX, TERMS_GIVEN>), dim3((rows + 255) / 256), dim3(256), 0, s, \
                     dst, dstride, src, sstride, rows, cols)
  /* rows that neither start nor end with a pack share cache lines with their neighbours */
  const bool whole = cols % 4 == 0 && dstride % 4 == 0 && sstride % 4 == 0 && Aligned16(dst) && Aligned16(src);
  /* ... and stream all the same where the rows, in and out, are about what L2 holds: up to 140 columns, 13 to 30 MB (us,
     ordinary accesses and streaming ones: 20000 x 127 10.6 and 10.1, 30000 x 75 11.0 and 10.4, 20000 x 129 13.9 and 13.1;
     but 9000 x 127 6.8 and 7.2, 40000 x 127 15.8 and 18.0, 20000 x 199 16.6 and 17.1) */
  const long long in_and_out = 8ll * rows * cols;
  const bool streams = whole || (cols <= 140 && in_and_out >= 13000000 && in_and_out <= 30000000);
#define SHORT_PART_AS(LANES, N, WHOLE) \
  LaunchKernelIfFits((SoftmaxPartWaveKernel<LANES, N, TERMS_GIVEN, WHOLE>), dim3((rows + 256 / LANES - 1) / (256 / LANES)), \
                     dim3(256), 0, s, dst, dstride, src, sstride, rows, cols)
#define SHORT_PART(LANES, N) do { if (streams) SHORT_PART_AS(LANES, N, true); else SHORT_PART_AS(LANES, N, false); } while (0)
#define WAVE_SLABS(SLABS) \
  LaunchKernelIfFits((SoftmaxWaveSlabsKernel<SLABS, TERMS_GIVEN>), dim3((rows + 3) / 4), dim3(256), 0, s, dst, \
                     dstride, src, sstride, rows, cols)
  const int cus = mshadow_abi::ComputeUnits();
  /* Four or two rows side by side in a wave are fewer instructions, a wave to itself brings a row to
     its end sooner: 4000 rows of 64 columns 3.8 us a wave each, 4.9 us in quarters, of 200 5.5 and
     6.8 us, 16000 of 200 11.2 and 12.3 us; 131072 rows of 128 56 and 35 us, of 193 69 and 63 us */
  const bool few = rows <= (cols <= 128 ? 16 : 64) * cus;
  /* not more than three loads of columns that are not there: each is a pass of its own over 64 cache lines
     (300 / 50000 rows of 17 columns: with 15 of them 6.1 / 9.1 us, with three 5.0 / 7.9) */
  if (cols <= 8) SHORT_THREAD(8);
  else if (cols <= 12) SHORT_THREAD(12);
  else if (cols <= 16) SHORT_THREAD(16);
  else if (cols <= 20) SHORT_THREAD(20);
  else if (cols <= 24) SHORT_THREAD(24);
  else if (cols <= 28) SHORT_THREAD(28);
  else if (cols <= 32) SHORT_THREAD(32);
  else if (cols <= 256 && few) WAVE_SLABS(1);
  else if (cols <= 64) SHORT_PART(16, 4);
  else if (cols <= 128) SHORT_PART(16, 8);
  else if (cols <= 256) SHORT_PART(32, 8);
  /* A wave per row for any number of rows of up to 512 columns, and for many of up to 3072: from 6 rows a CU on, above
     2048 columns from 4. In us, a workgroup a row and a wave: 100 rows of 500 columns 5.6 and 5.0; of 1000 columns 1024
     rows 7.4 and 7.3, 3000 12.7 and 9.7, 65536 174 and 90; 1024 / 1536 / 2304 rows of 1200 8.6 and 9.0, 10.2 and 9.9,
     13.0 and 11.0, of 2048 9.4 and 9.7, 10.9 and 10.6, 14.1 and 11.9, of 2300 11.7 and 10.9, 13.9 and 12.0, 18.0 and 13.6,
     of 3072 12.1 and 11.9, 14.4 and 13.2, 18.4 and 15.3; 8000 rows of 3072 43.5 and 39.4; 600 of 2688 10.6 and 10.9.
     The row sums alone from 6 rows a CU on at all lengths. */
  else if (cols <= 512) WAVE_SLABS(2);
  else if (cols > 3072 || rows < (cols > 2048 && !TERMS_GIVEN ? 4 : 6) * cus) return false;
  else if (cols <= 1024) WAVE_SLABS(4);
  else if (cols <= 2048) WAVE_SLABS(8);
  else if (cols <= 2560 && !TERMS_GIVEN) WAVE_SLABS(10);
  else WAVE_SLABS(12);
#undef SHORT_THREAD
#undef SHORT_PART
#undef SHORT_PART_AS
#undef WAVE_SLABS
  return true;
}
}  // namespace

/* Scratch memory of the split KeepHighDim reduction (kernels/reduce_dma.h): the inner results of
   a launch and the counter that tells the last workgroup. It is part of the library's image
   - a file-scope device array, one copy per GPU, nothing is allocated at run time - and is
   handed out per stream: launches on one stream run one after the other, so a stream's slot is
   never in use twice; a ninth stream on one GPU, or a launch with more inner results than a
   slot holds, gets none and its reduction runs the one-workgroup-per-kept-index kernel. */
namespace {
const int kReduceScratchSlots = 8;
const size_t kReduceScratchWords = 1u << 16;
struct ReduceScratchSlot {
  uint32_t partial[kReduceScratchWords];
  uint32_t counter[mshadow::hip::kSplitCounterWords];  // zero between launches
};
static __device__ __align__(256) ReduceScratchSlot g_reduce_scratch[kReduceScratchSlots];

struct ReduceScratchTable {
  std::mutex mu;
  ReduceScratchSlot *base[mshadow_abi::kScratchDevices];
  mshadow_abi::ScratchSlots<kReduceScratchSlots> slots;
};
ReduceScratchTable &ScratchTable() {
  static ReduceScratchTable t = {};
  return t;
}
}  // namespace

/* Scratch memory of the column sums by chunks (column_chunk_kernels.h): like the above a part of the
   image, a slot per stream that has asked for one, which keeps it until it is destroyed. A call is three launches that
   pass their results on in it, so the lock is held while they are queued: two threads that share a
   stream must not come between each other's. */
namespace {
const int kColumnScratchSlots = 4;
static __device__ __align__(256) ColumnChunkScratch g_column_scratch[kColumnScratchSlots];

struct ColumnScratchTable {
  std::mutex mu;
  ColumnChunkScratch *base[mshadow_abi::kScratchDevices];
  mshadow_abi::ScratchSlots<kColumnScratchSlots> slots;

  /* where the slots of the current device are, looked up once; mu is held */
  void Resolve(int dev) {
    if (base[dev] != NULL) return;
    void *p = NULL;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_column_scratch)) == hipSuccess) {
      base[dev] = static_cast<ColumnChunkScratch *>(p);
    } else {
      (void)hipGetLastError();
    }
  }
  /* the caller's slot on the current device, NULL where there is none to be had; mu is held */
  ColumnChunkScratch *Slot(void *stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= mshadow_abi::kScratchDevices) {
      (void)hipGetLastError();
      return NULL;
    }
    Resolve(dev);
    if (base[dev] == NULL) return NULL;
    const int slot = slots.Take(dev, stream);
    return slot < 0 ? NULL : base[dev] + slot;
  }
};
ColumnScratchTable &ColumnTable() {
  static ColumnScratchTable t = {};
  return t;
}

/* A recorded launch may be replayed on any stream, beside the one whose slot it would use; and the handle of the
   stream per thread is every thread's. */
bool HasNoSlot(hipStream_t s) {
  if (s == hipStreamPerThread) return true;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

/* whether the sums of the columns were queued, by chunks of their rows */
template <typename Saver>
bool LaunchColumnChunks(float *dst, const float *src, uint32_t stride, uint32_t rows, uint32_t cols, float scale,
                        hipStream_t s) {
  const uint32_t cus = mshadow_abi::ComputeUnits();
  if (!ColumnChunksAreSooner(rows, cols, cus) || HasNoSlot(s)) return false;
  ColumnScratchTable &t = ColumnTable();
  std::lock_guard<std::mutex> lock(t.mu);
  ColumnChunkScratch *w = t.Slot(s);
  if (w == NULL) return false;
  const uint32_t band = ChunkBandRows(rows, cols);
  for (uint32_t row0 = 0; row0 < rows; row0 += band) {
    ChunkShape g = MakeChunkShape(rows - row0 < band ? rows - row0 : band, cols, stride, cus);
    g.begun = row0 != 0;
    g.more = g.rows < rows - row0;
    const float *from = src + static_cast<size_t>(row0) * stride;
    const dim3 grid(g.groups * g.tiles), block(kChunkWaves * 64), columns(g.strips + cols), walk((1 + kWalkLoaders) * 64);
    LaunchKernelIfFits(ColumnChunkSumsKernel, grid, block, 0, s, from, g, w->before, w->group, w->bare);
    LaunchKernelIfFits(ColumnChunkMapsKernel, grid, block, 0, s, from, g, w->before, w->group, w->map, w->copy, w->bare,
                       w->carry);
#define WALK(AT_ONCE, RING)                                                                                             \
  LaunchKernelIfFits((ColumnChunkWalkKernel<Saver, AT_ONCE, RING>), columns, walk, 0, s, dst, from, g, w->map, w->copy, \
                     w->bare, w->carry, scale)
    if (cols <= ColumnsOfWideWalk(cus)) WALK(16, StripRingOfTwo);
    else WALK(4, StripRingOfSix);
#undef WALK
  }
  return true;
}
}  // namespace

namespace mshadow_abi {
bool HasReduceScratch(void *stream) {
  {
    ColumnScratchTable &c = ColumnTable();
    std::lock_guard<std::mutex> lock(c.mu);
    if (c.slots.Has(stream)) return true;
  }
  ReduceScratchTable &t = ScratchTable();
  std::lock_guard<std::mutex> lock(t.mu);
  return t.slots.Has(stream);
}
void ReleaseReduceScratch(void *stream, bool done) {
  {
    ColumnScratchTable &c = ColumnTable();
    std::lock_guard<std::mutex> lock(c.mu);
    c.slots.Release(stream, done);
  }
  ReduceScratchTable &t = ScratchTable();
  std::lock_guard<std::mutex> lock(t.mu);
  t.slots.Release(stream, done);
}
/* called when a device is selected: where the scratch arrays live on that device is looked up
   then, not inside the first reduction that wants a slot (which may be being recorded, or queued while
   the same thread records another stream) */
void ResolveReduceScratch() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchDevices) {
    (void)hipGetLastError();
    return;
  }
  ReduceScratchTable &t = ScratchTable();
  std::lock_guard<std::mutex> lock(t.mu);
  if (t.base[dev] == NULL) {
    void *p = NULL;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_reduce_scratch)) == hipSuccess) {
      t.base[dev] = static_cast<ReduceScratchSlot *>(p);
    } else {
      (void)hipGetLastError();
    }
  }
  ColumnScratchTable &c = ColumnTable();
  std::lock_guard<std::mutex> column_lock(c.mu);
  c.Resolve(dev);
}
}  // namespace mshadow_abi

extern "C" int mshadow_hip_reduce_scratch(void *stream, size_t words, uint32_t **partial,
                                          uint32_t **counter) {
  ABI_REQUIRE(partial != NULL && counter != NULL, "NULL result");
  *partial = NULL;
  *counter = NULL;
  if (words > kReduceScratchWords) return MSHADOW_HIP_OK;
  int dev = 0;
  ABI_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kScratchDevices) return MSHADOW_HIP_OK;
  ReduceScratchTable &t = ScratchTable();
  std::lock_guard<std::mutex> lock(t.mu);
  if (t.base[dev] == NULL) {
    /* the array's name is a host-side stand-in; this is its address on the current device */
    void *p = NULL;
    ABI_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(g_reduce_scratch)));
    t.base[dev] = static_cast<ReduceScratchSlot *>(p);
  }
  const int slot = t.slots.Take(dev, stream);
  if (slot < 0) return MSHADOW_HIP_OK;
  *partial = t.base[dev][slot].partial;
  *counter = t.base[dev][slot].counter;
  return MSHADOW_HIP_OK;
}

extern "C" {

/* ------------------------------------------------------------------ softmax */

int mshadow_hip_softmax_f32(float *dst, int dstride, const float *src, int sstride, int rows,
                            int cols, void *stream) {
  ABI_REQUIRE(rows >= 0 && cols >= 0, "negative shape");
  if (rows == 0 || cols == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= cols && sstride >= cols, "pitch smaller than the row");
  const int most = RowsOfLaunch(SoftmaxThreadsPerRow(cols));
  if (rows > most) {
    for (long long row = 0; row < rows; row += most) {
      const int st = mshadow_hip_softmax_f32(dst + row * dstride, dstride, src + row * sstride, sstride,
                                             rows - row < most ? static_cast<int>(rows - row) : most, cols, stream);
      if (st != MSHADOW_HIP_OK) return st;
    }
    return MSHADOW_HIP_OK;
  }
  hipStream_t s = AsStream(stream);
  if (LaunchShortSoftmax<false>(dst, dstride, src, sstride, rows, cols, s)) return AfterLaunch("softmax");
  /* 16-byte packs wherever the rows start and whatever their length (the accesses need no
     alignment; a row's last, partial pack is loaded as its last four columns and stored element by element) */
#define SOFTMAX_LAUNCH(T, S, V) \
  LaunchKernelIfFits((SoftmaxRowKernel<T, S, V, false>), dim3(rows), dim3(T), 0, s, dst, dstride, \
                     src, sstride, cols)
#define SOFTMAX_LAUNCH_LDS(T, S, L) \
  LaunchKernelIfFits((SoftmaxRowKernel<T, S, 4, false, 4, L>), dim3(rows), dim3(T), 0, s, dst, dstride, \
                     src, sstride, cols)
  const int cus = mshadow_abi::ComputeUnits();
  /* Up to two rows a CU: the CU has the row to itself, or nearly, and what counts is how soon the row is
     through, so it gets two to four times the waves (100 rows of 3000 / 7000 / 30000: 6.6 / 8.2 / 19.5
     against 8.3 / 11.0 / 21.6 us, 500 rows 9.8 / 13.2 / 36.4 against 9.9 / 14.7 / 38.3; 1000 rows are
     slower that way, 15.6 / 20.6 against 11.8 / 18.0). */
  if (rows <= 2 * cus && cols > 1024 && cols <= 32768) {
    if (cols <= 2048) SOFTMAX_LAUNCH(512, 1, 4);
    else if (cols <= 4096) SOFTMAX_LAUNCH(1024, 1, 4);
    else if (cols <= 8192) SOFTMAX_LAUNCH(1024, 2, 4);
    else if (cols <= 16384) SOFTMAX_LAUNCH(1024, 4, 4);
    else SOFTMAX_LAUNCH(1024, 8, 4);
  }
  else if (cols <= 1024) SOFTMAX_LAUNCH(256, 1, 4);
  else if (cols <= 2048) SOFTMAX_LAUNCH(256, 2, 4);
  else if (cols <= 4096) SOFTMAX_LAUNCH(256, 4, 4);
  else if (cols <= 8192) SOFTMAX_LAUNCH(256, 8, 4);
  else if (cols <= 16384) SOFTMAX_LAUNCH(512, 8, 4);
  else if (cols <= 32768) SOFTMAX_LAUNCH(512, 16, 4);
  /* longer rows, part of each in LDS: up to 51200 columns two rows share a CU still (2048 x 50257: 206 us,
     alone in its registers 264), from 65537 on a row that has the CU to itself stays on the chip
     (44 x 110032: 48 us, in stretches 77; 1000 x 80000: 179 us, 256; 2048 x 100000: 525 us, 636) */
  else if (cols <= 51200 && rows > cus) SOFTMAX_LAUNCH_LDS(512, 18, 7);
  else if (cols <= 65536) SOFTMAX_LAUNCH(1024, 16, 4);
  else if (cols <= 81920) SOFTMAX_LAUNCH_LDS(1024, 16, 4);
  /* ... but for one to two rows a CU, which stretches take two at a time (512 x 90000: 142 us, 155) */
  else if (cols <= 110592 && (rows <= cus || rows > 2 * cus)) SOFTMAX_LAUNCH_LDS(1024, 19, 8);
  /* longer ones yet: stretches of 32768 columns on 512 threads, two rows to a CU ((512,128000): 183 us
     against 271 us with stretches of 65536 on 1024 threads) */
  else if (cols > INT_MAX - 32768) {
    return Fail(MSHADOW_HIP_ERR_ARGUMENT, "softmax: row too long for 32-bit column counts");
  } else if (rows > cus) {
    LaunchKernelIfFits((SoftmaxStretchRowKernel<512, 16, false, 4>), dim3(rows), dim3(512), 0, s, dst,
                       dstride, src, sstride, cols);
  } else {
    LaunchKernelIfFits((SoftmaxStretchRowKernel<512, 16, false, 2>), dim3(rows), dim3(512), 0, s, dst,
                       dstride, src, sstride, cols);
  }
#undef SOFTMAX_LAUNCH_LDS
#undef SOFTMAX_LAUNCH
  return AfterLaunch("softmax");
}

int mshadow_hip_softmax_rowsum_f32(float *sums, const float *terms, int tstride, int rows,
                                   int cols, void *stream) {
  ABI_REQUIRE(rows >= 0 && cols >= 0, "negative shape");
  if (rows == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(sums != NULL && (terms != NULL || cols == 0), "NULL tensor");
  ABI_REQUIRE(tstride >= cols, "pitch smaller than the row");
  const int most = RowsOfLaunch(SoftmaxThreadsPerRow(cols));
  if (rows > most) {
    for (long long row = 0; row < rows; row += most) {
      const int st = mshadow_hip_softmax_rowsum_f32(sums + row, terms + row * tstride, tstride,
                                                    rows - row < most ? static_cast<int>(rows - row) : most, cols, stream);
      if (st != MSHADOW_HIP_OK) return st;
    }
    return MSHADOW_HIP_OK;
  }
  hipStream_t s = AsStream(stream);
  if (LaunchShortSoftmax<true>(sums, 0, terms, tstride, rows, cols, s)) return AfterLaunch("softmax_rowsum");
  const bool vec = Aligned16(terms) && tstride % 4 == 0 && cols % 4 == 0;
  /* rows longer than a workgroup's registers hold: stretch by stretch, at any alignment */
  if (cols > 65536 || (!vec && cols > 32768)) {
    ABI_REQUIRE(cols <= INT_MAX - 32768, "row too long for 32-bit column counts");
    LaunchKernelIfFits((SoftmaxStretchRowKernel<512, 16, true, 2>), dim3(rows), dim3(512), 0, s, sums, 0,
                       terms, tstride, cols);
    return AfterLaunch("softmax_rowsum");
  }
#define ROWSUM_LAUNCH(T, S, V) \
  LaunchKernelIfFits((SoftmaxRowKernel<T, S, V, true>), dim3(rows), dim3(T), 0, s, sums, 0, terms, \
                     tstride, cols)
  if (vec) {
    if (cols > 8192 && cols <= 16384 && rows >= 16 * mshadow_abi::ComputeUnits()) ROWSUM_LAUNCH(256, 16, 4);
    else if (cols <= 1024) ROWSUM_LAUNCH(256, 1, 4);
    else if (cols <= 2048) ROWSUM_LAUNCH(256, 2, 4);
    else if (cols <= 4096) ROWSUM_LAUNCH(256, 4, 4);
    else if (cols <= 8192) ROWSUM_LAUNCH(256, 8, 4);
    else if (cols <= 16384) ROWSUM_LAUNCH(512, 8, 4);
    else if (cols <= 32768) ROWSUM_LAUNCH(512, 16, 4);
    else ROWSUM_LAUNCH(1024, 16, 4);
  } else {
    if (cols <= 1024) ROWSUM_LAUNCH(256, 4, 1);
    else if (cols <= 4096) ROWSUM_LAUNCH(256, 16, 1);
    else if (cols <= 16384) ROWSUM_LAUNCH(1024, 16, 1);
    else ROWSUM_LAUNCH(1024, 32, 1);
  }
#undef ROWSUM_LAUNCH
  return AfterLaunch("softmax_rowsum");
}

int mshadow_hip_softmax_grad_ex_f32(float *dst, int dstride, const float *src, int sstride,
                                    const float *label, int rows, int cols, int flags,
                                    float ignore_label, float alpha, void *stream) {
  ABI_REQUIRE(rows >= 0 && cols >= 0, "negative shape");
  ABI_REQUIRE(flags >= 0 && flags <= 3, "unknown gradient flags");
  if (rows == 0 || cols == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL && label != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= cols && sstride >= cols, "pitch smaller than the row");
  const int per_block = kGradBlock * kGradPacks * 4;
  const unsigned chunks = (cols + per_block - 1) / per_block;
  const unsigned long long blocks = static_cast<unsigned long long>(rows) * chunks;
  ABI_REQUIRE(blocks < (1ull << 31), "too many workgroups");
  /* short rows go several to a workgroup, a pack a thread */
  const int ppr = (cols + 3) / 4, rows_per_block = cols <= 512 ? kGradBlock / ppr : 1;
  const int most = RowsOfLaunch((static_cast<unsigned>(kGradBlock) * chunks - 1) / rows_per_block + 1);
  if (rows > most) {
    for (long long row = 0; row < rows; row += most) {
      const int st = mshadow_hip_softmax_grad_ex_f32(dst + row * dstride, dstride, src + row * sstride, sstride, label + row,
                                                     rows - row < most ? static_cast<int>(rows - row) : most, cols, flags,
                                                     ignore_label, alpha, stream);
      if (st != MSHADOW_HIP_OK) return st;
    }
    return MSHADOW_HIP_OK;
  }
  /* alpha / (classes - 1) with the count converted from unsigned, as the reference writes it */
  const GradParams gp = {static_cast<int>(ignore_label), alpha,
                         alpha / static_cast<float>(static_cast<unsigned>(cols - 1))};
  if (cols <= 512) {
    const unsigned grid = static_cast<unsigned>((rows + rows_per_block - 1) / rows_per_block);
    const mshadow::FastDivU32 div_ppr(static_cast<uint32_t>(ppr));
#define GRAD_SHORT(FLAGS)                                                                            \
  LaunchKernelIfFits((SoftmaxGradShortRowsKernel<FLAGS>), dim3(grid), dim3(kGradBlock), 0, AsStream(stream), \
                     dst, dstride, src, sstride, label, rows, cols, rows_per_block, div_ppr, gp)
    switch (flags) {
      case 0: GRAD_SHORT(0); break;
      case 1: GRAD_SHORT(1); break;
      case 2: GRAD_SHORT(2); break;
      default: GRAD_SHORT(3); break;
    }
#undef GRAD_SHORT
    return AfterLaunch("softmax_grad");
  }
  GradLaunch gl = {dst, dstride, src, sstride, label, cols, chunks, gp,
                   static_cast<unsigned>(blocks), AsStream(stream)};
  LaunchGrad<true>(flags, gl);   // 16-byte packs wherever the rows start (no alignment needed)
  return AfterLaunch("softmax_grad");
}

int mshadow_hip_softmax_grad_f32(float *dst, int dstride, const float *src, int sstride,
                                 const float *label, int rows, int cols, void *stream) {
  return mshadow_hip_softmax_grad_ex_f32(dst, dstride, src, sstride, label, rows, cols, 0, 0.0f,
                                         0.0f, stream);
}

int mshadow_hip_softmax3d_f32(float *dst, int dstride, const float *src, int sstride, int d0,
                              int d1, int d2, void *stream) {
  ABI_REQUIRE(d0 >= 0 && d1 >= 0 && d2 >= 0, "negative shape");
  if (d0 == 0 || d1 == 0 || d2 == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= d2 && sstride >= d2, "pitch smaller than the row");
  ABI_REQUIRE(static_cast<long long>(d0) * d2 < (1ll << 31) &&
                  static_cast<long long>(d0) * d1 < (1ll << 31),
              "too large for 32-bit indices");
  const mshadow::FastDivU32 div_d2s(static_cast<uint32_t>(d2));
  const unsigned pairs = static_cast<unsigned>(d0) * d2;
  const unsigned one_each = (pairs + kSoftmax3dBlock - 1) / kSoftmax3dBlock;
  if (d1 <= 8) {
    LaunchKernelIfFits((Softmax3dSmallKernel<8>), dim3(one_each), dim3(kSoftmax3dBlock), 0,
                       AsStream(stream), dst, dstride, src, sstride, d0, d1, d2, div_d2s);
    return AfterLaunch("softmax3d");
  }
  if (d1 <= 32) {
    LaunchKernelIfFits((Softmax3dSmallKernel<32>), dim3(one_each), dim3(kSoftmax3dBlock), 0,
                       AsStream(stream), dst, dstride, src, sstride, d0, d1, d2, div_d2s);
    return AfterLaunch("softmax3d");
  }
  unsigned grid = 0;
  int st = mshadow_hip_suggest_grid(static_cast<size_t>(d0) * d2, kSoftmax3dBlock, 8, &grid);
  if (st != MSHADOW_HIP_OK) return st;
  LaunchKernelIfFits(Softmax3dKernel, dim3(grid), dim3(kSoftmax3dBlock), 0, AsStream(stream), dst,
                     dstride, src, sstride, d0, d1, d2,
                     mshadow::FastDivU32(static_cast<uint32_t>(d2)));
  return AfterLaunch("softmax3d");
}

int mshadow_hip_softmax3d_grad_f32(float *dst, int dstride, const float *src, int sstride,
                                   const float *label, int lstride, int d0, int d1, int d2,
                                   int flags, float ignore_label, float alpha, void *stream) {
  ABI_REQUIRE(d0 >= 0 && d1 >= 0 && d2 >= 0, "negative shape");
  ABI_REQUIRE(flags >= 0 && flags <= 3, "unknown gradient flags");
  if (d0 == 0 || d1 == 0 || d2 == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL && label != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= d2 && sstride >= d2 && lstride >= d2, "pitch smaller than the row");
  ABI_REQUIRE(static_cast<long long>(d0) * d1 * d2 < (1ll << 31), "too large for 32-bit indices");
  unsigned grid = 0;
  int st = mshadow_hip_suggest_grid(static_cast<size_t>(d0) * d1 * d2, kSoftmax3dBlock, 8, &grid);
  if (st != MSHADOW_HIP_OK) return st;
  const GradParams gp = {static_cast<int>(ignore_label), alpha,
                         alpha / static_cast<float>(static_cast<unsigned>(d1 - 1))};
  const mshadow::FastDivU32 div_d2(static_cast<uint32_t>(d2)), div_d1(static_cast<uint32_t>(d1));
  const bool vec = d2 % 4 == 0 && dstride % 4 == 0 && sstride % 4 == 0 && lstride % 4 == 0 &&
                   Aligned16(dst) && Aligned16(src) && Aligned16(label);
  if (vec) {
    const unsigned packs = static_cast<unsigned>(d0) * d1 * (d2 / 4);
    const unsigned vgrid = (packs + kSoftmax3dBlock - 1) / kSoftmax3dBlock;
    const mshadow::FastDivU32 div_q2(static_cast<uint32_t>(d2 / 4));
#define GRAD3DV(FLAGS)                                                                         \
  LaunchKernelIfFits((Softmax3dGradVecKernel<FLAGS>), dim3(vgrid), dim3(kSoftmax3dBlock), 0,   \
                     AsStream(stream), dst, dstride, src, sstride, label, lstride, d0, d1, d2, \
                     div_q2, div_d1, gp)
    switch (flags) {
      case 0: GRAD3DV(0); break;
      case 1: GRAD3DV(1); break;
      case 2: GRAD3DV(2); break;
      default: GRAD3DV(3); break;
    }
#undef GRAD3DV
    return AfterLaunch("softmax3d_grad");
  }
#define GRAD3D(FLAGS)                                                                          \
  LaunchKernelIfFits((Softmax3dGradKernel<FLAGS>), dim3(grid), dim3(kSoftmax3dBlock), 0,       \
                     AsStream(stream), dst, dstride, src, sstride, label, lstride, d0, d1, d2, \
                     div_d2, div_d1, gp)
  switch (flags) {
    case 0: GRAD3D(0); break;
    case 1: GRAD3D(1); break;
    case 2: GRAD3D(2); break;
    default: GRAD3D(3); break;
  }
#undef GRAD3D
  return AfterLaunch("softmax3d_grad");
}

static int RowOpCheck(const float *dst, int dstride, int k_rows, const void *index, int n_index,
                      const float *src, int sstride, int cols) {
  ABI_REQUIRE(k_rows >= 0 && n_index >= 0 && cols >= 0, "negative shape");
  if (k_rows == 0 || n_index == 0 || cols == 0) return -1;  // nothing to do
  ABI_REQUIRE(dst != NULL && src != NULL && index != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= cols && sstride >= cols, "pitch smaller than the row");
  return MSHADOW_HIP_OK;
}

int mshadow_hip_add_take_grad_f32(float *dst, int dstride, int k_rows, const void *index,
                                  int index_is_int, int n_index, const float *src, int sstride,
                                  int cols, void *stream) {
  const int chk = RowOpCheck(dst, dstride, k_rows, index, n_index, src, sstride, cols);
  if (chk != MSHADOW_HIP_OK) return chk < 0 ? MSHADOW_HIP_OK : chk;
  return LaunchRowsByIndex<kTakeGrad>(dst, dstride, k_rows, index, index, index_is_int, n_index,
                                      src, sstride, cols, stream, "add_take_grad");
}

int mshadow_hip_add_take_grad_large_batch_f32(float *dst, int dstride, int k_rows,
                                              const void *sorted, const void *index,
                                              int index_is_int, int n_index, const float *src,
                                              int sstride, int cols, void *stream) {
  const int chk = RowOpCheck(dst, dstride, k_rows, index, n_index, src, sstride, cols);
  if (chk != MSHADOW_HIP_OK) return chk < 0 ? MSHADOW_HIP_OK : chk;
  ABI_REQUIRE(sorted != NULL, "NULL tensor");
  return LaunchRowsByIndex<kTakeGradSorted>(dst, dstride, k_rows, sorted, index, index_is_int,
                                            n_index, src, sstride, cols, stream,
                                            "add_take_grad_large_batch");
}

int mshadow_hip_index_fill_f32(float *dst, int dstride, int k_rows, const void *index,
                               int index_is_int, int n_index, const float *src, int sstride,
                               int cols, void *stream) {
  const int chk = RowOpCheck(dst, dstride, k_rows, index, n_index, src, sstride, cols);
  if (chk != MSHADOW_HIP_OK) return chk < 0 ? MSHADOW_HIP_OK : chk;
  return LaunchRowsByIndex<kFill>(dst, dstride, k_rows, index, index, index_is_int, n_index, src,
                                  sstride, cols, stream, "index_fill");
}

/* ------------------------------------------------------------------ reductions */

int mshadow_hip_reduce_keep_lowest_f32(float *dst, const float *src, int sstride, int rows,
                                       int cols, int reducer, int saver, float scale,
                                       void *stream) {
  ABI_REQUIRE(rows >= 1, "can not reduce over empty tensor");
  ABI_REQUIRE(cols >= 0, "negative shape");
  if (cols == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL, "NULL tensor");
  ABI_REQUIRE(sstride >= cols, "pitch smaller than the row");
  hipStream_t s = AsStream(stream);
  const uint32_t cus = mshadow_abi::ComputeUnits();
  const int strip = mshadow::hip::LowestColumnsPerStrip(cols, cus);
  int st = DispatchReducer(reducer, [&](auto red) {
    return DispatchSaver(saver, [&](auto sv) {
      typedef decltype(red) R;
      typedef decltype(sv) S;
#define LOWEST_STRIP(STRIP)                                                                     \
  LaunchKernelIfFits((mshadow::hip::ReduceKeepLowestStripKernel<S, R, mshadow::hip::STRIP>),    \
                     dim3((cols + mshadow::hip::STRIP::kCols - 1) / mshadow::hip::STRIP::kCols), \
                     dim3(mshadow::hip::STRIP::kThreads), 0, s, dst, src,                       \
                     static_cast<uint32_t>(sstride), static_cast<uint32_t>(rows),               \
                     static_cast<uint32_t>(cols), scale)
      if (std::is_same<R, mshadow::red::sum>::value &&
          LaunchColumnChunks<S>(dst, src, static_cast<uint32_t>(sstride), static_cast<uint32_t>(rows),
                                static_cast<uint32_t>(cols), scale, s)) {
        return MSHADOW_HIP_OK;
      }
      /* a strip for each CU at most and a long chain: four rows to an LDS read and stages of
         512 rows make its step 3.5 instead of 4.2 ns (65536 x 1000: 231 against 276 us;
         8191 x 1000: 36.7 against 38.2 us; level at 6000; 4096 x 2000: 22 against 20 us). The fewer
         lines a row has the sooner they arrive and the earlier the step decides (10 columns:
         4000 rows 18.9 against 19.5 us, 6143 27.7 against 28.7, 3500 level; 64: 6000 rows 27.2
         against 27.8, 4500 level; one: 2500 rows 12.8 against 13.5, 2200 12.7 against 12.1) */
      const int long_chain = cols == 1 ? 2400 : cols <= 64 ? 4000 : kDmaMinRows;
      if (strip == 16 && rows >= long_chain) {
        LaunchKernelIfFits((mshadow::hip::ReduceKeepLowestDmaKernel<S, R>),
                           dim3((cols + mshadow::hip::kLowestCols - 1) / mshadow::hip::kLowestCols),
                           dim3(mshadow::hip::kDmaThreads), 0, s, dst, src,
                           static_cast<uint32_t>(sstride), static_cast<uint32_t>(rows),
                           static_cast<uint32_t>(cols), scale);
      } else if (strip == 16 && rows >= 2048) {
        LOWEST_STRIP(LowestStrip16Long);
      } else if (strip == 16) {
        LOWEST_STRIP(LowestStrip16);
      } else if (strip == 32) {
        LOWEST_STRIP(LowestStrip32);
      } else if (rows > 1024 || static_cast<uint32_t>(cols) <= 128 * cus) {
        LOWEST_STRIP(LowestStrip64);
      } else {
        LOWEST_STRIP(LowestStrip64Short);
      }
#undef LOWEST_STRIP
      return MSHADOW_HIP_OK;
    });
  });
  if (st != MSHADOW_HIP_OK) return st;
  return AfterLaunch("reduce_keep_lowest");
}

int mshadow_hip_reduce_keep_highdim_f32(float *dst, const float *src, int sstride, int n, int c,
                                        int y, int x, int reducer, int saver, float scale,
                                        void *stream) {
  ABI_REQUIRE(n >= 0 && c >= 0 && y >= 0 && x >= 0, "negative shape");
  if (c == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL, "NULL tensor");
  ABI_REQUIRE(src != NULL || static_cast<long long>(n) * y * x == 0, "NULL tensor");
  ABI_REQUIRE(sstride >= x, "pitch smaller than the row");
  /* the kernels that stream a tensor from memory compute row numbers in 64 bits; the
     register-staged ones for short reductions (fewer than 2^16 values per kept index) in 32 */
  ABI_REQUIRE(static_cast<long long>(n) * c < (1ll << 31), "too many (n, c) segments for 32-bit indices");
  ABI_REQUIRE(static_cast<long long>(n) * c * y < (1ll << 31) ||
                  static_cast<long long>(n) * y * x >= kDmaMinPerKept,
              "too many rows for 32-bit indices");
  ABI_REQUIRE(static_cast<long long>(y) * x < (1ll << 31), "inner extent too large for 32-bit indices");
  const mshadow::FastDivU32 div_x(static_cast<uint32_t>(x > 0 ? x : 1));
  hipStream_t s = AsStream(stream);
  /* The split kernel walks dense rows as one row per segment. It needs scratch memory for
     n * c inner results. */
  int v_y = y, v_x = x, v_stride = sstride;
  if (sstride == x) {
    v_x = v_stride = y * x;
    v_y = 1;
  }
  const mshadow::hip::SegmentsPlan seg =
      mshadow::hip::PlanSegments(n, c, static_cast<uint64_t>(y) * x, mshadow_abi::ComputeUnits(), 4);
  uint32_t *split_partial = NULL, *split_counter = NULL;
  /* With a kept index for (nearly) every CU the one-workgroup-per-kept-index kernel fills the
     chip and ends without a merge; with fewer the inner chains are dealt out by segments:
     16 per workgroup and a kilobyte of each per load where rows are whole 16-byte packs, else
     32 per workgroup and 256 bytes of each. */
  const bool few_kept = static_cast<long long>(c) * 4 < 3ll * mshadow_abi::ComputeUnits();
  const bool whole_packs = v_x % 4 == 0 && v_stride % 4 == 0 && Aligned16(src);
  if (few_kept && !(seg.use && sstride == x) && static_cast<long long>(n) * y * x >= kDmaMinPerKept &&
      static_cast<long long>(n) * c < (1ll << 31)) {
    const int sc = mshadow_hip_reduce_scratch(stream, static_cast<size_t>(n) * c, &split_partial,
                                              &split_counter);
    if (sc != MSHADOW_HIP_OK) return sc;
  }
  const mshadow::FastDivU32 v_div_x(static_cast<uint32_t>(v_x > 0 ? v_x : 1));
  int st = DispatchReducer(reducer, [&](auto red) {
    return DispatchSaver(saver, [&](auto sv) {
      typedef decltype(red) R;
      typedef decltype(sv) S;
#define HIGHDIM_LAUNCH_T(T, SEGS)                                                              \
  for (long long c0 = 0, most = RowsOfLaunch(T); c0 < c; c0 += most) {                         \
    RawPlan1D<float> d = {dst + c0};                                                           \
    RawPlan2D<const float> sp = {src + c0 * y * sstride, sstride};                             \
    LaunchKernelIfFits((mshadow::hip::ReduceKeepHighDimKernel<S, R, float, T, SEGS, RawPlan1D<float>, \
                                                              RawPlan2D<const float> >),       \
                       dim3(static_cast<unsigned>(c - c0 < most ? c - c0 : most)), dim3(T), 0, s, d, sp, \
                       static_cast<uint32_t>(n), static_cast<uint32_t>(c), static_cast<uint32_t>(y), \
                       static_cast<uint32_t>(x), div_x, scale);                                \
  }
#define HIGHDIM_LAUNCH(SEGS)                                                                   \
  if (large)                                                                                   \
    LaunchKernelIfFits((mshadow::hip::ReduceKeepHighDimDmaKernel<S, R, float, SEGS>), dim3(c),        \
                       dim3(mshadow::hip::kDmaThreads), 0, s, dst, src,                        \
                       static_cast<uint32_t>(sstride), static_cast<uint32_t>(n),               \
                       static_cast<uint32_t>(c), static_cast<uint32_t>(y),                     \
                       static_cast<uint32_t>(x), div_x, scale);                                \
  else HIGHDIM_LAUNCH_T(mshadow::hip::kRedBlockSmall, SEGS)
      if (seg.use && sstride == x) {  // dense planes: waves with sixteen of them each
#define SEGMENTS(L)                                                                                          \
  LaunchKernelIfFits((mshadow::hip::ReduceSegmentsKernel<S, R, float, L>),                                   \
                     dim3((static_cast<uint32_t>(c) + seg.kept - 1) / seg.kept), dim3(seg.waves * 64),          \
                     (mshadow::hip::SegSlice<float, L>::LdsBytes(seg.waves, seg.kept * n)), s, dst, src,       \
                     static_cast<uint32_t>(y * x), static_cast<uint32_t>(n), static_cast<uint32_t>(c), seg.kept, \
                     mshadow::FastDivU32(seg.kept), scale)
        if (seg.lanes == 8) SEGMENTS(8);
        else SEGMENTS(16);
#undef SEGMENTS
        return MSHADOW_HIP_OK;
      }
      const bool large = static_cast<long long>(n) * y * x >= kDmaMinPerKept;
      if (large && split_partial != NULL) {
#define HIGHDIM_SPLIT(RING)                                                                    \
  LaunchKernelIfFits((mshadow::hip::ReduceKeepHighDimSplitKernel<S, R, float, RING>),          \
                     dim3((static_cast<unsigned>(n) * c + RING::kSegs - 1) / RING::kSegs),      \
                     dim3(RING::kThreads), 0, s, dst, src, static_cast<uint32_t>(v_stride),    \
                     static_cast<uint32_t>(n), static_cast<uint32_t>(c),                       \
                     static_cast<uint32_t>(v_y), static_cast<uint32_t>(v_x), v_div_x, scale,   \
                     split_partial, split_counter)
        if (whole_packs && static_cast<long long>(n) * c > 16ll * mshadow_abi::ComputeUnits()) {
          HIGHDIM_SPLIT(mshadow::hip::HighDimSplitRingPacksWide);
        } else if (whole_packs) {
          HIGHDIM_SPLIT(mshadow::hip::HighDimSplitRingPacks);
        } else {
          HIGHDIM_SPLIT(mshadow::hip::HighDimSplitRing);
        }
#undef HIGHDIM_SPLIT
        return MSHADOW_HIP_OK;
      }
      if (n > 16) { HIGHDIM_LAUNCH(64); }
      else if (n > 4) { HIGHDIM_LAUNCH(16); }
      else if (n > 1) { HIGHDIM_LAUNCH(4); }
      else { HIGHDIM_LAUNCH(1); }
#undef HIGHDIM_LAUNCH_T
#undef HIGHDIM_LAUNCH
      return MSHADOW_HIP_OK;
    });
  });
  if (st != MSHADOW_HIP_OK) return st;
  return AfterLaunch("reduce_keep_highdim");
}

/* ------------------------------------------------------------------ pool / unpool */

static const size_t kPoolLdsBudget = 48 * 1024;  // per workgroup: three resident per CU
static const size_t kUnpoolLdsBudget = 16 * 1024;  // smaller bands: more workgroups in different phases per CU

/*! \brief strips of the stride-1 unpool kernel over `rows` rows of `w` columns per plane:
 *  sixteen rows a strip, fewer while that leaves the machine short of waves */
static SlideGeom MakeSlideGeom(int planes, int rows, int w, int k) {
  SlideGeom sg;
  sg.groups = static_cast<uint32_t>((w + 3) / 4);
  sg.strips_per_wave = 64u / sg.groups;
  /* equal strips of up to 16 rows (65 rows as 5 x 13, not 4 x 16 and one: 63 against 70 us) */
  const uint32_t least = static_cast<uint32_t>((rows + 15) / 16);
  uint32_t r = (static_cast<uint32_t>(rows) + least - 1) / least;
  const long long want = 16ll * mshadow_abi::ComputeUnits();  // waves
  const bool turns_of_two = k == 5 && (w >= 24 || (w >= 16 && w % 4 == 0));
  if (turns_of_two) {
    /* Two waves of the kernel for 5 x 5 windows fill a SIMD, so strips are cut no further than it takes
       to deal every SIMD two: a strip costs its rows and about two and a half for the four pooled rows
       above it, times the turns of eight waves a CU. Against strips cut until there are 16 waves a
       CU: 1.8 M pixels, 7x160 14.6 and 23.8 us, 9x50 13 and 21, 40x100 15 and 20; 4 M, 24x64 19 and 27,
       16x32 20 and 29; 12 M, 40x40 66 and 75; 0.6 M level. Narrow rows stay with those: a wave has
       many strips then, and long ones are far apart (224x7 319 and 252 us, 100x18 117 and 111). */
    long long best = -1;
    for (uint32_t longest = r; longest >= 2; --longest) {
      const uint32_t n = (static_cast<uint32_t>(rows) + longest - 1) / longest;
      const uint32_t each = (static_cast<uint32_t>(rows) + n - 1) / n;
      const long long waves = (static_cast<long long>(planes) * n + sg.strips_per_wave - 1) / sg.strips_per_wave;
      const long long turns = (waves + 8ll * mshadow_abi::ComputeUnits() - 1) / (8ll * mshadow_abi::ComputeUnits());
      const long long cost = turns * (2 * each + 5);
      if (best < 0 || cost * 10 < best * 9) { best = cost; r = each; }
    }
  }
  while (!turns_of_two && r > 2 && static_cast<long long>(planes) * ((rows + r - 1) / r) / sg.strips_per_wave < want) r = (r + 1) / 2;
  sg.strip_rows = r;
  sg.strips_per_plane = static_cast<uint32_t>((rows + r - 1) / r);
  sg.total_strips = static_cast<uint32_t>(planes) * sg.strips_per_plane;
  sg.div_groups = mshadow::FastDivU32(sg.groups);
  sg.div_spp = mshadow::FastDivU32(sg.strips_per_plane);
  return sg;
}

int mshadow_hip_pool_f32(float *dst, int dstride, const float *src, int sstride, int planes,
                         int h, int w, int ph, int pw, int ky, int kx, int sy, int sx,
                         int reducer, void *stream) {
  ABI_REQUIRE(planes >= 0 && h >= 0 && w >= 0 && ph >= 0 && pw >= 0, "negative shape");
  ABI_REQUIRE(ky >= 1 && kx >= 1 && sy >= 1 && sx >= 1, "kernel and stride must be positive");
  ABI_REQUIRE(h >= ky && w >= kx, "kernel must be smaller than image");
  ABI_REQUIRE(reducer >= MSHADOW_HIP_SUM && reducer <= MSHADOW_HIP_MIN, "unknown reducer");
  if (planes == 0 || ph == 0 || pw == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL, "NULL tensor");
  ABI_REQUIRE(dstride >= pw && sstride >= w, "pitch smaller than the row");
  ABI_REQUIRE(static_cast<long long>(planes) * h < (1ll << 31) &&
                  static_cast<long long>(planes) * ph * pw < (1ll << 32),
              "too large for 32-bit indices");
  PoolGeom g = {h, w, ph, pw, ky, kx, sy, sx, 0, 0, w};
  hipStream_t s = AsStream(stream);
  const size_t row_bytes = static_cast<size_t>(g.lds_pitch) * sizeof(float);
  /* output rows per band so that (band - 1) * sy + ky input rows fit the budget */
  long long max_in_rows = static_cast<long long>(kPoolLdsBudget / row_bytes);
  long long band = max_in_rows >= ky ? (max_in_rows - ky) / sy + 1 : 0;
  if (band > ph) band = ph;
  /* keep at least ~4 workgroups per CU in flight when planes are few */
  while (band > 8 && static_cast<long long>(planes) * ((ph + band - 1) / band) < 1024) {
    band = (band + 1) / 2;
  }
  if (band >= 1) {
    /* equal-sized bands of about 20 KB of input rows (but four output rows or more): seven or
       eight workgroups then share a CU, and while some wait at their barrier others load.
       (32,64,224,224) 2x2 stride 2: 80 us against 102 us with bands of 41 KB; 14 KB and less
       lose again to the rows that neighbouring bands both read. */
    long long nb = (ph + band - 1) / band;
    const long long target = 20 * 1024;
    const long long want = (static_cast<long long>(ph) * sy * row_bytes + target - 1) / target;
    if (want > nb) nb = want;
    if (nb > ph / 4 && ph >= 4) nb = ph / 4;
    band = (ph + nb - 1) / nb;
  }
#define POOL_SWITCH(KERNEL, ...)                                                               \
  switch (reducer) {                                                                           \
    case MSHADOW_HIP_SUM: LaunchKernelIfFits((KERNEL<MSHADOW_HIP_SUM>), __VA_ARGS__); break;    \
    case MSHADOW_HIP_MAX: LaunchKernelIfFits((KERNEL<MSHADOW_HIP_MAX>), __VA_ARGS__); break;    \
    default: LaunchKernelIfFits((KERNEL<MSHADOW_HIP_MIN>), __VA_ARGS__); break;                 \
  }
  /* windows that move by one element, all of them whole: PoolColumnsS1Kernel below has a variant */
  const bool columns = sy == 1 && sx == 1 && ky == kx && (ky == 2 || ky == 3 || ky == 5) &&
                       ph <= h - ky + 1 && pw <= w - kx + 1;
  /* small planes: several whole planes per workgroup, about 24 KB of them. Planes of 1024 pixels and
     more keep the threads of the columns kernel busy (12 M pixels, 5x5: 50x50 24 against 35 us, 3x3:
     100x30 21 against 28 us; level at 32x32, and 7x7 is 16 us here against 312 us there), but for the
     small windows on very narrow ones (3x3: 224x7 21 us here, 24 us there). With windows of two and
     three the two are close: where there are planes for full groups and whole rows fill a wave's
     lanes here, the columns kernel is the faster one only on larger planes (12 M pixels, 3x3, here
     and there: 61x17 25 and 32 us, 32x33 24 and 26, 17x63 24 and 30, 8x160 21 and 22, 45x33 26 and 23;
     31x35, half the lanes idle here, 35 and 28; 3 M pixels, 17x63: 10 and 9). Low wide planes whose rows are no
     packs, or with windows of three, come later still (2x2: 9x155 15 and 18.5 us, 9x187 11.7 and 13.3; 3x3: 9x148
     19 and 21, 11x161 17 and 19; 12x159 31 and 26;
     2x2 8x195, 48 of 64 lanes at work here, 35 and 31). */
  const long long plane_bytes = static_cast<long long>(h) * row_bytes;
  const auto columns_pay = [&]() {
    if (ky == 5) return h * w >= 1024;
    if (w < 16) return false;
    const bool full_groups = planes / ((24 * 1024) / plane_bytes) >= 4ll * mshadow_abi::ComputeUnits();
    const int lanes = pw < 64 ? pw * (64 / pw) : pw * 64 / ((pw + 63) / 64 * 64);  // of 64, at work here
    if (w > 100 && h < 14) return h * w >= (ky == 2 && (w % 4 == 0 || (pw > 192 && lanes < 51)) ? 1300 : 1750);
    return h * w >= (!full_groups || lanes < 51 ? 1024 : w % 4 == 0 && w > 16 ? 1100 : 1400);
  };
  if (plane_bytes * 2 <= 24 * 1024 && planes >= 2 && !(columns && band >= 1 && columns_pay())) {
    long long per_block = (24 * 1024) / plane_bytes;
    /* ... but no fewer workgroups than keep every CU busy four times over */
    while (per_block > 1 && (planes + per_block - 1) / per_block < 4ll * mshadow_abi::ComputeUnits()) {
      per_block = (per_block + 1) / 2;
    }
    if (per_block >= 2) {
      const size_t lds = static_cast<size_t>(per_block) * plane_bytes + 16;
      const unsigned blocks = static_cast<unsigned>((planes + per_block - 1) / per_block);
      const mshadow::FastDivU32 div_ph(static_cast<uint32_t>(ph));
#define POOL_PLANES(KY, KX)                                                                     \
  switch (reducer) {                                                                           \
    case MSHADOW_HIP_SUM:                                                                      \
      LaunchKernelIfFits((PoolPlanesKernel<MSHADOW_HIP_SUM, KY, KX>), dim3(blocks), dim3(kPoolBlock), \
                         lds, s, dst, dstride, src, sstride, g, planes, static_cast<int>(per_block), div_ph); \
      break;                                                                                   \
    case MSHADOW_HIP_MAX:                                                                      \
      LaunchKernelIfFits((PoolPlanesKernel<MSHADOW_HIP_MAX, KY, KX>), dim3(blocks), dim3(kPoolBlock), \
                         lds, s, dst, dstride, src, sstride, g, planes, static_cast<int>(per_block), div_ph); \
      break;                                                                                   \
    default:                                                                                   \
      LaunchKernelIfFits((PoolPlanesKernel<MSHADOW_HIP_MIN, KY, KX>), dim3(blocks), dim3(kPoolBlock), \
                         lds, s, dst, dstride, src, sstride, g, planes, static_cast<int>(per_block), div_ph); \
      break;                                                                                   \
  }
      if (ky == 3 && kx == 3) { POOL_PLANES(3, 3) }
      else if (ky == 2 && kx == 2) { POOL_PLANES(2, 2) }
      else if (ky == 5 && kx == 5) { POOL_PLANES(5, 5) }
      else { POOL_PLANES(0, 0) }
#undef POOL_PLANES
      return AfterLaunch("pool");
    }
  }
  if (band >= 1) {
    g.band = static_cast<int>(band);
    g.bands = (ph + g.band - 1) / g.band;
    const size_t lds = (static_cast<size_t>(g.band - 1) * sy + ky) * row_bytes + 16;
    const long long blocks = static_cast<long long>(planes) * g.bands;
    ABI_REQUIRE(blocks < (1ll << 31), "too many workgroups");
    /* windows that move by one element: a thread walks down an output column, KX reads of LDS an
       output. The band's rows are cut into `nruns` runs so that the columns of all runs fill the
       workgroup's threads in as few, as short rounds as can be. */
    if (columns) {
      int nruns = 1, run_len = g.band;
      long long best = -1;
      for (int n = 1; n <= g.band; ++n) {
        const int rl = (g.band + n - 1) / n;
        const long long rounds = (static_cast<long long>(n) * pw + kPoolBlock - 1) / kPoolBlock;
        const long long cost = rounds * (rl + ky - 1);
        if (best < 0 || cost < best) { best = cost; nruns = n; run_len = rl; }
      }
      const mshadow::FastDivU32 div_pw(static_cast<uint32_t>(pw));
#define POOL_COLUMNS(K)                                                                        \
  switch (reducer) {                                                                           \
    case MSHADOW_HIP_SUM:                                                                      \
      LaunchKernelIfFits((PoolColumnsS1Kernel<MSHADOW_HIP_SUM, K, K>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g, nruns, run_len, div_pw); \
      break;                                                                                   \
    case MSHADOW_HIP_MAX:                                                                      \
      LaunchKernelIfFits((PoolColumnsS1Kernel<MSHADOW_HIP_MAX, K, K>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g, nruns, run_len, div_pw); \
      break;                                                                                   \
    default:                                                                                   \
      LaunchKernelIfFits((PoolColumnsS1Kernel<MSHADOW_HIP_MIN, K, K>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g, nruns, run_len, div_pw); \
      break;                                                                                   \
  }
      if (ky == 2) { POOL_COLUMNS(2) }
      else if (ky == 3) { POOL_COLUMNS(3) }
      else { POOL_COLUMNS(5) }
#undef POOL_COLUMNS
      return AfterLaunch("pool");
    }
#define POOL_TILED(KY, KX)                                                                     \
  switch (reducer) {                                                                           \
    case MSHADOW_HIP_SUM:                                                                      \
      LaunchKernelIfFits((PoolKernel<MSHADOW_HIP_SUM, KY, KX>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g);             \
      break;                                                                                   \
    case MSHADOW_HIP_MAX:                                                                      \
      LaunchKernelIfFits((PoolKernel<MSHADOW_HIP_MAX, KY, KX>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g);             \
      break;                                                                                   \
    default:                                                                                   \
      LaunchKernelIfFits((PoolKernel<MSHADOW_HIP_MIN, KY, KX>), dim3(static_cast<unsigned>(blocks)), \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, g);             \
      break;                                                                                   \
  }
    if (ky == 3 && kx == 3) { POOL_TILED(3, 3) }
    else if (ky == 2 && kx == 2) { POOL_TILED(2, 2) }
    else { POOL_TILED(0, 0) }
#undef POOL_TILED
  } else {
    const unsigned total = static_cast<unsigned>(planes) * ph * pw;
    unsigned grid = 0;
    int st = mshadow_hip_suggest_grid(total, kPoolBlock, 4, &grid);
    if (st != MSHADOW_HIP_OK) return st;
    POOL_SWITCH(PoolDirectKernel, dim3(grid), dim3(kPoolBlock), 0, s, dst, dstride, src, sstride,
                g, total)
  }
  return AfterLaunch("pool");
}

int mshadow_hip_unpool_f32(float *dst, int dstride, const float *src, int sstride,
                           const float *pooled, int pstride, const float *grad, int gstride,
                           int planes, int h, int w, int ph, int pw, int ky, int kx, int sy,
                           int sx, int reducer, void *stream) {
  ABI_REQUIRE(planes >= 0 && h >= 0 && w >= 0 && ph >= 0 && pw >= 0, "negative shape");
  ABI_REQUIRE(ky >= 1 && kx >= 1 && sy >= 1 && sx >= 1, "kernel and stride must be positive");
  ABI_REQUIRE(reducer >= MSHADOW_HIP_SUM && reducer <= MSHADOW_HIP_MIN, "unknown reducer");
  if (planes == 0 || h == 0 || w == 0) return MSHADOW_HIP_OK;
  ABI_REQUIRE(dst != NULL && src != NULL, "NULL tensor");
  ABI_REQUIRE((pooled != NULL && grad != NULL) || ph == 0 || pw == 0, "NULL tensor");
  ABI_REQUIRE(dstride >= w && sstride >= w && pstride >= pw && gstride >= pw,
              "pitch smaller than the row");
  ABI_REQUIRE(static_cast<long long>(planes) * h * w < (1ll << 32) &&
                  static_cast<long long>(planes) * h < (1ll << 31),
              "too large for 32-bit indices");
  PoolGeom g = {h, w, ph, pw, ky, kx, sy, sx, 0, 0, pw};
  hipStream_t s = AsStream(stream);
  /* 3 x 3 windows with stride 2 on rows of up to 256 pixels: no staging. Even heights and rows of
     whole aligned packs take the plain form, everything else the one that moves packs anywhere */
  if (ky == 3 && kx == 3 && sy == 2 && sx == 2 && w <= 256 && ph >= 1 && pw >= 1 &&
      static_cast<long long>(planes) * ph * pw >= 2) {
    const bool whole = h % 2 == 0 && w % 4 == 0 && dstride % 4 == 0 && sstride % 4 == 0 &&
                       Aligned16(dst) && Aligned16(src);
    UnpoolRowsGeom rg;
    rg.half_h = static_cast<uint32_t>((h + 1) / 2);
    rg.total_rows = static_cast<uint32_t>(planes) * rg.half_h;
    rg.groups = static_cast<uint32_t>((w + 3) / 4);
    rg.rows_per_wave = 64u / rg.groups;
    rg.div_groups = mshadow::FastDivU32(rg.groups);
    rg.div_half_h = mshadow::FastDivU32(rg.half_h);
    rg.pooled_floats = (static_cast<size_t>(planes) * ph - 1) * pstride + pw;
    rg.grad_floats = (static_cast<size_t>(planes) * ph - 1) * gstride + pw;
    rg.src_floats = (static_cast<size_t>(planes) * h - 1) * sstride + w;
    const uint32_t waves = (rg.total_rows + rg.rows_per_wave - 1) / rg.rows_per_wave;
    const uint32_t blocks = (waves + kPoolBlock / 64 - 1) / (kPoolBlock / 64);
#define UNPOOL_ROWS(R)                                                                          \
  do {                                                                                          \
    if (whole) {                                                                                \
      LaunchKernelIfFits((UnpoolRows3x3s2Kernel<R, false>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, \
                         dstride, src, sstride, pooled, pstride, grad, gstride, g, rg);         \
    } else {                                                                                    \
      LaunchKernelIfFits((UnpoolRows3x3s2Kernel<R, true>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, \
                         dstride, src, sstride, pooled, pstride, grad, gstride, g, rg);         \
    }                                                                                           \
  } while (0)
    if (reducer == MSHADOW_HIP_SUM) UNPOOL_ROWS(MSHADOW_HIP_SUM);
    else if (reducer == MSHADOW_HIP_MAX) UNPOOL_ROWS(MSHADOW_HIP_MAX);
    else UNPOOL_ROWS(MSHADOW_HIP_MIN);
#undef UNPOOL_ROWS
    return AfterLaunch("unpool");
  }
  /* 2 x 2, 3 x 3 and 5 x 5 windows with stride 1 on rows of up to 256 pixels: no staging, the pooled
     rows over the current source row in registers ((128,64,112,112) 3 x 3: 368 us against 513 us for
     the kernels below). A lane has four pixels of a row, so narrow planes make its accesses short
     and scattered, which the staged kernels do not mind; what those mind is many windows a pixel.
     12 M pixels: 3 x 3 56x56 54 us against 51, 63x70 58 against 52, 20x200 46 against 56; 2 x 2 28x28 74 against 64,
     56x56 50 against 65; 5 x 5 13x13 145 against 127, 16x16 73 against 102, 8x40 69 against 121,
     28x28 78 against 105, and beyond 4 KB a plane - one plane per workgroup there - 100x14 130 against
     317, 224x7 251 against 470. Low planes whose rows leave a third of the lanes idle are made twice
     over here, most of their windows being cut off: 7x160 80 against 71 us, 8x140 (24 M pixels) 168
     against 153, 5x128 57 against 46 - unless there are waves for one turn only (1.8 M pixels, 7x160
     14.6 against 15.5 us). Rows of 33 to 63 columns that are no packs, 2 x 2: as long as the four tensors
     stay in the memory-side cache (4 M pixels, 56x50 23 against 30; 12 M 78 and 74; 36 M, 56x34 279 and 239).
     5 x 5 on few low planes: a strip's rows wait for one another, and the staged kernel has a pixel a
     thread (103 planes of 8x34 5.3 against 7.2 us, 464 of 8x36 6.3 and 7.1, 23 of 14x32 5.8 and 6.4; 301 of
     14x25 8.5 and 7.2, 573 of 10x56 9.6 and 7.7, and with two rounds of its lanes 10 of 8x77 7.7 and 6.4). */
  const int slide_lanes = w <= 256 ? (w + 3) / 4 * (64 / ((w + 3) / 4)) : 0;  // of 64 with pixels: 40 at 140 columns
  const bool slides = ky == 5 ? (static_cast<long long>(h) * w > 1024 || (h > 5 && (w >= 24 || (w >= 16 && w % 4 == 0)))) &&
                                    !(slide_lanes < 44 && h <= 9 && static_cast<long long>(h) * w <= 1280 &&
                                      planes > 8 * mshadow_abi::ComputeUnits()) &&
                                    !(w >= (h < 8 ? 16 : 20) && w <= 64 && h <= 16 &&
                                      static_cast<long long>(planes) * h * w < (w < 20 || h > 9 ? 40000 : h == 9 ? 60000 : 150000))
                      : ky == 2 ? w >= 64 || (w >= 32 && (w % 4 == 0 || static_cast<long long>(planes) * h * w <= 12000000))
                                : w >= 64 && (h >= 64 || (w >= 96 && h >= 16));
  if (ky == kx && (ky == 2 || ky == 3 || ky == 5) && sy == 1 && sx == 1 && w <= 256 && slides && ph >= 1 && pw >= 1 &&
      static_cast<long long>(planes) * ph * pw >= 4 && static_cast<long long>(planes) * ((h + 1) / 2) < (1ll << 31)) {
    SlideGeom sg = MakeSlideGeom(planes, h, w, ky);
    sg.src_floats = (static_cast<size_t>(planes) * h - 1) * sstride + w;
    sg.pooled_floats = (static_cast<size_t>(planes) * ph - 1) * pstride + pw;
    sg.grad_floats = (static_cast<size_t>(planes) * ph - 1) * gstride + pw;
    const uint32_t waves = (sg.total_strips + sg.strips_per_wave - 1) / sg.strips_per_wave;
    const uint32_t blocks = (waves + kPoolBlock / 64 - 1) / (kPoolBlock / 64);
#define UNPOOL_SLIDE(R)                                                                        \
  do {                                                                                         \
    if (ky == 2) {                                                                             \
      LaunchKernelIfFits((UnpoolSlideS1Kernel<R, 2, 4>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, dstride, \
                         src, sstride, pooled, pstride, grad, gstride, g, sg);                 \
    } else if (ky == 3) {                                                                      \
      LaunchKernelIfFits((UnpoolSlideS1Kernel<R, 3, 3>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, dstride, \
                         src, sstride, pooled, pstride, grad, gstride, g, sg);                 \
    } else {                                                                                   \
      LaunchKernelIfFits((UnpoolSlideS1Kernel<R, 5, 5>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, dstride, \
                         src, sstride, pooled, pstride, grad, gstride, g, sg);                 \
    }                                                                                          \
  } while (0)
    if (reducer == MSHADOW_HIP_SUM) UNPOOL_SLIDE(MSHADOW_HIP_SUM);
    else if (reducer == MSHADOW_HIP_MAX) UNPOOL_SLIDE(MSHADOW_HIP_MAX);
    else UNPOOL_SLIDE(MSHADOW_HIP_MIN);
#undef UNPOOL_SLIDE
    return AfterLaunch("unpool");
  }
  /* 2 x 2 windows, stride 2: a pixel has one window at most; four pixels and two windows per thread */
  if (ky == 2 && kx == 2 && sy == 2 && sx == 2 && w >= 4 && ph >= 1 && pw >= 1 &&
      static_cast<long long>(planes) * ph * pw >= 2) {
    const long long wpk = (w + 3) / 4;
    const long long packs = static_cast<long long>(planes) * h * wpk;
    if (packs + kPoolBlock < (1ll << 31)) {
      const unsigned blocks = static_cast<unsigned>((packs + kPoolBlock - 1) / kPoolBlock);
#define UNPOOL_2X2(R, WHOLE)                                                                                        \
  LaunchKernelIfFits((Unpool2x2s2Kernel<R, WHOLE>), dim3(blocks), dim3(kPoolBlock), 0, s, dst, dstride, src, sstride, \
                     pooled, pstride, grad, gstride, g, mshadow::FastDivU32(static_cast<uint32_t>(wpk)),            \
                     mshadow::FastDivU32(static_cast<uint32_t>(h)), static_cast<uint32_t>(packs),                   \
                     (static_cast<size_t>(planes) * h - 1) * sstride + w,                                           \
                     (static_cast<size_t>(planes) * ph - 1) * pstride + pw,                                         \
                     (static_cast<size_t>(planes) * ph - 1) * gstride + pw)
#define UNPOOL_2X2_OF(R) do { if (w % 4 == 0) UNPOOL_2X2(R, true); else UNPOOL_2X2(R, false); } while (0)
      if (reducer == MSHADOW_HIP_SUM) UNPOOL_2X2_OF(MSHADOW_HIP_SUM);
      else if (reducer == MSHADOW_HIP_MAX) UNPOOL_2X2_OF(MSHADOW_HIP_MAX);
      else UNPOOL_2X2_OF(MSHADOW_HIP_MIN);
#undef UNPOOL_2X2_OF
#undef UNPOOL_2X2
      return AfterLaunch("unpool");
    }
  }
  /* small planes under a stride of 2 or more (a pixel has few windows): no staging. Measured on
     (128,256,28,28), 2x2 stride 2: 56 us against 96 us for the kernels below; on large planes or
     with stride 1 the staged kernels are faster. */
  if (static_cast<long long>(h) * w * sizeof(float) <= 4 * 1024 && sy >= 2 && sx >= 2 && w >= 4) {
    const long long wpk = (w + 3) / 4;
    const long long packs = static_cast<long long>(planes) * h * wpk;
    if (packs + kPoolBlock < (1ll << 31)) {
      const unsigned blocks = static_cast<unsigned>((packs + kPoolBlock - 1) / kPoolBlock);
      POOL_SWITCH(UnpoolGatherKernel, dim3(blocks), dim3(kPoolBlock), 0, s, dst, dstride, src, sstride,
                  pooled, pstride, grad, gstride, g, mshadow::FastDivU32(static_cast<uint32_t>(sy)),
                  mshadow::FastDivU32(static_cast<uint32_t>(sx)),
                  mshadow::FastDivU32(static_cast<uint32_t>(wpk)),
                  mshadow::FastDivU32(static_cast<uint32_t>(h)), static_cast<uint32_t>(packs))
      return AfterLaunch("unpool");
    }
  }
  /* small planes: several whole planes per workgroup (about 24 KB of pooled values and gradients) */
  {
    const long long plane_bytes = static_cast<long long>(ph) * g.lds_pitch * sizeof(float) * 2;
    const long long src_plane_bytes = static_cast<long long>(h) * w * sizeof(float);
    if (plane_bytes > 0 && plane_bytes * 2 <= 24 * 1024 && src_plane_bytes <= 4 * 1024 && planes >= 2) {
      long long per_block = (24 * 1024) / plane_bytes;
      while (per_block > 1 &&
             (planes + per_block - 1) / per_block < 4ll * mshadow_abi::ComputeUnits()) {
        per_block = (per_block + 1) / 2;
      }
      if (per_block >= 2) {
        const size_t lds = static_cast<size_t>(per_block) * plane_bytes + 32;
        const unsigned blocks = static_cast<unsigned>((planes + per_block - 1) / per_block);
        const mshadow::FastDivU32 div_h(static_cast<uint32_t>(h));
#define UNPOOL_PLANES(KY, KX, SY, SX)                                                          \
  switch (reducer) {                                                                           \
    case MSHADOW_HIP_SUM:                                                                      \
      LaunchKernelIfFits((UnpoolPlanesKernel<MSHADOW_HIP_SUM, KY, KX, SY, SX>), dim3(blocks),   \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, pooled, pstride, \
                         grad, gstride, g, planes, static_cast<int>(per_block), div_h);        \
      break;                                                                                   \
    case MSHADOW_HIP_MAX:                                                                      \
      LaunchKernelIfFits((UnpoolPlanesKernel<MSHADOW_HIP_MAX, KY, KX, SY, SX>), dim3(blocks),   \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, pooled, pstride, \
                         grad, gstride, g, planes, static_cast<int>(per_block), div_h);        \
      break;                                                                                   \
    default:                                                                                   \
      LaunchKernelIfFits((UnpoolPlanesKernel<MSHADOW_HIP_MIN, KY, KX, SY, SX>), dim3(blocks),   \
                         dim3(kPoolBlock), lds, s, dst, dstride, src, sstride, pooled, pstride, \
                         grad, gstride, g, planes, static_cast<int>(per_block), div_h);        \
      break;                                                                                   \
  }
        if (ky == 3 && kx == 3 && sy == 2 && sx == 2) { UNPOOL_PLANES(3, 3, 2, 2) }
        else if (ky == 2 && kx == 2 && sy == 2 && sx == 2) { UNPOOL_PLANES(2, 2, 2, 2) }
        else if (ky == 3 && kx == 3 && sy == 1 && sx == 1) { UNPOOL_PLANES(3, 3, 1, 1) }
        else { UNPOOL_PLANES(0, 0, 0, 0) }
#undef UNPOOL_PLANES
        return AfterLaunch("unpool");
      }
    }
  }
  const size_t row_bytes = static_cast<size_t>(g.lds_pitch) * sizeof(float) * 2;  // pooled + grad
  /* source rows per band: prow_max = (band + ky - 2) / sy + 2 pooled rows must fit */
  long long max_prow = static_cast<long long>(kUnpoolLdsBudget / row_bytes);
  long long band = (max_prow - 2) * sy - ky + 2;
  if (band > h) band = h;
  while (band > 8 && static_cast<long long>(planes) * ((h + band - 1) / band) < 1024) {
    band = (band + 1) / 2;
  }
  if (band >= 1) {  // equal-sized bands, starting at multiples of the stride
    const long long nb = (h + band - 1) / band;
    band = (h + nb - 1) / nb;
    band = (band + sy - 1) / sy * sy;
  }
  if (band >= 1 && max_prow >= 3) {
    g.band = static_cast<int>(band);
    g.bands = (h + g.band - 1) / g.band;
    const int prow_max = (g.band + ky - 2) / sy + 2;
    const size_t lds = static_cast<size_t>(prow_max) * row_bytes + 32;
    const long long blocks = static_cast<long long>(planes) * g.bands;
    ABI_REQUIRE(blocks < (1ll << 31), "too many workgroups");
    ABI_REQUIRE(lds <= 160 * 1024, "pooled rows too long for the LDS-tiled kernel");
    const mshadow::FastDivU32 div_bw(static_cast<uint32_t>((w + sx - 1) / sx));
    /* whole, aligned blocks of sx pixels per row: a block row is one memory access */
    const bool vec = (sx == 2 || sx == 4) && w % sx == 0 && dstride % sx == 0 && sstride % sx == 0 &&
                     reinterpret_cast<uintptr_t>(dst) % (sx * 4) == 0 &&
                     reinterpret_cast<uintptr_t>(src) % (sx * 4) == 0;
    const UnpoolArgs ua = {dst, dstride, src, sstride, pooled, pstride, grad, gstride, g, prow_max,
                           static_cast<unsigned>(blocks), lds, s};
    if (ky == 3 && kx == 3 && sy == 2 && sx == 2) {
      if (vec) LaunchUnpoolBlock<3, 3, 2, 2, true>(reducer, ua, div_bw);
      else LaunchUnpoolBlock<3, 3, 2, 2, false>(reducer, ua, div_bw);
    } else if (ky == 2 && kx == 2 && sy == 2 && sx == 2) {
      if (vec) LaunchUnpoolBlock<2, 2, 2, 2, true>(reducer, ua, div_bw);
      else LaunchUnpoolBlock<2, 2, 2, 2, false>(reducer, ua, div_bw);
    } else if (ky == 3 && kx == 3 && sy == 1 && sx == 1) {
      LaunchUnpoolBlock<3, 3, 1, 1, false>(reducer, ua, div_bw);
    } else {
      LaunchUnpoolGeneric(reducer, ua);
    }
  } else {
    const unsigned total = static_cast<unsigned>(planes) * h * w;
    unsigned grid = 0;
    int st = mshadow_hip_suggest_grid(total, kPoolBlock, 4, &grid);
    if (st != MSHADOW_HIP_OK) return st;
    POOL_SWITCH(UnpoolDirectKernel, dim3(grid), dim3(kPoolBlock), 0, s, dst, dstride, src,
                sstride, pooled, pstride, grad, gstride, g, total)
  }
#undef POOL_SWITCH
  return AfterLaunch("unpool");
}

/* ------------------------------------------------------------------ im2col / col2im */

#define PATCH_ENTRY(NAME, T, FN, A, AS, B, BS)                                                 \
  int NAME(T *A, int AS, const T *B, int BS, int n, int c, int h, int w, int ky, int kx, int sy, \
           int sx, int dy, int dx, int pad_y, int pad_x, void *stream) {                        \
    PatchGeom g;                                                                               \
    int st = MakePatchGeom(&g, n, c, h, w, ky, kx, sy, sx, dy, dx, pad_y, pad_x);              \
    if (st != MSHADOW_HIP_OK) return st;                                                       \
    return FN<T>(A, AS, B, BS, g, stream);                                                     \
  }
PATCH_ENTRY(mshadow_hip_im2col_f16, uint16_t, Im2Col, col, cstride, img, istride)
PATCH_ENTRY(mshadow_hip_im2col_f32, float, Im2Col, col, cstride, img, istride)
PATCH_ENTRY(mshadow_hip_col2im_f16, uint16_t, Col2Im, img, istride, col, cstride)
PATCH_ENTRY(mshadow_hip_col2im_f32, float, Col2Im, img, istride, col, cstride)
#undef PATCH_ENTRY

}  // extern "C"
