/*
 * Which im2col kernel takes patch rows shorter than a 16-byte pack: plain C++, so that a host program can look at the
 * choice without a GPU.
 */
#ifndef MSHADOW_AMD_CSRC_PATCH_PLAN_H_
#define MSHADOW_AMD_CSRC_PATCH_PLAN_H_

#include <stdint.h>

namespace mshadow_hipk {

const int kPatchBlock = 256;  // threads of a workgroup of the im2col and col2im kernels

/*! \brief workgroups of Im2ColKernel for a column matrix of rows x cols, packs of `ept` elements */
inline int64_t Im2ColPackBlocks(int64_t rows, int64_t cols, int ept) {
  const int64_t per = static_cast<int64_t>(kPatchBlock) * ept;
  return (cols + per - 1) / per * rows;
}
/*! \brief ... and whether they are a launch: fewer than 2^32 threads. Every row of the matrix is a workgroup at
 *  least, however few columns it has, so a single image of very many channels is none (3x3 on (1,1900000,7,7)). */
inline bool Im2ColPacksFit(int64_t rows, int64_t cols, int ept) {
  return cols < (1ll << 31) && Im2ColPackBlocks(rows, cols, ept) < (1ll << 32) / kPatchBlock;
}

}  // namespace mshadow_hipk

#endif  // MSHADOW_AMD_CSRC_PATCH_PLAN_H_
