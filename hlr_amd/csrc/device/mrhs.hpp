// mrhs.hpp -- products with several right-hand sides (matrix cores).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "kernels.hpp"

namespace hmvm {

constexpr int kMrhsMax = 64;   // right-hand sides per launch sequence

// Y += alpha op(A) X for 1 <= R <= kMrhsMax right-hand sides, op the
// transpose when trans; vdt 0: FP64 vectors, 1: FP32; fam: the plan's format
// family (kFamHw, kFamBfp, kFamAfl or kFamF64), rows64: whether its
// workspace rows are FP64 (HostLayout::rows64).  ws holds mrhs_ws_doubles doubles (partials, t and the
// transposed copy of X), 8-byte aligned.  Returns 0 on success.
int launch_apply_mrhs(const DevPlan& D, int fam, bool rows64, bool trans, double alpha, const void* x, int64_t ldx,
                      void* y, int64_t ldy, int R, int vdt, double* ws, hipStream_t st);

// workspace of such a call; partials: psize (forward) or qsize (transposed)
// of the plan, nin: length of the input vectors.  INT64_MAX where R
// right-hand sides are too many for the kernels' 32-bit offsets.
int64_t mrhs_ws_doubles(int fam, bool rows64, bool trans, int64_t partials, int64_t ntent, int64_t nin, int R);

} // namespace hmvm
