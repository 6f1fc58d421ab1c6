// The instantiations of fused_4bit_kernel for lists that also hold tensors with fp32 moments, and their selection.
#include <hip/hip_runtime.h>

#include "q4adamw_pick.h"
#include "q4adamw_step.h"

namespace q4 {

template <bool EXT, bool SR, bool EXACT>
static FusedKernel pick_pg(int p_dtype, int g_dtype) {
  Q4_PICK_PG(fused_4bit_kernel, EXT, SR, EXACT, true)
}

template <bool EXT, bool SR>
static FusedKernel pick_exact(int p_dtype, int g_dtype, bool exact) {
  return exact ? pick_pg<EXT, SR, true>(p_dtype, g_dtype) : pick_pg<EXT, SR, false>(p_dtype, g_dtype);
}

FusedKernel pick_mixed(int p_dtype, int g_dtype, bool ext, bool sr, bool exact) {
  if (sr) return ext ? pick_exact<true, true>(p_dtype, g_dtype, exact) : pick_exact<false, true>(p_dtype, g_dtype, exact);
  return ext ? pick_exact<true, false>(p_dtype, g_dtype, exact) : pick_exact<false, false>(p_dtype, g_dtype, exact);
}

}  // namespace q4
