// The split f32 GEMM (gemm_f32_split.h) with A M-contiguous.
#include "gemm_f32_split.h"

namespace nova_hip {
namespace split {

int32_t launch_a_mcontig(int form, const SplitArgs &r, bool bkc, unsigned grid, hipStream_t s) {
  return bkc ? launch_form<false, true>(form, r, grid, s) : launch_form<false, false>(form, r, grid, s);
}

}  // namespace split
}  // namespace nova_hip
