// The ring GEMM (gemm_ring.h) for f16 operands: every tile form and layout.
#include "gemm_ring.h"

namespace nova_hip {
namespace ring {

int32_t launch_f16(int form, const RingArgs &r, bool akc, bool bkc, hipStream_t s) {
  return launch_form<NOVA_HIP_DT_F16>(form, r, akc, bkc, s);
}

}  // namespace ring
}  // namespace nova_hip
