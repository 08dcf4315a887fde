// bf16 MFMA GEMM, 256 x 256 block tile (2 x 2 waves), rows of any length and alignment.
#include "rp_gemm_mfma16_kernel.h"

namespace rp {

int launch_mfma16_256_ragged_bf16(const GemmArgs& g, const Plan& p) { return m16_launch_layout<bf16_t, 256, 256, 2, M16_RAGGED>(g, p); }

}  // namespace rp
