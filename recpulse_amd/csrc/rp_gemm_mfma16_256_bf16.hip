// bf16 MFMA GEMM, 256 x 256 block tile (2 x 2 waves).
#include "rp_gemm_mfma16_kernel.h"

namespace rp {

int launch_mfma16_256_bf16(const GemmArgs& g, const Plan& p) { return p.edge ? m16_launch_layout<bf16_t, 256, 256, 2, M16_EDGE>(g, p) : m16_launch_layout<bf16_t, 256, 256, 2, M16_WHOLE>(g, p); }

}  // namespace rp
