// bf16 / fp16 MFMA GEMM, 256 x 256 block tile: selection across its translation units (each kernel of this tile compiles
// for about twenty seconds).
#include "rp_gemm.h"

namespace rp {

int launch_mfma16_256_bf16(const GemmArgs& g, const Plan& p);
int launch_mfma16_256_ragged_bf16(const GemmArgs& g, const Plan& p);
int launch_mfma16_256_f16(const GemmArgs& g, const Plan& p);
int launch_mfma16_256_ragged_f16(const GemmArgs& g, const Plan& p);

int launch_mfma16_256(const GemmArgs& g, const Plan& p, int dtype) {
    if (dtype == RP_DTYPE_BFLOAT16) return p.ragged ? launch_mfma16_256_ragged_bf16(g, p) : launch_mfma16_256_bf16(g, p);
    if (dtype == RP_DTYPE_FLOAT16) return p.ragged ? launch_mfma16_256_ragged_f16(g, p) : launch_mfma16_256_f16(g, p);
    set_error("mfma16 GEMM: unsupported dtype %d", dtype);
    return -1;
}

}  // namespace rp
