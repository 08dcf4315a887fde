// bf16 / fp16 MFMA GEMM, 64 x 64 block tile (2 x 2 waves).
#include "rp_gemm_mfma16_kernel.h"

namespace rp {

int launch_mfma16_64(const GemmArgs& g, const Plan& p, int dtype) { return m16_launch_tile_dtype<64, 64, 2>(g, p, dtype); }

// Both matrix gradients of a Linear layer in one launch: the first workgroups compute dX = dY . W^T (k-contiguous operands), the
// others dW = X^T . dY (free-index-contiguous ones), tile for tile what the two launches would do, so the same bits.
// A 64 x 64 tile is bound by the latency of its slab chain with one workgroup per CU (1024^3: 19.1 K cycles for 2.05 K of MFMA);
// two or three of them share a CU's LDS, and the two products' chains run side by side.
// bf16 layer of 1024 x 1024 x 1024 (bias too), forward and backward: 31.3 us with two launches, 24.6 with this one.
template <typename T, int EDGE, int PF>
__global__ void __launch_bounds__(256, m16_blocks_per_cu(64, 64, EDGE, PF)) linear_backward16_kernel(GemmArgs gx, GemmArgs gw, int x_tiles_m, int x_tiles_n, int w_tiles_m, int w_tiles_n, int x_slots, int w_slots) {
    const int b = blockIdx.x;
    if (b < x_slots) gemm_mfma16_block<T, 64, 64, 2, false, false, EDGE, false, PF>(gx, x_tiles_m, x_tiles_n, nullptr, 0, x_slots, b, 0, x_slots);
    else gemm_mfma16_block<T, 64, 64, 2, true, true, EDGE, false, PF>(gw, w_tiles_m, w_tiles_n, nullptr, 0, w_slots, b - x_slots, 0, w_slots);
}

template <typename T, int EDGE, int PF>
static int launch_linear_backward16_t(const GemmArgs& gx, const GemmArgs& gw) {
    const int xm = (gx.m + 63) / 64, xn = (gx.n + 63) / 64, wm = (gw.m + 63) / 64, wn = (gw.n + 63) / 64;
    const int x_slots = scheduled_grid(xm, xn), w_slots = scheduled_grid(wm, wn);
    constexpr size_t x_smem = m16_smem_bytes(64, 64, 2, false, false, 2, 32), w_smem = m16_smem_bytes(64, 64, 2, true, true, 2, 32);
    constexpr size_t smem = x_smem > w_smem ? x_smem : w_smem;
    static_assert(smem <= 64 * 1024, "no attribute needed");
    hipLaunchKernelGGL((linear_backward16_kernel<T, EDGE, PF>), dim3(x_slots + w_slots), dim3(256), smem, current_stream(), gx, gw, xm, xn, wm, wn, x_slots, w_slots);
    return check_launch("linear_backward16_kernel") ? 0 : -1;
}

template <typename T>
static int launch_linear_backward16_d(const GemmArgs& gx, const GemmArgs& gw, bool edge) {
    if (m16_deep(gx.k) && m16_deep(gw.k)) return edge ? launch_linear_backward16_t<T, M16_EDGE, M16_DEEP_SETS>(gx, gw) : launch_linear_backward16_t<T, M16_WHOLE, M16_DEEP_SETS>(gx, gw);
    return edge ? launch_linear_backward16_t<T, M16_EDGE, 1>(gx, gw) : launch_linear_backward16_t<T, M16_WHOLE, 1>(gx, gw);
}

int launch_linear_backward16(const GemmArgs& gx, const GemmArgs& gw, bool edge, int dtype) {
    return dtype == RP_DTYPE_BFLOAT16 ? launch_linear_backward16_d<bf16_t>(gx, gw, edge) : launch_linear_backward16_d<f16_t>(gx, gw, edge);
}

}  // namespace rp
