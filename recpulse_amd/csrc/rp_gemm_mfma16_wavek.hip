// bf16 / fp16 MFMA GEMM for few output tiles and deep k, A k-contiguous (a small batch's y = x . W and dX = dY . W^T): the waves of a
// workgroup split k.
//
// A workgroup owns one 16 TM x 16 TN tile of the output.  Wave w takes the 64-element pieces w, w + NW, ... of k, a cache line of
// every row: it loads U of them at once, eight whole lines an instruction, turns a piece into fragments through LDS of its
// own (a wave's LDS operations are executed in order: no barrier), and the NW partial tiles meet in LDS and are added in wave order.  One
// launch, no workspace.  Bound by what a CU can load, (TM + TN) * 32 * k bytes (256 KB: 2.3 us) behind 3.5 us of launch and latency.
// (Loading in the fragments' own layout, sixteen half lines an instruction and no LDS, took twice as long for them: 64 x 4096 x 1024 9.4 us, not 5.7.)
// bf16, us, before (64 x 64 tiles, or a k split over workgroups and a launch that adds it up) and here: 64 x 4096 x 1024 10.3 / 5.7,
// 256 x 4096 x 256 16.5 / 6.0, 64 x 1024 x 4096 7.0 / 5.0, 512 x 1024 x 512 6.9 / 4.8, 33 x 5000 x 72 25.2 / 6.3, 32 x 8192 x 8192 37.6 / 29.3;
// B row-major (k x 128 bytes of it a workgroup) 64 x 1024 x 4096 7.1 / 5.4, 256 x 4096 x 256 17.5 / 11.8, 300 x 1536 x 304 11.2 / 6.8, 33 x 5000 x 72 25.7 / 11.5.
#include "rp_gemm_mfma16_wavek.h"

namespace rp {

template <typename T, int TM, int TN, int NW, bool B_MC, bool RAGGED>
__global__ void __launch_bounds__(64 * NW) gemm_mfma16_wavek_kernel(GemmArgs g, int tiles_m, int tiles_n) {
    extern __shared__ __attribute__((aligned(16))) uint16_t wk_lds[];
    gemm_mfma16_wavek_block<T, TM, TN, NW, B_MC, NW, RAGGED>(g, tiles_m, tiles_n, blockIdx.x, wk_lds);
}

template <typename T, bool RAGGED, int TM, int TN, int NW, bool B_MC = false>
static int launch_wavek_t(const GemmArgs& g) {
    constexpr int smem = wk_smem<TM, TN, NW, B_MC>();
    const int tiles_m = (g.m + 16 * TM - 1) / (16 * TM), tiles_n = (g.n + 16 * TN - 1) / (16 * TN);
    auto kern = gemm_mfma16_wavek_kernel<T, TM, TN, NW, B_MC, RAGGED>;
    if (smem > 64 * 1024 && !check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem), "hipFuncSetAttribute")) return -1;
    hipLaunchKernelGGL(kern, dim3((unsigned)((tiles_m * tiles_n + 7) / 8 * 8)), dim3(64 * NW), smem, current_stream(), g, tiles_m, tiles_n);
    return check_launch("gemm_mfma16_wavek_kernel") ? 0 : -1;
}

template <typename T, bool RAGGED>
static int launch_wavek_type(const GemmArgs& g) {
    // B row-major: four waves where eight would leave some without a piece (us, four and eight: 7 x 608 x 152 4.9 / 5.3, 256 x 1024 x 256
    // 5.6 / 5.4; tiles of twice the rows 6.2 for 64 x 1024 x 4096, not 5.4)
    if (g.b_rs != 1) return g.k < 1024 ? launch_wavek_t<T, RAGGED, 1, 4, 4, true>(g) : launch_wavek_t<T, RAGGED, 1, 4, 8, true>(g);
    switch (wavek_tile(g)) {
        case WK_16X16_16: return launch_wavek_t<T, RAGGED, 1, 1, 16>(g);
        case WK_16X16: return launch_wavek_t<T, RAGGED, 1, 1, 8>(g);
        case WK_32X16: return launch_wavek_t<T, RAGGED, 2, 1, 8>(g);
        default: return launch_wavek_t<T, RAGGED, 2, 2, 8>(g);
    }
}

int launch_mfma16_wavek(const GemmArgs& g, bool ragged, int dtype) {
    if (dtype == RP_DTYPE_BFLOAT16) return ragged ? launch_wavek_type<bf16_t, true>(g) : launch_wavek_type<bf16_t, false>(g);
    return ragged ? launch_wavek_type<f16_t, true>(g) : launch_wavek_type<f16_t, false>(g);
}

}  // namespace rp
