// bf16 / fp16 MFMA GEMM, 64 x 64 block tile (2 x 2 waves).
#include "rp_column_sums.h"
#include "rp_gemm_mfma16_kernel.h"
#include "rp_gemm_mfma16_wavek.h"

namespace rp {

int launch_mfma16_64(const GemmArgs& g, const Plan& p, int dtype) { return m16_launch_tile_dtype<64, 64, 2>(g, p, dtype); }

// All gradients of a Linear layer in one launch: the first workgroups add up the columns of dY (their chain of chunks is the longest of
// any), the next ones compute dX = dY . W^T (k-contiguous operands), the others dW = X^T . dY (free-index-contiguous ones), tile for
// tile and chunk for chunk what separate launches would do, so the same bits.
// A 64 x 64 tile is bound by the latency of its slab chain with one workgroup per CU (1024^3: 19.1 K cycles for 2.05 K of MFMA);
// two or three of them share a CU's LDS, and the two products' chains run side by side.
// bf16 layer of 1024 x 1024 x 1024 (bias too), forward and backward: 31.3 us with a launch per gradient, 24.6 with the matrices in one,
// 21 with the column sums in it too.  (Three slabs in flight, as for a product with one workgroup per CU, give nothing here:
// 768 x 768 x 768 8.6 us either way, 1280 x 768 x 1280 15.7 and 16.6.)
// DX: how a workgroup makes its tile of dX.  Few tiles with a deep k are cut up as the separate product would cut them (WavekTile), by four
// waves with two or four shares of k each; all others are 64 x 64 ones.  dW's chains are the longer ones then and go first (512 x 512 x 640
// 7.3 us, 7.9 with dX first).  bf16 layer with bias of m x k x n, us, dX on 64 x 64 tiles, in a launch of its own, and here:
// 64 x 1024 x 1024 6.8 / 7.2 / 4.3, 256 x 256 x 4096 23 / 12 / 8.4, 512 x 512 x 640 6.8 / 11.1 / 6.8, 1024 x 256 x 640 10.9 / 16.1 / 11.7
// (the column sums' chain, beside more workgroups than before).
// Ragged rows do the same through the ragged variants (119 x 57 x 245 a layer's forward and backward 22.1 us, 9.6 now; 754 x 43 x 201 23.5 / 14.5; 280 x 610 x 2347 42 / 24).
constexpr int DX_64X64 = -1;
template <int DX>
struct WavekShape {
    static constexpr int TM = DX == WK_32X16 || DX == WK_32X32 ? 2 : 1, TN = DX == WK_32X32 ? 2 : 1, NW = DX == WK_16X16_16 ? 16 : 8;
    static constexpr int SMEM = wk_smem<TM, TN, NW, false, 4>();
};

template <typename T, int EDGE, int DX>
__global__ void __launch_bounds__(256) linear_backward16_kernel(GemmArgs gx, GemmArgs gw, BiasGradient db, int x_tiles_m, int x_tiles_n, int w_tiles_m, int w_tiles_n, int x_slots, int w_slots) {
    constexpr bool WAVEK = DX != DX_64X64;
    const int b = (int)blockIdx.x - db.blocks, x_slot = WAVEK ? b - w_slots : b, w_slot = WAVEK ? b : b - x_slots;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    if (b < 0) {
        if ((int)blockIdx.x * StripSums<T, 256>::COLS < db.cols) StripSums<T, 256>::run((T*)db.out, (const T*)gx.A, gx.m, db.cols, db.accumulate, blockIdx.x, (unsigned char*)smem);
    } else if (WAVEK ? w_slot < w_slots : x_slot >= x_slots) {
        gemm_mfma16_block<T, 64, 64, 2, true, true, EDGE, false, 1>(gw, w_tiles_m, w_tiles_n, nullptr, 0, w_slots, w_slot, 0, w_slots);
    } else if constexpr (WAVEK) {
        gemm_mfma16_wavek_block<T, WavekShape<DX>::TM, WavekShape<DX>::TN, WavekShape<DX>::NW, false, 4, EDGE == M16_RAGGED>(gx, x_tiles_m, x_tiles_n, x_slot, smem);
    } else {
        gemm_mfma16_block<T, 64, 64, 2, false, false, EDGE, false, 1>(gx, x_tiles_m, x_tiles_n, nullptr, 0, x_slots, x_slot, 0, x_slots);
    }
}

template <typename T, int EDGE, int DX>
static int launch_linear_backward16_t(const GemmArgs& gx, const GemmArgs& gw, void* db, int accumulate_db) {
    constexpr bool wavek = DX != DX_64X64;
    constexpr int rows = wavek ? 16 * WavekShape<DX>::TM : 64, cols = wavek ? 16 * WavekShape<DX>::TN : 64;
    const int xm = (gx.m + rows - 1) / rows, xn = (gx.n + cols - 1) / cols, wm = (gw.m + 63) / 64, wn = (gw.n + 63) / 64;
    const int x_slots = wavek ? (xm * xn + 7) / 8 * 8 : scheduled_grid(xm, xn), w_slots = scheduled_grid(wm, wn);
    constexpr size_t x_smem = wavek ? WavekShape<DX>::SMEM : m16_smem_bytes(64, 64, 2, false, false, 2, 32), w_smem = m16_smem_bytes(64, 64, 2, true, true, 2, 32);
    constexpr size_t smem = x_smem > w_smem ? x_smem : w_smem;
    static_assert(StripSums<T, 256>::LDS <= smem, "the column sums use the tiles' LDS");
    // whole rounds of the XCDs, so that the tiles' workgroups stay where the schedule wants them
    const BiasGradient sums{db, gx.k, accumulate_db, db ? ((gx.k - 1) / StripSums<T, 256>::COLS + 8) / 8 * 8 : 0};
    static_assert(smem <= 64 * 1024, "no attribute needed");
    hipLaunchKernelGGL((linear_backward16_kernel<T, EDGE, DX>), dim3(sums.blocks + x_slots + w_slots), dim3(256), smem, current_stream(), gx, gw, sums, xm, xn, wm, wn, x_slots, w_slots);
    return check_launch("linear_backward16_kernel") ? 0 : -1;
}

template <typename T, int EDGE>
static int launch_linear_backward16_edge(const GemmArgs& gx, const GemmArgs& gw, bool dx_wavek, void* db, int accumulate_db) {
    switch (dx_wavek ? (int)wavek_tile(gx) : DX_64X64) {
        case WK_16X16_16: return launch_linear_backward16_t<T, EDGE, WK_16X16_16>(gx, gw, db, accumulate_db);
        case WK_16X16: return launch_linear_backward16_t<T, EDGE, WK_16X16>(gx, gw, db, accumulate_db);
        case WK_32X16: return launch_linear_backward16_t<T, EDGE, WK_32X16>(gx, gw, db, accumulate_db);
        case WK_32X32: return launch_linear_backward16_t<T, EDGE, WK_32X32>(gx, gw, db, accumulate_db);
        default: return launch_linear_backward16_t<T, EDGE, DX_64X64>(gx, gw, db, accumulate_db);
    }
}

template <typename T>
static int launch_linear_backward16_type(const GemmArgs& gx, const GemmArgs& gw, bool dx_wavek, void* db, int accumulate_db, bool edge, bool ragged) {
    if (ragged) return launch_linear_backward16_edge<T, M16_RAGGED>(gx, gw, dx_wavek, db, accumulate_db);
    return edge ? launch_linear_backward16_edge<T, M16_EDGE>(gx, gw, dx_wavek, db, accumulate_db) : launch_linear_backward16_edge<T, M16_WHOLE>(gx, gw, dx_wavek, db, accumulate_db);
}

// gx.A is dY [gx.m, gx.k], dense; dx_wavek: the product alone would go to the kernel whose waves split k; edge, ragged: of the 64 x 64 tiles;
// db: gx.k column sums of dY, or null
int launch_linear_backward16(const GemmArgs& gx, const GemmArgs& gw, bool dx_wavek, void* db, int accumulate_db, bool edge, bool ragged, int dtype) {
    if (dtype == RP_DTYPE_BFLOAT16) return launch_linear_backward16_type<bf16_t>(gx, gw, dx_wavek, db, accumulate_db, edge, ragged);
    return launch_linear_backward16_type<f16_t>(gx, gw, dx_wavek, db, accumulate_db, edge, ragged);
}

}  // namespace rp
