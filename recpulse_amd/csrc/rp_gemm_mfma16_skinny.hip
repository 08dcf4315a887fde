// bf16 / fp16 GEMMs with few rows and deep k: the cost is streaming B once from HBM.
//
// Row-major A times row-major B with at most 32 rows takes the streaming kernel (rp_gemm_mfma16_stream128.hip), in
// which B never touches LDS and the k splits are added inside the same launch by the last block to arrive.  Other
// operand layouts, more rows, and the shapes that kernel declines take the tiled kernel with a 32 x 128 block tile
// below, whose fp32 partials a second kernel combines.  Both split k across the grid so that enough waves stream B to
// saturate HBM, and both add the splits in split order.
#include "rp_gemm_mfma16_kernel.h"


namespace rp {

template <typename T, int EDGE>
static int launch_skinny16_t(const GemmArgs& g, const Plan& p, float* partials, int nsplit, int k_per_split) {
    constexpr int BM = 32, BN = 128, WGM = 1;
    if (!p.a_mc && p.b_mc) return m16_launch<T, BM, BN, WGM, false, true, EDGE, true>(g, partials, nsplit, k_per_split);
    if (!p.a_mc && !p.b_mc) return m16_launch<T, BM, BN, WGM, false, false, EDGE, true>(g, partials, nsplit, k_per_split);
    if (p.a_mc && p.b_mc) return m16_launch<T, BM, BN, WGM, true, true, EDGE, true>(g, partials, nsplit, k_per_split);
    return m16_launch<T, BM, BN, WGM, true, false, EDGE, true>(g, partials, nsplit, k_per_split);
}

static int skinny16_splits(int batch, int m, int k, int n, int& k_per_split) {
    constexpr int BN = 128;
    const int tiles = ((n + BN - 1) / BN) * ((m + 31) / 32) * batch;
    // about three blocks per CU in flight, each split at least four slabs deep
    int nsplit = (768 + tiles - 1) / tiles;
    int max_split = k / (4 * M16_BK) > 0 ? k / (4 * M16_BK) : 1;
    if (nsplit > max_split) nsplit = max_split;
    k_per_split = ((k + nsplit - 1) / nsplit + M16_BK - 1) / M16_BK * M16_BK;
    return (k + k_per_split - 1) / k_per_split;
}

size_t skinny16_workspace(int batch, int m, int k, int n) {
    int k_per_split;
    return (size_t)batch * skinny16_splits(batch, m, k, n, k_per_split) * m * n * sizeof(float);
}

int launch_mfma16_skinny(const GemmArgs& g, const Plan& p, int dtype) {
    if (dtype != RP_DTYPE_BFLOAT16 && dtype != RP_DTYPE_FLOAT16) { set_error("mfma16 skinny GEMM: unsupported dtype %d", dtype); return -1; }
    if (!p.ragged && !p.a_mc && p.b_mc && stream128_takes(g)) return launch_stream128(g, dtype);
    int k_per_split;
    const int nsplit = skinny16_splits(g.batch, g.m, g.k, g.n, k_per_split);
    void* ws = nullptr;
    if (gemm_workspace(&ws, (size_t)g.batch * nsplit * g.m * g.n * sizeof(float)) != 0) return -1;
    int rc;
    const bool bf = dtype == RP_DTYPE_BFLOAT16;
    if (p.ragged) rc = bf ? launch_skinny16_t<bf16_t, M16_RAGGED>(g, p, (float*)ws, nsplit, k_per_split) : launch_skinny16_t<f16_t, M16_RAGGED>(g, p, (float*)ws, nsplit, k_per_split);
    else rc = bf ? launch_skinny16_t<bf16_t, M16_EDGE>(g, p, (float*)ws, nsplit, k_per_split) : launch_skinny16_t<f16_t, M16_EDGE>(g, p, (float*)ws, nsplit, k_per_split);
    if (rc == 0) rc = launch_splitk_combine(g, (const float*)ws, nsplit, g.m, dtype);
    gemm_workspace_release(ws);          // back to the pool while the kernels are still queued: safe for later work on this stream; held with the graph while one is being recorded
    return rc;
}

}  // namespace rp
