// fp32 GEMMs whose whole output is a few hundred 16 x 16 tiles (the layers of a small MLP: 256 x 784 by 784 x 256 and
// smaller).  Such a product is over in microseconds, so what it costs is latency: a 64 x 64 tile leaves 240 CUs
// idle unless k is split over blocks, and a split needs a second launch (or a device-scope exchange) to add the
// partial tiles, which costs as much again as the multiplication.  Here a workgroup owns one 16 x 16 tile of C, its four
// waves each take a quarter of k with v_mfma_f32_16x16x4_f32, and the four partial tiles meet in LDS: one launch, a
// fixed order of additions, up to about a thousand workgroups in flight.  Operands are read straight from global
// memory with any strides (16-byte loads along k where k is the unit-stride axis, at any element: four loads of a value each, which
// rows of no whole vectors had before, made a backward of 935 x 213 x 862 take 44.6 us here, 24.4 with vectors; waves that share k have
// it now, 19.8); nothing is staged, every value is
// used once per workgroup.
#include "rp_column_sums.h"
#include "rp_gemm_tiny.h"

namespace rp {

template <bool A_VEC, bool B_VEC>
__global__ void __launch_bounds__(256) gemm_tiny32_kernel(GemmArgs g) {
    __shared__ float red[3][256];
    tiny_tile<A_VEC, B_VEC>(g, blockIdx.z, blockIdx.y, blockIdx.x, red, threadIdx.x);
}

// The backward of a small Linear layer in one launch: the tiles of dX = dY . W^T, then the tiles of dW = X^T . dY, then
// the column sums of dY for db (in reduce_rows' order).  Every block
// does what it would have done in three separate launches, so the bits are the same; what goes away is two launch
// latencies, which is most of the time of such a layer.  Either GEMM or the sums may be absent (zero tiles / blocks).
constexpr int DB_WIDTH = 64;            // bytes of a row that one workgroup sums
struct ColumnSums {
    float* out;
    const float* grad;       // [rows, cols], dense
    int rows, cols, accumulate;
};

__global__ void __launch_bounds__(256) linear_backward_tiny32_kernel(GemmArgs gx, GemmArgs gw, ColumnSums db, int tiles_x, int blocks_db, int vec_flags) {
    constexpr int DB_ROWS = COLSUM_CHUNK;
    using Tile = ColumnTile<float, DB_WIDTH, DB_ROWS>;
    __shared__ __attribute__((aligned(16))) float tile[DB_ROWS * Tile::COLS];       // column sums (16 KB: eight workgroups still share a CU); the GEMM tiles meet in its first 3 KB
    float (*red)[256] = (float (*)[256])tile;
    const int b = (int)blockIdx.x - blocks_db;           // the column sums go first: their chain of additions is the longest of any workgroup
    if (b >= 0 && b < tiles_x) { tiny_tile_any(gx, vec_flags & 1, vec_flags & 2, b, red, threadIdx.x); return; }
    if (b >= 0) { tiny_tile_any(gw, vec_flags & 4, vec_flags & 8, b - tiles_x, red, threadIdx.x); return; }
    // column sums in the order of rp_column_sums.h, a chunk of 256 rows per tile: the next one is on its way while the first
    // wave adds this one.  Its 64 lanes are 16 columns times the four runs of a chunk, so the runs are added side by side
    // (one after another, with two tiles a chunk, 768 rows took 3 us longer).
    constexpr int COLS = Tile::COLS;
    static_assert(COLS * (COLSUM_CHUNK / COLSUM_RUN) == 64, "one wave adds the runs of a chunk");
    const int t = threadIdx.x, c0 = (int)blockIdx.x * COLS, col = t % COLS, run = t / COLS;
    float total = 0.f;
    Tile regs;
    regs.load(db.grad, 0, db.rows, c0, db.cols, t);
    for (int r = 0; r < db.rows; r += DB_ROWS) {
        regs.store(tile, t);
        __syncthreads();
        if (r + DB_ROWS < db.rows) regs.load(db.grad, r + DB_ROWS, db.rows, c0, db.cols, t);
        if (db.rows <= COLSUM_CHUNK) {
            if (t < COLS) total = Tile::add(0.f, tile, col, db.rows);
        } else if (t < 64) {
            const int n = db.rows - r - run * COLSUM_RUN;
            const float s = n > 0 ? Tile::add(0.f, tile + run * COLSUM_RUN * COLS, col, n < COLSUM_RUN ? n : COLSUM_RUN) : 0.f;
            float chunk = 0.f;
#pragma unroll
            for (int q = 0; q < COLSUM_CHUNK / COLSUM_RUN; q++) chunk += __shfl(s, q * COLS + col);       // (a run past the last row adds nothing)
            total += chunk;
        }
        __syncthreads();
    }
    if (t < COLS && c0 + col < db.cols) db.out[c0 + col] = db.accumulate ? db.out[c0 + col] + total : total;
}

// gx / gw: batch 1, fp32, each taken by the tiny kernel on its own (the caller checks); m == 0 marks an absent GEMM,
// cols == 0 absent sums.
int launch_linear_backward_tiny(const GemmArgs& gx, const GemmArgs& gw, void* db, const void* dy, int rows, int cols, int accumulate_db) {
    const int tiles_x = gx.m > 0 ? ((gx.m + 15) / 16) * ((gx.n + 15) / 16) : 0;
    const int tiles_w = gw.m > 0 ? ((gw.m + 15) / 16) * ((gw.n + 15) / 16) : 0;
    const int blocks_db = db ? (cols + DB_WIDTH / 4 - 1) / (DB_WIDTH / 4) : 0;
    if (tiles_x + tiles_w + blocks_db == 0) return 0;
    ColumnSums cs{(float*)db, (const float*)dy, rows, db ? cols : 0, accumulate_db};
    const int flags = (gx.m > 0 && tiny_a_vec(gx) ? 1 : 0) | (gx.m > 0 && tiny_b_vec(gx) ? 2 : 0) | (gw.m > 0 && tiny_a_vec(gw) ? 4 : 0) | (gw.m > 0 && tiny_b_vec(gw) ? 8 : 0);
    hipLaunchKernelGGL(linear_backward_tiny32_kernel, dim3(tiles_x + tiles_w + blocks_db), dim3(256), 0, current_stream(), gx, gw, cs, tiles_x, blocks_db, flags);
    return check_launch("linear_backward_tiny32_kernel") ? 0 : -1;
}

int launch_tiny(const GemmArgs& g, int dtype) {
    if (dtype != RP_DTYPE_FLOAT32) { set_error("tiny GEMM: float32 only (dtype %d)", dtype); return -1; }
    const dim3 grid((g.n + 15) / 16, (g.m + 15) / 16, g.batch);
    if (grid.y > 65535 || grid.z > 65535) { set_error("tiny GEMM: output too large for the grid"); return -1; }
    const bool a_vec = tiny_a_vec(g), b_vec = tiny_b_vec(g);
    if (a_vec && b_vec) hipLaunchKernelGGL((gemm_tiny32_kernel<true, true>), grid, dim3(256), 0, current_stream(), g);
    else if (a_vec) hipLaunchKernelGGL((gemm_tiny32_kernel<true, false>), grid, dim3(256), 0, current_stream(), g);
    else if (b_vec) hipLaunchKernelGGL((gemm_tiny32_kernel<false, true>), grid, dim3(256), 0, current_stream(), g);
    else hipLaunchKernelGGL((gemm_tiny32_kernel<false, false>), grid, dim3(256), 0, current_stream(), g);
    return check_launch("gemm_tiny32_kernel") ? 0 : -1;
}

}  // namespace rp
