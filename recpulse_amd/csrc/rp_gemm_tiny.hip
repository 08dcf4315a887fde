// fp32 GEMMs whose whole output is a few hundred 16 x 16 tiles (the layers of a small MLP: 256 x 784 by 784 x 256 and
// smaller).  Such a product is over in microseconds, so what it costs is latency: a 64 x 64 tile leaves 240 CUs
// idle unless k is split over blocks, and a split needs a second launch (or a device-scope exchange) to add the
// partial tiles, which costs as much again as the multiplication.  Here a workgroup owns one 16 x 16 tile of C, its four
// waves each take a quarter of k with v_mfma_f32_16x16x4_f32, and the four partial tiles meet in LDS: one launch, a
// fixed order of additions, up to about a thousand workgroups in flight.  Operands are read straight from global
// memory with any strides (16-byte loads along k where k is the unit-stride axis, at any element: four loads of a value each, which
// rows of no whole vectors had before, made a backward of 935 x 213 x 862 take 44.6 us, 24.4 now); nothing is staged, every value is
// used once per workgroup.
#include "rp_column_sums.h"
#include "rp_gemm.h"

namespace rp {

typedef __attribute__((ext_vector_type(4))) float f32x4t_t;

// MFMA step j of a 16-deep chunk uses k = chunk + 4*(lane / 16) + j for the four k slots: a permutation of k that both
// operands share, chosen so that a lane's four values are consecutive in k.  p points at the lane's first value.
typedef f32x4t_t __attribute__((aligned(4))) f32x4_any_t;       // four values at any element
template <bool VEC>
__device__ __forceinline__ f32x4t_t tiny_load4(const float* p, long long k_stride) {
    if (VEC) return *(const f32x4_any_t*)p;
    return f32x4t_t{p[0], p[k_stride], p[2 * k_stride], p[3 * k_stride]};
}
// the same with zeros from k_end on
__device__ __forceinline__ f32x4t_t tiny_load4_masked(const float* p, long long k_stride, int k0, int k_end) {
    f32x4t_t v;
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = (k0 + j < k_end) ? p[(long long)j * k_stride] : 0.f;
    return v;
}

// U whole chunks from chunk c on: all of their loads are requested before the first is multiplied
template <bool A_VEC, bool B_VEC, int U>
__device__ __forceinline__ void tiny_chunks(f32x4t_t& acc, const float* ap, const float* bp, long long a_ks, long long b_ks, int c, int kq) {
    f32x4t_t a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const long long k0 = 16 * (c + u) + 4 * kq;
        a[u] = tiny_load4<A_VEC>(ap + k0 * a_ks, a_ks);
        b[u] = tiny_load4<B_VEC>(bp + k0 * b_ks, b_ks);
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][j], b[u][j], acc, 0, 0, 0);
}

// One 16 x 16 tile of C_z (tile row tm, tile column tn) by the 256 threads of a workgroup; red: 3 x 256 floats of LDS.
template <bool A_VEC, bool B_VEC>
__device__ __forceinline__ void tiny_tile(const GemmArgs& g, int z, int tm, int tn, float (*red)[256]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = lane >> 4;
    const int m0 = tm * 16, n0 = tn * 16;
    // rows past m and columns past n read the last valid row / column: their products land in output elements that
    // are never written
    const int row = m0 + r16 < g.m ? m0 + r16 : g.m - 1;
    const int col = n0 + r16 < g.n ? n0 + r16 : g.n - 1;
    const float* ap = (const float*)g.A + (long long)z * g.a_bs + (long long)row * g.a_rs;
    const float* bp = (const float*)g.B + (long long)z * g.b_bs + (long long)col * g.b_cs;

    // chunks of 16 k, a contiguous quarter of them per wave.  Every batch of loads is one memory round trip, which is most
    // of what such a product costs: up to eight chunks (64 values per lane) go in one batch.
    const int chunks = (g.k + 15) / 16, per_wave = (chunks + 3) / 4;
    const int c_begin = wave * per_wave, c_end = c_begin + per_wave < chunks ? c_begin + per_wave : chunks;
    const int whole = g.k / 16 < c_end ? g.k / 16 : c_end;         // chunks before this one are not cut off by the end of k
    f32x4t_t acc = {0.f, 0.f, 0.f, 0.f};
    f32x4t_t a_tail = {0.f, 0.f, 0.f, 0.f}, b_tail = {0.f, 0.f, 0.f, 0.f};
    const bool cut = c_end == chunks && c_begin < chunks && g.k % 16 != 0;
    if (cut) {                                                     // the cut-off chunk: requested first, multiplied last
        const int k0 = 16 * (chunks - 1) + 4 * kq;
        a_tail = tiny_load4_masked(ap + (long long)k0 * g.a_cs, g.a_cs, k0, g.k);
        b_tail = tiny_load4_masked(bp + (long long)k0 * g.b_rs, g.b_rs, k0, g.k);
    }
    int c = c_begin;
    for (; c + 8 <= whole; c += 8) tiny_chunks<A_VEC, B_VEC, 8>(acc, ap, bp, g.a_cs, g.b_rs, c, kq);
    switch (whole - c) {                                           // (negative when the wave has no whole chunk)
        case 7: tiny_chunks<A_VEC, B_VEC, 7>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 6: tiny_chunks<A_VEC, B_VEC, 6>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 5: tiny_chunks<A_VEC, B_VEC, 5>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 4: tiny_chunks<A_VEC, B_VEC, 4>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 3: tiny_chunks<A_VEC, B_VEC, 3>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 2: tiny_chunks<A_VEC, B_VEC, 2>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        case 1: tiny_chunks<A_VEC, B_VEC, 1>(acc, ap, bp, g.a_cs, g.b_rs, c, kq); break;
        default: break;
    }
    if (cut) {
#pragma unroll
        for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a_tail[j], b_tail[j], acc, 0, 0, 0);
    }

    // the four partial tiles meet in LDS and are added in wave order
    if (wave > 0) *(f32x4t_t*)&red[wave - 1][lane * 4] = acc;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < 3; w++) {
        const f32x4t_t part = *(const f32x4t_t*)&red[w][lane * 4];
        acc += part;
    }
    // accumulator register v of lane (kq, r16) is C[m0 + 4*kq + v][n0 + r16]
    const int gc = n0 + r16;
    if (gc >= g.n) return;
    const float* bias = (const float*)g.bias;
    const bool has_bias = bias != nullptr, accum = g.accumulate != 0;
    const float bv = has_bias ? bias[gc] : 0.f;
    float* cp = (float*)g.C + (long long)z * g.c_bs + (long long)gc * g.c_cs;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int gr = m0 + 4 * kq + v;
        if (gr >= g.m) break;
        float* p = cp + (long long)gr * g.c_rs;
        *p = finish<float>(acc[v], has_bias, bv, accum, accum ? *p : 0.f);
    }
}

template <bool A_VEC, bool B_VEC>
__global__ void __launch_bounds__(256) gemm_tiny32_kernel(GemmArgs g) {
    __shared__ float red[3][256];
    tiny_tile<A_VEC, B_VEC>(g, blockIdx.z, blockIdx.y, blockIdx.x, red);
}

// 16-byte loads along k need k to be the unit-stride axis; rows may start at any element
static bool tiny_a_vec(const GemmArgs& g) { return g.a_cs == 1; }
static bool tiny_b_vec(const GemmArgs& g) { return g.b_rs == 1; }

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

template <bool A_VEC, bool B_VEC>
__device__ __forceinline__ void tiny_tile_of(const GemmArgs& g, int tile, float (*red)[256]) {
    const int tiles_n = (g.n + 15) / 16;
    tiny_tile<A_VEC, B_VEC>(g, 0, tile / tiles_n, tile % tiles_n, red);
}

__device__ __forceinline__ void tiny_tile_any(const GemmArgs& g, bool a_vec, bool b_vec, int tile, float (*red)[256]) {
    if (a_vec && b_vec) tiny_tile_of<true, true>(g, tile, red);
    else if (a_vec) tiny_tile_of<true, false>(g, tile, red);
    else if (b_vec) tiny_tile_of<false, true>(g, tile, red);
    else tiny_tile_of<false, false>(g, tile, red);
}

__global__ void __launch_bounds__(256) linear_backward_tiny32_kernel(GemmArgs gx, GemmArgs gw, ColumnSums db, int tiles_x, int blocks_db, int vec_flags) {
    constexpr int DB_ROWS = COLSUM_CHUNK;
    using Tile = ColumnTile<float, DB_WIDTH, DB_ROWS>;
    __shared__ __attribute__((aligned(16))) float tile[DB_ROWS * Tile::COLS];       // column sums (16 KB: eight workgroups still share a CU); the GEMM tiles meet in its first 3 KB
    float (*red)[256] = (float (*)[256])tile;
    const int b = (int)blockIdx.x - blocks_db;           // the column sums go first: their chain of additions is the longest of any workgroup
    if (b >= 0 && b < tiles_x) { tiny_tile_any(gx, vec_flags & 1, vec_flags & 2, b, red); return; }
    if (b >= 0) { tiny_tile_any(gw, vec_flags & 4, vec_flags & 8, b - tiles_x, red); return; }
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
