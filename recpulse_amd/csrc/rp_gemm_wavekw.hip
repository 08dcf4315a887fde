// fp32 / fp64 MFMA GEMM whose waves share k: products of few tiles or a k that is long for them.
//
// A workgroup of eight waves owns one tile of 16 x 16 to 64 x 64 of the output, and wave w takes the pieces w, w + 8, ... of k, a cache line
// of every row that has unit stride along k: straight from memory into registers (16 rows of such an operand through LDS of the wave's own, so
// that its loads take whole lines), any element the rows may start at.  The eight partial tiles meet in LDS and are added in wave order.  One launch,
// no workspace.  Bound by what a CU takes in, 35 to 95 GB/s a CU behind 2.7 us of launch and latency, and from 64 x 64 tiles of 1024^3 on by the
// MFMAs (14.6 us of 25).  What it replaces staged 64 x 64 tiles slab by slab, one wave a SIMD, with a k split and a launch that adds it
// up in fp32 and without either in fp64.  us, before and here:
//   fp32 1024^3 30.4 / 25, 512^3 12.9 / 6.2, 935 x 862 x 398 32.0 / 12.9, 25 x 3120 x 2446 38.1 / 13.7, 32 x 8192 x 8192 141 / 60, 17 x 6048 x 173 (B^T)
//   190 / 11.1, 64 x 4096 x 1024 (B^T) 18.8 / 9.6; fp64 89 x 2787 x 286 390 / 15.5, 2054 x 1064 x 52 (B^T) 120 / 15, 512^3 (A^T) 25.9 / 8.7, 300^3 (B^T) 38 / 5.8.
// Over 330 drawn fp32 products 0.78 of the time, the slowest 1.03, over 170 fp64 ones 0.19 and 1.01.  k is summed in 8 to 64 chains, so the error against 64 bits is smaller than in one
// (1024^3 2.1e-7, 5.8e-7 before; 64 x 4096 x 1024 2.2e-7 and 3.0e-7); wavekw_takes leaves products alone whose kernel sums shorter chains.
#include "rp_column_sums.h"
#include "rp_gemm_tiny.h"
#include "rp_gemm_wavekw.h"

namespace rp {

// waves a SIMD whose registers have to fit: two workgroups on a CU, one of the 64 x 64 tile
constexpr int wkw_waves(int tiles) { return tiles <= 4 ? 4 : 2; }

template <typename E, bool A_KC, bool B_KC, int TM, int TN, int NW, bool SEG>
__global__ void __launch_bounds__(64 * NW, wkw_waves(TM * TN)) gemm_wavekw_kernel(GemmArgs g, int tiles_m, int tiles_n) {
    extern __shared__ __attribute__((aligned(16))) unsigned char wkw_lds[];
    gemm_wavekw_block<E, A_KC, B_KC, TM, TN, NW, SEG>(g, tiles_m, tiles_n, blockIdx.x, g.batch, wkw_lds);
}

template <typename E, bool A_KC, bool B_KC, int TM, int TN, int NW, bool SEG = false>
static int launch_wavekw_t(const GemmArgs& g) {
    constexpr size_t smem = wkw_smem<E, A_KC, B_KC, TM, TN, NW>();
    const int tiles_m = (g.m + 16 * TM - 1) / (16 * TM), tiles_n = (g.n + 16 * TN - 1) / (16 * TN);
    auto kern = gemm_wavekw_kernel<E, A_KC, B_KC, TM, TN, NW, SEG>;
    if (smem > 64 * 1024 && !check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem), "hipFuncSetAttribute")) return -1;
    hipLaunchKernelGGL(kern, dim3((unsigned)(((long long)tiles_m * tiles_n * g.batch + 7) / 8 * 8)), dim3(64 * NW), smem, current_stream(), g, tiles_m, tiles_n);
    return check_launch("gemm_wavekw_kernel") ? 0 : -1;
}

template <typename E, int TM, int TN, int NW>
static int launch_wavekw_layout(const GemmArgs& g) {
    const bool a_kc = wkw_a_kc(g), b_kc = wkw_b_kc(g);
    if (a_kc && !b_kc) return launch_wavekw_t<E, true, false, TM, TN, NW>(g);
    if (a_kc) return launch_wavekw_t<E, true, true, TM, TN, NW>(g);
    if (!b_kc) return launch_wavekw_t<E, false, false, TM, TN, NW>(g);
    return launch_wavekw_t<E, false, true, TM, TN, NW>(g);
}

// The tile with the least time over the drawn products (2 % from the best of all on the average): 32 x 32 where those occupy three quarters of the CUs (half in
// fp64), else 16 x 16, or 16 x 32 where an operand's k rows are read (its loads of 16 elements are half a line).  One 64 x 64 tile a CU with a k that is worth
// its prologue (1024^3 24 us, 28.5 on 32 x 32); 16 x 64 where one fills the chip once with a row-major B, whose lines it takes whole
// (128 x 5888 x 1600 27.9 us, 33.3 on 16 x 32; 935 x 862 x 398, 413 of them, 14.2 and 12.7 on 32 x 32).
constexpr long long WKW_MAX_SLOTS = (1ll << 32) / 512 - 8;       // workgroups of 512 threads in a launch of fewer than 2^32 threads, less what rounds them up to eights
WkwTile wavekw_tile(const GemmArgs& g, int dtype) {
    const bool a_kc = wkw_a_kc(g), b_kc = wkw_b_kc(g);
    if (!(a_kc || g.a_rs == 1) || !(b_kc || g.b_cs == 1) || g.batch > 65535) return WKW_NONE;
    const long long esz = (long long)dtype_size(dtype), cus = device_cu_count() > 0 ? device_cu_count() : 256, limit = 1ll << 31;
    // a tile is addressed with 32-bit byte offsets from its first row
    const auto span = [&](bool kc, long long fs, long long ks) { return ((kc ? 63 * fs + g.k : (long long)(g.k - 1) * ks + 64) * esz); };
    if (span(a_kc, g.a_rs, g.a_cs) >= limit || span(b_kc, g.b_cs, g.b_rs) >= limit) return WKW_NONE;
    const auto tiles = [&](int tm, int tn) { return (long long)((g.m + 16 * tm - 1) / (16 * tm)) * ((g.n + 16 * tn - 1) / (16 * tn)) * g.batch; };
    const auto fits = [&](int tm, int tn) { return (a_kc || g.m >= 16 * tm) && (b_kc || g.n >= 16 * tn); };       // see ms, ns in gemm_wavekw_block
    if (!fits(1, 1) || tiles(1, 1) >= 1ll << 24) return WKW_NONE;
    if (dtype == RP_DTYPE_FLOAT64 && fits(2, 2) && tiles(2, 2) >= cus / 2) return WKW_32X32;
    if (dtype != RP_DTYPE_FLOAT64) {
        if (fits(4, 4) && g.k >= 512 && tiles(4, 4) >= cus * 3 / 4 && tiles(4, 4) <= cus) return WKW_64X64;
        if (a_kc && !b_kc && fits(1, 4) && g.k >= 512 && tiles(1, 4) >= cus / 2 && tiles(1, 4) <= cus) return WKW_16X64;
        if (fits(2, 2) && tiles(2, 2) >= cus * 3 / 4) return WKW_32X32;
        if (!(a_kc && b_kc) && fits(1, 2) && tiles(1, 2) >= cus / 2) return tiles(1, 2) <= WKW_MAX_SLOTS ? WKW_16X32 : WKW_NONE;
    }
    return tiles(1, 1) <= WKW_MAX_SLOTS ? WKW_16X16 : WKW_NONE;       // (many tiles where an operand is only 16 to 31 wide)
}

const char* wavekw_name(WkwTile tile, int dtype) {
    if (dtype == RP_DTYPE_FLOAT64) return tile == WKW_32X32 ? "mfma64_wavek_32x32" : "mfma64_wavek_16x16";
    switch (tile) {
        case WKW_64X64: return "mfma32_wavek_64x64";
        case WKW_16X64: return "mfma32_wavek_16x64";
        case WKW_32X32: return "mfma32_wavek_32x32";
        case WKW_16X32: return "mfma32_wavek_16x32";
        case WKW_FEW_ROWS: return "mfma32_wavek_few_rows";
        default: return "mfma32_wavek_16x16";
    }
}

int launch_wavekw(const GemmArgs& g, WkwTile tile, int dtype) {
    if (dtype == RP_DTYPE_FLOAT64) return tile == WKW_32X32 ? launch_wavekw_layout<double, 2, 2, 8>(g) : launch_wavekw_layout<double, 1, 1, 8>(g);
    switch (tile) {
        case WKW_64X64: return launch_wavekw_layout<float, 4, 4, 8>(g);
        case WKW_16X64: return launch_wavekw_t<float, true, false, 1, 4, 8>(g);
        case WKW_32X32: return launch_wavekw_layout<float, 2, 2, 8>(g);
        case WKW_16X32: return launch_wavekw_layout<float, 1, 2, 8>(g);
        case WKW_FEW_ROWS: return g.k <= 640 ? launch_wavekw_t<float, true, false, 1, 2, 8>(g) : launch_wavekw_t<float, true, false, 1, 2, 16>(g);
        default: return launch_wavekw_layout<float, 1, 1, 8>(g);
    }
}

template <int TM, int TN>
static int launch_wavekw_segmented_t(const GemmArgs& g) {
    return g.seg_k > 0 ? launch_wavekw_t<float, true, false, TM, TN, 8, true>(g) : launch_wavekw_t<float, true, true, TM, TN, 8, true>(g);
}
int launch_wavekw_segmented(const GemmArgs& g, WkwTile tile) {
    switch (tile) {
        case WKW_64X64: return launch_wavekw_segmented_t<4, 4>(g);
        case WKW_32X32: return launch_wavekw_segmented_t<2, 2>(g);
        case WKW_16X32: return launch_wavekw_segmented_t<1, 2>(g);
        default: return launch_wavekw_segmented_t<1, 1>(g);
    }
}

// All gradients of a Linear layer in one launch: the first workgroups add up the columns of dY, then come the tiles of the product with the longer k,
// then the other's, each doing what it would do in a launch of its own, so the same bits.  What goes away is two launches of three, 4.7 us each
// behind another one.  fp32 layers with bias, forward and backward, us, apart and here: 512^3 22.1 / 17.4,
// 935 x 213 x 862 34.5 / 28.8, 64 x 4544 x 128 25.8 / 21.4; fp64 208 x 299 x 482 18.9 / 12.7.
// Either product may be on the 16 x 16 tiles of four waves, two of which share a workgroup.
template <WkwTile K> struct WkwShape { static constexpr int TM = K == WKW_32X32 ? 2 : 1, TN = K == WKW_32X32 || K == WKW_16X32 ? 2 : 1; };

template <typename E, WkwTile K, bool KC>
constexpr size_t wkw_part_smem() {
    if constexpr (K == WKW_TINY) return 2 * 3 * 256 * sizeof(float);
    else return wkw_smem<E, KC, KC, WkwShape<K>::TM, WkwShape<K>::TN, 8>();
}
// Slot `block` of one product: KC, KC for dX = dY . W^T, MC, MC for dW = X^T . dY
template <typename E, WkwTile K, bool KC>
__device__ __forceinline__ void wkw_part(const GemmArgs& g, int tiles_m, int tiles_n, int block, int vec_flags, unsigned char* lds) {
    if constexpr (K == WKW_TINY) {
        const int half = threadIdx.x >> 8, tile = 2 * block + half, tiles = tiles_m * tiles_n;
        if (2 * block >= tiles) return;
        tiny_tile_any(g, vec_flags & 1, vec_flags & 2, tile < tiles ? tile : tiles - 1, (float (*)[256])lds + 3 * half, threadIdx.x & 255, tile < tiles);
    } else {
        gemm_wavekw_block<E, KC, KC, WkwShape<K>::TM, WkwShape<K>::TN, 8>(g, tiles_m, tiles_n, block, 1, lds);
    }
}

template <typename E, WkwTile X, WkwTile W>
__global__ void __launch_bounds__(512, 4) linear_backward_wavekw_kernel(GemmArgs gx, GemmArgs gw, BiasGradient db, int x_tiles_m, int x_tiles_n, int w_tiles_m, int w_tiles_n, int x_slots, int w_slots, int x_first, int vec_flags) {
    extern __shared__ __attribute__((aligned(16))) unsigned char wkw_lds[];
    const int b = (int)blockIdx.x - db.blocks, first = x_first ? x_slots : w_slots;
    if (b < 0) {
        if ((int)blockIdx.x * StripSums<E, 512>::COLS < db.cols) StripSums<E, 512>::run((E*)db.out, (const E*)gx.A, gx.m, db.cols, db.accumulate, blockIdx.x, wkw_lds);
    } else if ((b < first) == (x_first != 0)) {
        wkw_part<E, X, true>(gx, x_tiles_m, x_tiles_n, b < first ? b : b - first, vec_flags, wkw_lds);
    } else {
        wkw_part<E, W, false>(gw, w_tiles_m, w_tiles_n, b < first ? b : b - first, vec_flags >> 2, wkw_lds);
    }
}

template <typename E, WkwTile X, WkwTile W>
static int launch_linear_backward_wavekw_t(const GemmArgs& gx, const GemmArgs& gw, void* db, int accumulate_db) {
    const int xm = (gx.m + 16 * WkwShape<X>::TM - 1) / (16 * WkwShape<X>::TM), xn = (gx.n + 16 * WkwShape<X>::TN - 1) / (16 * WkwShape<X>::TN);
    const int wm = (gw.m + 16 * WkwShape<W>::TM - 1) / (16 * WkwShape<W>::TM), wn = (gw.n + 16 * WkwShape<W>::TN - 1) / (16 * WkwShape<W>::TN);
    // whole rounds of the XCDs, so that the tiles' workgroups stay where their schedules want them
    const auto slots = [](WkwTile k, int tiles) { return ((k == WKW_TINY ? (tiles + 1) / 2 : tiles) + 7) / 8 * 8; };
    const BiasGradient sums{db, gx.k, accumulate_db, db ? ((gx.k - 1) / StripSums<E, 512>::COLS + 8) / 8 * 8 : 0};
    constexpr size_t xs = wkw_part_smem<E, X, true>(), ws = wkw_part_smem<E, W, false>(), part = xs > ws ? xs : ws, smem = part > StripSums<E, 512>::LDS ? part : StripSums<E, 512>::LDS;
    static_assert(smem <= 64 * 1024, "no attribute needed");
    const int x_slots = slots(X, xm * xn), w_slots = slots(W, wm * wn);
    const int flags = (tiny_a_vec(gx) ? 1 : 0) | (tiny_b_vec(gx) ? 2 : 0) | (tiny_a_vec(gw) ? 4 : 0) | (tiny_b_vec(gw) ? 8 : 0);
    hipLaunchKernelGGL((linear_backward_wavekw_kernel<E, X, W>), dim3(sums.blocks + x_slots + w_slots), dim3(512), smem, current_stream(), gx, gw, sums, xm, xn, wm, wn, x_slots, w_slots, gx.k >= gw.k, flags);
    return check_launch("linear_backward_wavekw_kernel") ? 0 : -1;
}

bool linear_backward_wavekw_takes(const GemmArgs& gx, const GemmArgs& gw, WkwTile x, WkwTile w, int dtype) {
    const auto tiles16 = [](const GemmArgs& g) { return (long long)((g.m + 15) / 16) * ((g.n + 15) / 16); };
    if (tiles16(gx) + tiles16(gw) + gx.k / 8 + 16 > WKW_MAX_SLOTS) return false;
    const bool f32 = dtype == RP_DTYPE_FLOAT32;
    const auto small = [&](WkwTile k) { return k == WKW_16X16 || k == WKW_32X32 || (f32 && k == WKW_TINY); };
    return small(x) && (small(w) || (f32 && w == WKW_16X32)) && !(x == WKW_TINY && w == WKW_TINY);
}

template <typename E, WkwTile X>
static int launch_linear_backward_wavekw_x(const GemmArgs& gx, const GemmArgs& gw, WkwTile w, void* db, int accumulate_db) {
    if constexpr (sizeof(E) == 4) {
        if (w == WKW_16X32) return launch_linear_backward_wavekw_t<E, X, WKW_16X32>(gx, gw, db, accumulate_db);
        if constexpr (X != WKW_TINY)
            if (w == WKW_TINY) return launch_linear_backward_wavekw_t<E, X, WKW_TINY>(gx, gw, db, accumulate_db);
    }
    return w == WKW_32X32 ? launch_linear_backward_wavekw_t<E, X, WKW_32X32>(gx, gw, db, accumulate_db) : launch_linear_backward_wavekw_t<E, X, WKW_16X16>(gx, gw, db, accumulate_db);
}

int launch_linear_backward_wavekw(const GemmArgs& gx, const GemmArgs& gw, WkwTile x, WkwTile w, void* db, int accumulate_db, int dtype) {
    if (dtype == RP_DTYPE_FLOAT64) return x == WKW_32X32 ? launch_linear_backward_wavekw_x<double, WKW_32X32>(gx, gw, w, db, accumulate_db) : launch_linear_backward_wavekw_x<double, WKW_16X16>(gx, gw, w, db, accumulate_db);
    switch (x) {
        case WKW_TINY: return launch_linear_backward_wavekw_x<float, WKW_TINY>(gx, gw, w, db, accumulate_db);
        case WKW_32X32: return launch_linear_backward_wavekw_x<float, WKW_32X32>(gx, gw, w, db, accumulate_db);
        default: return launch_linear_backward_wavekw_x<float, WKW_16X16>(gx, gw, w, db, accumulate_db);
    }
}

}  // namespace rp
