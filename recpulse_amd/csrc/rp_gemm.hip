// GEMM kernels for gfx950 and their dispatcher.
//
//   C_z[m,n] = A_z[m,k] · B_z[k,n] (+ bias[n]) (+ C_z)      z in [0, batch)
//
// Operands are described by (batch, row, column) strides in elements, so
// transposed and permuted views are read in place.  Each operand is in one of
// two fast layouts, chosen from its strides:
//   KC  the reduction (k) axis is the unit-stride one      (A row-major, or Bᵀ stored)
//   MC  the free (m or n) axis is the unit-stride one       (B row-major, or Aᵀ stored)
// Rows that are no whole number of 16-byte vectors, or start at any element, have
// "ragged" variants of the MFMA kernels.  Anything else (both strides > 1, rows that
// overlap, small outputs between small ragged operands) takes the generic strided kernel.
//
// Kernel families:
//   mfma16   bf16 / fp16 inputs, fp32 accumulate, v_mfma_f32_32x32x16_{bf16,f16};
//            KC tiles are read from LDS with ds_read_b128, MC tiles with the
//            transposing ds_read_b64_tr_b16, so no layout needs a copy.
//   mfmaw    fp32 (v_mfma_f32_32x32x2_f32) and fp64 (v_mfma_f64_16x16x4_f64).
//   split32  fp32 outputs of 128 x 128 tiles on the bf16 matrix cores, every value split in three (a kernel of family mfmaw).
//   skinny   m <= 8 against a row-major B: a split-k streaming kernel bound by HBM.
//   tiny     fp32 outputs of a few hundred 16 x 16 tiles: one launch, k split over the waves of a workgroup.
//   wavekw   fp32 / fp64 products of few tiles, or a k that is long for them: the waves of a workgroup share k.
//   generic  any strides, any shape; LDS-tiled scalar FMA.
#include "rp_gemm.h"
#include "rp_gemm_wavekw.h"

#include <mutex>

namespace rp {

// ============================================================================
// dispatch
// ============================================================================
static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// rows up to which a deep 16-bit GEMM with few output tiles splits k
constexpr int SKINNY_MAX_ROWS = 128;

// Tile counts that decide between kernels stand for "one tile per CU" and "half of the CUs": they follow the device
// (whole rounds of the 8 XCDs, as the launchers size their grids); 256 where no device can be asked.
static int cu_tiles() {
    const int n = device_cu_count() / 8 * 8;
    return n >= 8 ? n : 256;
}

// Whether 128 x 128 tiles are faster than 256 x 256 ones, by what the CU with the most tiles takes.  us on one CU, measured: a slab of
// the large tile 1.32 while at most three quarters of the CUs have one, 1.55 (the power limit) when all do, and 7 a tile for its
// prologue and epilogue, 16 where the tile hangs over the output (that kernel spills registers); a slab of the small tile 0.53 and
// 1.2 a tile with two of them on a CU, 0.62 and 2 alone, a fifth more where small tiles hang over the output or k, a third with both
// operands k-contiguous (3600 x 816 x 7904 that way 80 / 109, 3368 x 5960 x 3440 fp16, A^T and B^T, 175 / 212), and a tenth more from five tiles
// a CU on (the power limit again: 7168 x 6144 x 2944 fp16 315 / 386).  The large tile keeps what is within 5 % (and ragged rows, whose
// loads take twice as long to issue: it issues half as many).  Over 450 drawn outputs the choice costs 1.7 % against the better of the two
// and saves 11 % against large tiles alone.  bf16, us, 256 and 128:
// 8000 x 1152 x 1024 46.7 / 27.3, 5696 x 384 x 3584 50.8 / 28.8, 3328 x 640 x 5056 65.9 / 35.4, 4096 x 8192 x 2048 171 / 141,
// 6144 x 1024 x 4096 62.1 / 59.4; 3072^3 71.8 / 77.7, 4096^3 108 / 140, 7808 x 3520 x 4928 279 / 292.  From six slabs on: below, the
// two are a microsecond or two apart (3072 x 256 x 3072 15.8 / 14.1).
static bool small_tiles_win(long long tiles256, long long tiles128, int m, int n, int k, bool both_kc) {
    const int cus = cu_tiles();
    const double slabs = (k + M16_BK - 1) / M16_BK;
    if (slabs < 6) return false;
    const long long most256 = (tiles256 + cus - 1) / cus, most128 = (tiles128 + cus - 1) / cus;
    const bool hangs_over = m % 256 || n % 256 || k % M16_BK, hangs_over128 = m % 128 || n % 128 || k % M16_BK;
    const double slabs128 = slabs * (!hangs_over128 ? 1 : both_kc ? 1.35 : 1.2) * (most128 >= 5 ? 1.1 : 1);
    const double t256 = 3 + most256 * (slabs * (tiles256 * 4 <= cus * 3ll ? 1.32 : 1.55) + (hangs_over ? 16 : 7));
    const double t128 = 3 + (most128 == 1 ? slabs128 * 0.62 + 2 : most128 * (slabs128 * 0.53 + 1.2));
    return t128 < 0.95 * t256;
}

// Tile of the 16-bit MFMA kernel for an output of batch x m x n with reduction length k.
static void choose_tile16(Plan& p, int batch, int m, int k, int n) {
    p.fam = FAM_MFMA16;
    const long long tiles256 = (long long)((m + 255) / 256) * ((n + 255) / 256) * batch;
    const long long tiles128 = (long long)((m + 127) / 128) * ((n + 127) / 128) * batch;
    // the 256 x 256 tile runs one block per CU, so it needs a k loop long enough to hide its prologue and
    // epilogue; with fewer than four slabs the smaller tile (two blocks per CU) overlaps them instead
    if (m >= 256 && n >= 256 && tiles256 >= cu_tiles() / 2 && k >= 4 * M16_BK && (p.ragged || !small_tiles_win(tiles256, tiles128, m, n, k, !p.a_mc && !p.b_mc))) { p.bm = 256; p.bn = 256; p.name = "mfma16_256x256"; }
    // fewer than 128 tiles of 128 x 128 would leave over half the CUs idle: the 64 x 64 tile quadruples the workgroups
    // (1024^3: 10.9 -> 7.3 us)
    // at most 64 rows: a 64 x 256 tile (the same 64 x 64 patch per wave as the 128 x 128 tile, none of it past the last row)
    // (64 x 128 while k is short: two blocks share a CU and one's loads and stores overlap the other's few slabs)
    else if (m <= 64 && n >= 256 && !path_disabled("wide64") && (long long)((n + 255) / 256) * batch >= cu_tiles() / 2) {
        p.bm = 64; p.bn = k <= 1024 ? 128 : 256; p.name = k <= 1024 ? "mfma16_64x128" : "mfma16_64x256";
    }
    else if ((m > 64 || n > 64) && tiles128 >= cu_tiles() / 2) { p.bm = 128; p.bn = 128; p.name = "mfma16_128x128"; }
    else { p.bm = 64; p.bn = 64; p.name = "mfma16_64x64"; }
    p.edge = (m % p.bm) || (n % p.bn) || (k % M16_BK);
}

// Tile of the fp32 / fp64 MFMA kernel.
static void choose_tile_wide(Plan& p, int batch, int m, int k, int n, int dtype) {
    p.fam = FAM_MFMAW;
    const long long tiles128 = (long long)((m + 127) / 128) * ((n + 127) / 128) * batch;
    // a 128 x 128 tile over a 64-wide output would compute and fetch half of it for nothing.  Ragged rows take it only in fp32 on the
    // bf16 matrix cores, and only for k that is worth that kernel's prologue: the 128 x 128 tile of the fp32 / fp64 MFMA kernel holds
    // a CU by itself and cannot cover its unaligned loads (us, 128 x 128 and 64 x 64: fp64 501 x 1025 x 4001 376 / 164, 1411 x 129 x 1500 60 / 31,
    // 4999 x 513 x 4999 921 / 689; fp32 in bf16 501 x 33 x 4001 16.4 / 9.4, 3001 x 49 x 2999 31.7 / 28.3, 4999 x 49 x 4999 62.3 / 63.8, 2001 x 97 x 2003 20.5 / 22.4).
    const bool tile128 = !p.ragged || (dtype == RP_DTYPE_FLOAT32 && k > 48 && !path_disabled("split32"));
    if (tile128 && m > 64 && n > 64 && tiles128 >= cu_tiles() / 2) { p.bm = 128; p.bn = 128; p.name = (dtype == RP_DTYPE_FLOAT32) ? "mfma32_128x128" : "mfma64_128x128"; }
    else { p.bm = 64; p.bn = 64; p.name = (dtype == RP_DTYPE_FLOAT32) ? "mfma32_64x64" : "mfma64_64x64"; }
    p.edge = (m % p.bm) || (n % p.bn) || (k % (dtype == RP_DTYPE_FLOAT32 ? 32 : 16));
}

// With k = 1 nothing is ever read along the k axis and its strides may hold anything: a contiguous [m, 1] has (1, 1), an
// expanded one 0.  The 16-bit kernels mask k rows past the end of a free-axis-contiguous operand by the end of its
// buffer descriptor alone, which holds only if such rows start behind the operand: give the axis the stride of dense rows.
static void plain_k_strides(int m, int k, int n, long long a_rs, long long& a_cs, long long& b_rs, long long b_cs) {
    if (k != 1) return;
    if (a_rs == 1) a_cs = m;
    if (b_cs == 1) b_rs = n;
}

// Decide the kernel family and tile from shapes and strides alone (pointer
// alignment is checked by the caller, which may still fall back to generic).
static Plan make_plan(int batch, int m, int k, int n, long long a_rs, long long a_cs, long long b_rs, long long b_cs,
                      long long c_rs, long long c_cs, long long a_bs, long long b_bs, int dtype, bool allow_direct = true, bool bases_aligned = true) {
    Plan p{FAM_GENERIC, 64, 64, false, false, true, "generic"};
    if (path_disabled("mfma")) return p;
    plain_k_strides(m, k, n, a_rs, a_cs, b_rs, b_cs);
    const int vec = 16 / (int)dtype_size(dtype);                // elements per 16-byte vector
    // operand layouts: KC = unit stride along k, MC = unit stride along the free axis.
    // Extent-1 axes make the other stride irrelevant, but vector loads still need alignment of the non-unit stride.
    bool a_kc = (a_cs == 1) && (a_rs % vec == 0) && (k % vec == 0);
    bool a_mc = (a_rs == 1) && (a_cs % vec == 0) && (m % vec == 0);
    bool b_mc = (b_cs == 1) && (b_rs % vec == 0) && (n % vec == 0);
    bool b_kc = (b_rs == 1) && (b_cs % vec == 0) && (k % vec == 0);
    bool batch_ok = bases_aligned && ((batch == 1) || ((a_bs % vec == 0) && (b_bs % vec == 0)));

    // the MFMA kernels address a tile with 32-bit byte offsets from a 64-bit tile pointer
    const long long max_stride = 1ll << 22;
    const bool strides_ok = a_rs < max_stride && a_cs < max_stride && b_rs < max_stride && b_cs < max_stride;
    const bool is16 = dtype == RP_DTYPE_FLOAT16 || dtype == RP_DTYPE_BFLOAT16;
    // k rows that overlap (an operand expanded along k): rows past the end of k lie inside the buffer (see plain_k_strides),
    // which is harmless only if no slab hangs over
    const bool overlapping_k = is16 && k % M16_BK != 0 && ((a_mc && !a_kc && a_cs < m) || (b_mc && b_rs < n));
    const bool mfma_ok = (a_kc || a_mc) && (b_kc || b_mc) && batch_ok && strides_ok && !overlapping_k;

    // 16-bit, few rows, deep k: split k over many blocks so that B streams at HBM speed (output columns in whole 8s).
    // Up to 32 rows always; up to SKINNY_MAX_ROWS when the 128 x 128 tiles of the output would occupy under half the
    // CUs and k is deep enough to be worth a second launch for the partial sums (64 x 1024 x 4096: 6.6 us on 64 x 64 tiles
    // in one launch against 9.4 us split; 64 x 4096 x 1024: 16.4 against 9.1).  A short batch of such products is
    // split the same way while its tiles together stay under half the CUs.
    const long long tiles128_16 = (long long)((m + 127) / 128) * ((n + 127) / 128) * batch;
    const bool few_rows = batch == 1 ? (m <= 32 || (m <= SKINNY_MAX_ROWS && tiles128_16 < cu_tiles() / 2 && k >= 2048))
                                     : (m <= SKINNY_MAX_ROWS && tiles128_16 < cu_tiles() / 2 && k >= 2048);
    if (is16 && mfma_ok && few_rows && n % 8 == 0 && n >= 256 && k >= 1024 &&
        (long long)k * n >= (1ll << 22)) {
        p.fam = FAM_MFMA16_SKINNY; p.bm = 32; p.bn = 128; p.edge = true; p.a_mc = !a_kc; p.b_mc = b_mc;
        // row-major A and B with at most 32 rows: the streaming kernel, for the shapes it is the right one for
        p.name = (batch == 1 && !p.a_mc && p.b_mc && stream128_shape(batch, m, k, n)) ? "mfma16_stream_32x128" : "mfma16_skinny_32x128";
        return p;
    }
    // VALU skinny: few rows, row-major B, enough columns and depth to be worth streaming
    const int valu_rows = (dtype == RP_DTYPE_FLOAT32) ? SK_MAX_M : 4;
    if (batch_ok && batch == 1 && dtype != RP_DTYPE_FLOAT64 && m <= valu_rows && b_mc && n >= 64 * vec && (long long)k * n >= (1ll << 20) &&
        (n + 64 * vec - 1) / (64 * vec) <= SK_MAX_GROUPS) {
        p.fam = FAM_SKINNY; p.name = "skinny"; p.b_mc = true;
        return p;
    }
    // fp32, an output of fewer than 64 tiles of 64 x 64 and a k that one workgroup walks in a few microseconds: one launch
    // of 16 x 16 tiles with k split over the four waves of a workgroup, any strides (no split over workgroups, no second launch)
    if (dtype == RP_DTYPE_FLOAT32 && k <= 2048 && (long long)((m + 63) / 64) * ((n + 63) / 64) * batch < 64 && !path_disabled("tiny")) {
        p.fam = FAM_TINY; p.bm = 16; p.bn = 16; p.name = "tiny32_16x16";
        return p;
    }
    // fp32 with k <= 64, any operand layout with a unit stride and at least one 128 x 128 tile per CU: one resident workgroup per
    // CU whose fetching waves fill LDS directly and whose multiplying waves store the previous tile between the MFMAs
    if (dtype == RP_DTYPE_FLOAT32 && allow_direct && !path_disabled("pipe32") && k <= 64 && k % 4 == 0 && ((a_cs == 1 && a_rs % 4 == 0) || (a_rs == 1 && a_cs % 4 == 0)) &&
        ((b_rs == 1 && b_cs % 4 == 0) || (b_cs == 1 && b_rs % 4 == 0)) &&
        batch_ok && m > 64 && n > 64 && (long long)((m + 127) / 128) * ((n + 127) / 128) * batch >= cu_tiles()) {
        p.fam = FAM_PIPE32; p.bm = 128; p.bn = 128; p.a_mc = !(a_cs == 1 && a_rs % 4 == 0); p.b_mc = !(b_rs == 1 && b_cs % 4 == 0); p.edge = (m % 128) || (n % 128); p.name = "pipe32_128x128";
        return p;
    }
    // fp32 with 32 < k <= 64, both operands with unit stride along their free index and an output of at least 128 tiles of
    // 128 x 128: no k loop to pipeline, so every wave multiplies a 64 x 64 patch straight out of registers (no LDS, no
    // barrier).  (With unit stride along k a lane's loads touch 64 cache lines per instruction and the vector cache's
    // tag lookups take longer than the MFMAs: those layouts keep LDS.)
    if (dtype == RP_DTYPE_FLOAT32 && allow_direct && !path_disabled("direct32") && k > 32 && k <= 64 && a_rs == 1 && a_cs != 1 && b_cs == 1 && b_rs != 1 &&
        (a_cs != 1 || (k % 4 == 0 && a_rs % 4 == 0 && a_bs % 4 == 0)) && (b_rs != 1 || (k % 4 == 0 && b_cs % 4 == 0 && b_bs % 4 == 0)) &&
        m >= 64 && n >= 64 && (long long)((m + 127) / 128) * ((n + 127) / 128) * batch >= cu_tiles() / 2) {
        p.fam = FAM_DIRECT32; p.bm = 128; p.bn = 128; p.a_mc = a_cs != 1; p.b_mc = b_rs != 1; p.name = "direct32_128x128";
        return p;
    }
    // the same for bf16 / fp16 (C row-major): there the stores and the narrowing are what takes time
    if (is16 && allow_direct && !path_disabled("pipe16") && k <= 64 && k % 8 == 0 && (a_kc || a_mc) && (b_kc || b_mc) && batch_ok &&
        c_cs == 1 && c_rs % 8 == 0 && n % 8 == 0 && m > 64 && n > 64 && (long long)((m + 127) / 128) * ((n + 127) / 128) * batch >= cu_tiles()) {
        p.fam = FAM_PIPE16; p.bm = 128; p.bn = 128; p.a_mc = !a_kc; p.b_mc = !b_kc; p.edge = (m % 128) || (n % 128); p.name = "pipe16_128x128";
        return p;
    }
    // bf16 / fp16, at most 64 output columns, at least one 128-row tile per CU (O = P.V per head, a tall matrix times a narrow
    // one): bound by reading A; the resident kernel whose fetching waves keep three k slabs in flight into LDS
    if (is16 && allow_direct && !path_disabled("pipe16k") && n <= 64 && n % 8 == 0 && k % 8 == 0 && k >= 64 && (a_kc || a_mc) && (b_kc || b_mc) && batch_ok &&
        c_cs == 1 && c_rs % 8 == 0 && m > 64 && (long long)((m + 127) / 128) * batch >= cu_tiles()) {
        p.fam = FAM_PIPE16K; p.bm = 128; p.bn = 64; p.a_mc = !a_kc; p.b_mc = !b_kc; p.edge = (m % 128) || n != 64; p.name = "pipe16k_128x64";
        return p;
    }
    // the same in fp32 (any C strides): bound by the MFMAs, which the resident kernel keeps fed without a wait per slab
    if (dtype == RP_DTYPE_FLOAT32 && allow_direct && !path_disabled("pipe32k") && n <= 64 && k % 4 == 0 && k >= 32 && (a_kc || (a_rs == 1 && a_cs % 4 == 0)) &&
        (b_kc || (b_cs == 1 && b_rs % 4 == 0)) && batch_ok && m > 64 && (long long)((m + 127) / 128) * batch >= cu_tiles()) {
        p.fam = FAM_PIPE32K; p.bm = 128; p.bn = 64; p.a_mc = !a_kc; p.b_mc = !b_kc; p.edge = (m % 128) || n != 64; p.name = "pipe32k_128x64";
        return p;
    }
    if (!mfma_ok && strides_ok && !path_disabled("ragged")) {
        // Rows that are no whole number of 16-byte vectors or start anywhere: the MFMA kernels' ragged variants.  They need a
        // vector's worth of elements along the unit-stride axis and rows that do not overlap.  Outputs of less than two
        // 64 x 64 tiles between small operands stay on the generic kernel, which splits their k over the chip (a handful of
        // MFMA workgroups would walk it slab by slab).
        const bool ak = a_cs == 1 && k >= vec && (a_rs >= k || m == 1), am = a_rs == 1 && m >= vec && a_cs >= m;
        const bool bn = b_cs == 1 && n >= vec && b_rs >= n, bk = b_rs == 1 && k >= vec && (b_cs >= k || n == 1);
        const bool worth = (long long)m * n * batch >= 8192 || (long long)k * n >= (1 << 18) || (long long)m * k >= (1 << 18);
        // The same for 16-bit outputs of up to four tiles whose k is deeper than ten slabs a tile (bf16, us, MFMA and generic: 156 x 4097 x 59
        // 26.7 / 20.5, 33 x 8001 x 129 47.4 / 29.8, 65 x 2049 x 127 16.0 / 17.5; nine tiles, 130 x 8001 x 130 47.7 / 78)
        const int tiles64 = ((m + 63) / 64) * ((n + 63) / 64);
        const bool too_deep = is16 && batch == 1 && tiles64 <= 4 && k > 10 * M16_BK * tiles64;
        if ((ak || am) && (bn || bk) && worth && !too_deep) {
            p.ragged = true;
            p.a_mc = !ak;
            p.b_mc = bn;
            if (!is16) {
                choose_tile_wide(p, batch, m, k, n, dtype);
            } else if (few_rows && n >= 256 && k >= 1024 && (long long)k * n >= (1ll << 22) &&
                       skinny16_workspace(batch, m, k, n) <= (size_t)RP_HIP_NOALLOC_WORKSPACE_BYTES) {
                // (partial sums beyond the fixed array of the entry point that allocates nothing: unsplit tiles, which need none.  That
                // entry point takes ragged products of any size, with the bits of the one that allocates: one rule for both.  At that size
                // the split pays no more: bf16 96 x 2049 x 16201 47.8 us split and 39.4 unsplit, 32 x 8193 x 140001 523 and 495)
                p.fam = FAM_MFMA16_SKINNY; p.bm = 32; p.bn = 128; p.edge = true; p.name = "mfma16_skinny_32x128";
            } else {
                choose_tile16(p, batch, m, k, n);
            }
            return p;
        }
    }
    if (!mfma_ok) return p;
    p.a_mc = !a_kc;             // when both qualify (extent-1 corner cases) keep the row-major reading
    p.b_mc = b_mc;

    if (is16) {
        choose_tile16(p, batch, m, k, n);
    } else {
        choose_tile_wide(p, batch, m, k, n, dtype);
    }
    return p;
}

// First byte and one past the last of an operand of a product
struct Span { const char* lo; const char* hi; };
static Span span_of(const void* p, int rows, int cols, long long rs, long long cs, int esz) {
    return {(const char*)p, (const char*)p + ((rows - 1) * rs + (cols - 1) * cs + 1) * esz};
}
static bool overlap(const Span& a, const Span& b) { return a.lo < b.hi && b.lo < a.hi; }

// Few 16-bit output tiles, deep k, A k-contiguous: the waves of a workgroup split k (rp_gemm_mfma16_wavek.hip).  B k-contiguous too: up to
// one 32 x 32 tile per CU, against the k split in two launches two while a tile's rows are no longer than 4096 (us, before and here: 256 of them
// 64 x 1024 x 4096 7.0 / 5.0, 128 x 8192 x 2048 18.8 / 14.7; 384 and 512 96 x 2048 x 4096 16.1 / 8.9, 64 x 4096 x 8192 19.6 / 15.1, 64 x 8192 x 8192
// 40.7 / 42.5; against 64 x 64 tiles 256 x 2048 x 2048 10.6 / 9.0, 1024 x 4096 x 512 16.9 / 22).
// B row-major: up to one 16 x 64 tile per CU, against the k split while k is up to 2048 (64 x 2048 x 2048 9.7 / 6.9, 64 x 4096 x 1024 10.0 / 11.7,
// 96 x 4096 x 4096 with 384 tiles 16.4 / 19.2).
// From ten slabs on: the eight of 128 x 512 x 512 take 5.3 and 4.8.  A small layer's dX in one launch with dW follows the same rule.
// Ragged rows: with any k, and in place of the generic kernel and its k split too, whose loads are of single elements (511 x 4001 x 513 31.8 / 18.1,
// 53 x 1434 x 14 13.1 / 7.8; 220 drawn ones 0.56 of the time), unless a row-major B of very few tiles has a long k (3 x 3261 x 63 13.0 / 15.1); and of
// the few rows that the row-streaming kernel took those with k up to 1024 (3 x 281 x 5216 20.5 / 4.7).
// (The k split with a launch of its own for the sums read all of its operands before it wrote C: outputs over an operand stay there.)
static bool wavek16_takes(const GemmArgs& g, const Plan& p, int dtype, bool& ragged) {
    if ((dtype != RP_DTYPE_BFLOAT16 && dtype != RP_DTYPE_FLOAT16) || g.batch != 1 || path_disabled("wavek")) return false;
    const bool split = p.fam == FAM_MFMA16_SKINNY, generic = p.fam == FAM_GENERIC || (p.fam == FAM_SKINNY && g.k <= 1024);      // (whose operands no MFMA kernel has looked at)
    if (!split && !generic && !(p.fam == FAM_MFMA16 && p.bm == 64 && p.bn == 64)) return false;
    ragged = p.ragged || generic;
    const bool b_mc = generic ? !(g.b_rs == 1 && g.k >= 8 && (g.b_cs >= g.k || g.n == 1)) : p.b_mc;
    if (generic) {
        if (path_disabled("mfma") || path_disabled("ragged") || !(g.a_cs == 1 && g.k >= 8 && (g.a_rs >= g.k || g.m == 1))) return false;
        if (b_mc && !(g.b_cs == 1 && g.n >= 8 && g.b_rs >= g.n)) return false;
        if (g.a_rs >= (1ll << 22) || g.b_rs >= (1ll << 22) || g.b_cs >= (1ll << 22)) return false;
    } else if (p.a_mc) {
        return false;
    }
    if ((!ragged && g.k < 10 * M16_BK) || g.k >= (1 << 24)) return false;
    if (b_mc) {
        const long long tiles = (long long)((g.m + 15) / 16) * ((g.n + 63) / 64);
        if (generic && g.k > 2048 && g.k > 512 * tiles) return false;
        if (tiles > cu_tiles() || g.k * g.b_rs >= (1ll << 30)) return false;
        if (split && (g.k > 2048 || (!ragged && stream128_shape(g.batch, g.m, g.k, g.n)))) return false;
    } else {
        const long long tiles = (long long)((g.m + 31) / 32) * ((g.n + 31) / 32);
        if (!(tiles <= cu_tiles() || (split && g.k <= 4096 && tiles <= 2 * cu_tiles()))) return false;
    }
    if (g.seg_k || g.seg_n || g.bias_by_row || g.c_fold_from) return false;
    const Span c = span_of(g.C, g.m, g.n, g.c_rs, g.c_cs, 2);
    return !overlap(c, span_of(g.A, g.m, g.k, g.a_rs, g.a_cs, 2)) && !overlap(c, span_of(g.B, g.k, g.n, g.b_rs, g.b_cs, 2)) &&
           !(g.bias && overlap(c, span_of(g.bias, 1, g.n, 0, 1, 2)));
}

// Of the generic kernel's fp64 products (expanded or overlapping rows, very small outputs): not those of few slabs of 16 values of k and many tiles.  A tile of
// 32 x 32 costs the chip 5.8 ns here whatever k is, one of 16 x 16 half of that; a 64 x 64 one costs 6 (nearly empty) to 12 ns there with one slab, 15 with two,
// 21 with three, 27 with four.  us there and here: 3000 x 64 x 5 x 64 36.7 / 71.9, 3000 x 33 x 5 x 65 46.3 / 103.8, 400 x 64 x 5 x 64 10.7 / 13.6, 3001 x 3 x 2001 23.7 / 37.4, 3000 x 20 x 5 x 20
// 24.7 / 34.2, but 8000 x 1 x 3 x 1 49.8 / 41.4, 100 x 64 x 5 x 64 6.9 / 4.9; 3000 x 64 x 17 x 64 45.3 / 75.5, 3000 x 20 x 17 x 20 41.6 / 35.4, 400 x 33 x 17 x 65 18.5 / 17.9; 3000 x 64 x 48 x 64
// 62.9 / 78.0, 3001 x 40 x 2001 35.7 / 40.3, 3000 x 33 x 33 x 65 113 / 112, 400 x 64 x 48 x 64 16.8 / 14.2; 3000 x 64 x 64 x 64 81 / 82; 3000 x 64 x 130 x 64 171 / 121, 8000 x 1 x 1001 x 1 2999 / 256.
static bool generic64_wins(const GemmArgs& g, WkwTile tile) {
    const long long cus = cu_tiles(), tiles64 = (long long)((g.m + 63) / 64) * ((g.n + 63) / 64) * g.batch;
    const long long work = tile == WKW_32X32 ? (long long)((g.m + 31) / 32) * ((g.n + 31) / 32) * g.batch : (long long)((g.m + 15) / 16) * ((g.n + 15) / 16) * g.batch / 2;       // in tiles of 32 x 32
    if (g.k <= 16) return work >= 4 * cus && work * 2 >= tiles64 * 3;
    if (g.k <= 32) return work >= 10 * cus && work * 2 >= tiles64 * 5;
    return g.k <= 48 && work >= 16 * cus && work * 2 >= tiles64 * 7;
}

// fp32 and fp64 products that the waves of a workgroup share (rp_gemm_wavekw.hip, which has figures): those of 64 x 64 tiles, fp64 ones of the generic
// kernel, and fp32 ones that 16 x 16 tiles of four waves or the row-streaming kernel took.  Stays where it was: fp32 with k up to 512 on 16 x 16 tiles (60 x 443 x 65 3.55 / 3.67 us; 256 x 784 x 256
// 6.95 / 5.0-6.0); a k too short for the number of tiles (fp32 2384 x 32 x 368
// 5.2 / 6.5, 944 x 144 x 1648 14.0 / 16.2; fp64 832 x 48 x 2128 14.6 / 22.7); fp32 outputs of a few tiles whose long k the split deals to more CUs
// (16 x 5744 x 48 11.5 / 14.4) and sums in shorter chains; batches of more than one 64 x 64 tile a CU that fill those as well as 32 x 32 ones (fp32
// 128 x 512 x 128 100 of them 26.8 / 33.2, 60 21.2 / 14.9; 20 x 600 x 20 1000 of them 50.8 / 26.1; fp64 40 x 100 x 40 3000 of them 84 / 124) or, in fp32, of a k up
// to 64 (128 x 64 x 128, 50 of them 6.2 / 7.6).  (The k split read all of its operands before it wrote C: outputs over an operand stay there.)
// Of the row-streaming kernel's products (up to 8 rows), which sums chains of 32 values: those with 168 <= k <= 1024, on 16 x 32 tiles alone, whose waves'
// chains are no longer (relative error of 8 x k x 16384, there and here: k = 128 8.7e-8 / 8.9e-8, 168 9.5e-8 / 9.2e-8, 256 1.13e-7 / 9.6e-8, 640 1.15e-7 / 1.13e-7, 1024 1.19e-7 / 1.13e-7
// with 16 waves, 1.25e-7 with 8; the larger tiles' chains are of k / 16 and k / 8: 1024 1.6e-7 and 2.1e-7), us there and here: 8 x 256 x 8192 22.0 / 5.0, 1 x 1024 x 8192 11.4 / 5.8, 8 x 1024 x 16384 24.2 / 14.2.
// Up to four rows of very many columns stay where k is short or takes 16 waves: 1 x 200 x 49152 7.9 / 10.6, 4 x 200 x 65000 13.1 / 15.0, 1 x 1000 x 32768 23.6 / 25.2 (1 x 200 x 24576 7.1 / 6.0,
// 1 x 384 x 49152 16.7 / 14.7, 1 x 1000 x 16384 15.5 / 13.9, 5 x 176 x 65000 16.6 / 14.0).
static WkwTile wavekw_takes(const GemmArgs& g, const Plan& p, int dtype) {
    const bool f32 = dtype == RP_DTYPE_FLOAT32;
    if (!(f32 || dtype == RP_DTYPE_FLOAT64) || g.seg_k || g.seg_n || g.bias_by_row || g.c_fold_from || path_disabled("wavekw")) return WKW_NONE;
    const long long tiles64 = (long long)((g.m + 63) / 64) * ((g.n + 63) / 64) * g.batch, tiles16 = (long long)((g.m + 15) / 16) * ((g.n + 15) / 16) * g.batch;
    if (p.fam == FAM_MFMAW && p.bm == 64) {
        const long long tiles32 = (long long)((g.m + 31) / 32) * ((g.n + 31) / 32) * g.batch;
        if (g.batch > 1 && ((tiles64 > cu_tiles() && tiles32 * 2 >= tiles64 * 7) || (f32 && g.k <= 64 && tiles64 > cu_tiles() / 2))) return WKW_NONE;
        if (f32 ? g.k <= 32 || (tiles64 > cu_tiles() && g.k < 256) : g.k <= 48 && tiles64 > cu_tiles() / 2) return WKW_NONE;
        const bool splits = f32 && (g.n % 4 == 0 || p.ragged), both_kc = g.a_cs == 1 && g.b_rs == 1 && g.b_cs != 1;
        if (splits && g.k > 2048 && (tiles64 < cu_tiles() / 32 || (!both_kc && tiles16 < cu_tiles() / 4))) return WKW_NONE;
    } else if (p.fam == FAM_TINY) {
        if (g.k <= 512) return WKW_NONE;
    } else if (p.fam == FAM_SKINNY) {
        if (!f32 || g.k < 168 || g.k > 1024) return WKW_NONE;
        if (g.m <= 4 && (g.k > 640 ? g.n > 16384 : g.n > 24576 && g.k < 384)) return WKW_NONE;
    } else if (!(p.fam == FAM_GENERIC && !f32 && !path_disabled("mfma"))) {
        return WKW_NONE;
    }
    const WkwTile tile = wavekw_tile(g, dtype);
    if (tile == WKW_NONE || (p.fam == FAM_GENERIC && generic64_wins(g, tile))) return WKW_NONE;
    const int esz = (int)dtype_size(dtype);
    auto span = [&](const void* base, int rows, int cols, long long bs, long long rs, long long cs) {
        Span s = span_of(base, rows, cols, rs, cs, esz);
        (bs < 0 ? s.lo : s.hi) += (g.batch - 1) * bs * esz;
        return s;
    };
    const Span c = span(g.C, g.m, g.n, g.c_bs, g.c_rs, g.c_cs);
    const bool apart = !overlap(c, span(g.A, g.m, g.k, g.a_bs, g.a_rs, g.a_cs)) && !overlap(c, span(g.B, g.k, g.n, g.b_bs, g.b_rs, g.b_cs)) &&
                       !(g.bias && overlap(c, span_of(g.bias, 1, g.n, 0, 1, esz)));
    return !apart ? WKW_NONE : p.fam == FAM_SKINNY ? WKW_FEW_ROWS : tile;
}

static thread_local const char *g_last_kernel = "none", *g_last_launch = "none";      // what rp_hip_last_gemm_kernel and rp_hip_last_gemm_launch report
void report_kernel(const char* name, const char* launched) { g_last_kernel = name; g_last_launch = launched ? launched : name; }
void report_launch(const char* launched) { g_last_launch = launched; }

static int run_gemm(GemmArgs g, int dtype) {
    plain_k_strides(g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs);
    Plan p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype);
    if (p.fam == FAM_PIPE32) {
        if (pipe32_takes(g)) { report_kernel(p.name); return launch_pipe32(g); }
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false);     // options, base pointers or spans it does not take
    }
    if (p.fam == FAM_PIPE16) {
        if (pipe16_takes(g)) { report_kernel(p.name); return launch_pipe16(g, dtype); }
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false);
    }
    if (p.fam == FAM_PIPE16K) {
        if (pipe16k_takes(g)) { report_kernel(p.name); return launch_pipe16k(g, dtype); }
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false);
    }
    if (p.fam == FAM_PIPE32K) {
        if (pipe32k_takes(g)) { report_kernel(p.name); return launch_pipe32k(g); }
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false);
    }
    if (p.fam == FAM_DIRECT32) {
        if (direct32_takes(g)) { report_kernel(p.name); return launch_direct32(g); }
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false);     // base pointers or spans it cannot address
    }
    if (p.fam != FAM_GENERIC && p.fam != FAM_TINY && !p.ragged && !(aligned16(g.A) && aligned16(g.B)))
        p = make_plan(g.batch, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, g.a_bs, g.b_bs, dtype, false, false);
    bool wavek_ragged = false;
    if (wavek16_takes(g, p, dtype, wavek_ragged)) {
        report_kernel(wavek_ragged ? p.name : "mfma16_wavek", wavek_ragged ? "mfma16_wavek_ragged" : "mfma16_wavek");      // (ragged rows: by the name of the kernel that it stands in for)
        return launch_mfma16_wavek(g, wavek_ragged, dtype);
    }
    const WkwTile shared_k = wavekw_takes(g, p, dtype);
    if (shared_k != WKW_NONE) {
        report_kernel(p.fam == FAM_MFMAW ? p.name : dtype == RP_DTYPE_FLOAT32 ? "mfma32_wavek" : "mfma64_wavek", wavekw_name(shared_k, dtype));      // (among the 64 x 64 tiles by their name)
        return launch_wavekw(g, shared_k, dtype);
    }
    report_kernel(p.name);
    switch (p.fam) {
        case FAM_MFMA16:
        case FAM_MFMA16_SKINNY: return launch_mfma16(g, p, dtype);
        case FAM_MFMAW:  return launch_mfmaw(g, p, dtype);
        case FAM_SKINNY: return launch_skinny(g, dtype);
        case FAM_TINY:   return launch_tiny(g, dtype);
        default:         return launch_generic(g, dtype);
    }
}

// fp32 products with segments that the waves of a workgroup share; WKW_NONE: the 64 x 64 and 128 x 128 tiles of four waves that share the output.
// us of the products of layers [batch, C_in, H, W, C_out, k], before and here; a convolution is one product per image, so what counts is the tiles of all of them.
// Segments along k (forward and input gradient: m = C_out, n = positions, k = taps C_in): 16 x 32 tiles, 16 x 16 where those are fewer than the CUs,
// [1, 128, 28, 28, 64, 5] 105.7 / 16.4, [2, 256, 15, 15, 64, 3] 88.9 / 15.2, [8, 192, 14, 14, 128, 5] 185 / 64, [40, 128, 28, 28, 64, 3] 95 / 83.  They read A and B once per
// 16 x 32 values, so with enough 64 x 64 tiles to fill the chip they are left behind, sooner where k is short: 64 channels of 3 x 3, 64 -> 64 at 28 x 28,
// 26 images (364 tiles) 42.6 / 41.5, 33 45.0 / 50.4, 54 58.6 / 74.9; from 1024 on [60, 128, 28, 28, 64, 3] (840 tiles) 109 / 112.
// From 192 rows on the 64 x 64 tile with k shared takes over there: [12, 64, 55, 55, 192, 3] 186 / 134 (16 x 32: 156), [9, 192, 28, 28, 256, 3] 111 / 87 (96).
// Segments along n (weight gradients: m = C_out, n = taps C_in, k = positions): 32 x 32 up to one 64 x 64 tile a CU ([1, 128, 28, 28, 64, 5] 40.1 / 19.4, [5, 64, 56, 15, 64, 3]
// 48.7 / 22.7, [22, 64, 48, 48, 64, 3] 96 / 85).  With nearly that many and a long k those of more than 64 rows are 64 x 64 tiles, [1, 256, 56, 56, 128, 5] 123 / 86 (32 x 32: 116), and
// those of 64 stay what they were, [10, 64, 56, 56, 64, 5] 121 / 139.  Up to four a CU where C_out is more than 64
// and the positions many ([18, 128, 28, 28, 192, 3] 152 / 107, but [31, 256, 26, 26, 64, 3] 109 / 143, [13, 192, 7, 7, 256, 3] 45.5 / 56.5).
// samples: how many the whole call has, of which g.batch go out now.  The tile follows all of them, so that the bits do not depend on how the batch is cut.
static WkwTile segmented_wavek_tile(const GemmArgs& g, long long samples) {
    if (path_disabled("wavekw") || g.a_cs != 1 || g.n < 64 || g.accumulate || (long long)((g.m + 15) / 16) * ((g.n + 15) / 16) * samples >= (1ll << 23) - 8 || g.b_extent * 4 >= (1ll << 31) || (63 * g.a_rs + g.k) * 4 >= (1ll << 31)) return WKW_NONE;
    const long long cus = cu_tiles(), tiles64 = (long long)((g.m + 63) / 64) * ((g.n + 63) / 64) * samples;
    if (g.seg_k > 0) {
        if (g.seg_k % 32) return WKW_NONE;
        if (g.m >= 192) { if (tiles64 * 4 >= cus * 7) return WKW_64X64; }
        else if (g.k < 1024 ? tiles64 * 4 > cus * 5 : tiles64 > cus * 3) return WKW_NONE;
        return (long long)((g.m + 15) / 16) * ((g.n + 31) / 32) * samples >= cus ? WKW_16X32 : WKW_16X16;
    }
    if (tiles64 <= cus) {
        if (g.k < 2048 || tiles64 * 4 < cus * 3) return WKW_32X32;
        return g.m > 64 ? WKW_64X64 : tiles64 * 8 > cus * 7 ? WKW_NONE : WKW_32X32;
    }
    return g.m > 64 && g.k >= 640 && tiles64 <= 4 * cus ? WKW_32X32 : WKW_NONE;
}

// C_z = A_z . B_z with B's k axis or its n axis given as segments (GemmArgs::seg_*): the MFMA kernels read every
// segment in place, at any alignment of whole elements.  For callers inside the library (the convolution), which
// guarantee: A with unit stride along k or m, B with unit stride along n and k a whole number of segments of whole
// slabs, or B with unit stride along k and n a whole number of segments.  samples: matrices of the whole call, of which g is a part.
int launch_gemm_segmented_b(const GemmArgs& g, int samples, int dtype) {
    const bool is16 = dtype == RP_DTYPE_FLOAT16 || dtype == RP_DTYPE_BFLOAT16;
    const int vec = 16 / (int)dtype_size(dtype);
    const int bk = is16 ? M16_BK : (dtype == RP_DTYPE_FLOAT32 ? 32 : 16);           // k slab of the kernel that will run
    const bool a_kc = g.a_cs == 1, a_mc = g.a_rs == 1 && g.m % vec == 0;
    const long long max_stride = 1ll << 22;
    bool ok = dtype_size(dtype) && (a_kc || a_mc) && g.seg_w > 0 && g.a_rs < max_stride && g.a_cs < max_stride && g.b_rs < max_stride && g.b_cs < max_stride &&
              g.batch <= 65535 && g.b_extent > 0 && g.b_extent < (1ll << 30);
    if (!is16) ok = ok && (a_kc ? g.a_rs % vec == 0 && g.k % vec == 0 : g.a_cs % vec == 0) && g.a_bs % vec == 0;     // the fp32 / fp64 kernel loads A with plain vector loads
    if (g.seg_k > 0) ok = ok && g.seg_n == 0 && g.b_cs == 1 && g.n % vec == 0 && g.seg_k % bk == 0 && g.k % g.seg_k == 0;    // segments along k
    else ok = ok && g.seg_n > 0 && g.b_rs == 1 && g.k % vec == 0 && g.n % g.seg_n == 0;                                     // segments along n
    // the folded store and the per-row bias exist on the vector path of the epilogue only
    if (g.c_fold_from > 0)
        ok = ok && g.c_cs == 1 && g.c_rs % vec == 0 && g.c_bs % vec == 0 && aligned16(g.C) && g.c_fold_from % vec == 0 && g.c_fold_to % vec == 0 &&
             g.c_fold_to <= g.c_fold_from && g.n % g.c_fold_from == 0;
    if (!ok) {
        set_error("segmented GEMM: operands outside what the MFMA kernels read in place");
        return -1;
    }
    if (is16) {
        Plan p{FAM_MFMA16, 64, 64, !a_kc, g.seg_k > 0, true, "mfma16"};
        choose_tile16(p, g.batch, g.m, g.k, g.n);
        return launch_mfma16(g, p, dtype);
    }
    if (dtype == RP_DTYPE_FLOAT32) {
        const WkwTile tile = segmented_wavek_tile(g, samples);
        if (tile != WKW_NONE) { report_launch(wavekw_name(tile, dtype)); return launch_wavekw_segmented(g, tile); }
    }
    Plan p{FAM_MFMAW, 64, 64, !a_kc, g.seg_k > 0, true, "mfmaw"};
    const long long tiles128 = (long long)((g.m + 127) / 128) * ((g.n + 127) / 128) * g.batch;
    if (g.m > 64 && g.n > 64 && tiles128 >= cu_tiles() / 2) { p.bm = 128; p.bn = 128; }
    p.edge = (g.m % p.bm) || (g.n % p.bn) || (g.k % bk);
    return launch_mfmaw(g, p, dtype);
}

// ============================================================================
// The entry point that allocates nothing (rp_hip_gemm_strided_batched_noalloc).
// Its split-k launchers take their workspace and arrival counters from one fixed
// device array instead of the pool.  Every GPU the library runs on holds its own
// copy of the array at its own address for the life of the process; host code
// never uses the array's name as an address, only the pointer that
// hipGetSymbolAddress returned for the device that was current.
// ============================================================================
constexpr size_t NOALLOC_COUNTER_BYTES = (size_t)SPLITK_MAX_TILES * sizeof(int);      // arrival counters, then the partial sums
constexpr size_t NOALLOC_WORKSPACE_BYTES = (size_t)RP_HIP_NOALLOC_WORKSPACE_BYTES;
static __device__ __align__(256) unsigned char scratch[NOALLOC_COUNTER_BYTES + NOALLOC_WORKSPACE_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};      // per device: where that device's copy of `scratch` lives
static thread_local unsigned char* g_noalloc_base = nullptr;        // non-null while the calling thread is inside the entry point
static thread_local bool g_noalloc_busy = false;                    // its workspace is handed out (one launcher at a time)
static thread_local bool g_noalloc_cleared = false;                 // this call has cleared the arrival counters

// Address of the current device's copy of the array, resolved once per device.
static unsigned char* noalloc_scratch_of_current_device() {
    int dev = 0;
    if (!check_hip(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) { set_error("rp_hip_gemm_strided_batched_noalloc: device ordinal %d is beyond the %d this entry point tracks", dev, NOALLOC_MAX_DEVICES); return nullptr; }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (!check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return nullptr;
        g_scratch_ptr[dev] = (unsigned char*)p;
    }
    return g_scratch_ptr[dev];
}

int gemm_workspace(void** ws, size_t bytes) {
    if (!g_noalloc_base) return rp_hip_malloc(ws, bytes);
    *ws = nullptr;
    if (bytes > NOALLOC_WORKSPACE_BYTES) {
        set_error("rp_hip_gemm_strided_batched_noalloc: this shape needs %zu bytes of split-k workspace, the fixed array holds %zu", bytes, NOALLOC_WORKSPACE_BYTES);
        return -1;
    }
    if (g_noalloc_busy) { set_error("rp_hip_gemm_strided_batched_noalloc: workspace requested twice"); return -1; }
    g_noalloc_busy = true;
    *ws = g_noalloc_base + NOALLOC_COUNTER_BYTES;
    return 0;
}

void gemm_workspace_release(void* ws) {
    if (!ws) return;
    if (g_noalloc_base && ws == g_noalloc_base + NOALLOC_COUNTER_BYTES) { g_noalloc_busy = false; return; }
    rp_hip_free(ws);
}

__global__ void __launch_bounds__(256) clear_counters_kernel(int* counters, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) counters[i] = 0;
}

bool noalloc_active() { return g_noalloc_base != nullptr; }

// The array keeps what the last call left.  The partial sums are fully overwritten before they are read; the arrival
// counters must read zero, and a launch that was cut short could have left some standing: the first launcher of a call
// that wants them has them cleared by a kernel (stream-ordered before the GEMM; not a memset node, so the call can be
// recorded into a graph).  Calls whose kernels use no counters launch nothing extra.
int* noalloc_arrival_counters() {
    if (!g_noalloc_base) return nullptr;
    if (!g_noalloc_cleared) {
        hipLaunchKernelGGL(clear_counters_kernel, dim3((SPLITK_MAX_TILES + 255) / 256), dim3(256), 0, current_stream(), (int*)g_noalloc_base, SPLITK_MAX_TILES);
        if (!check_launch("clear_counters_kernel")) return nullptr;
        g_noalloc_cleared = true;
    }
    return (int*)g_noalloc_base;
}

// Rows up to which the column sums of dY join the other gradients of a 16-bit layer: four chunks of 256, three where a strip of 64 bytes
// hangs over the columns.  A strip's chunks are a chain that uneven strips walk at up to 2.2 us a chunk, and a launch of their own
// costs 3 to 4 us (bf16, us, in the launch and apart: 256 x 256 x 1024 7.0 / 11.4, 1024 x 512 x 512 10.0 / 12.5, 1024 x 16 x 64 8.3 / 11.2,
// 2048 x 512 x 512 21.2 / 19.3; uneven 768 x 16 x 184 10.1 / 10.2, 904 x 16 x 184 12.1 / 11.2, 1024 x 512 x 184 12.9 / 12.0,
// 1280 x 768 x 264 16.4 / 15.1, 2048 x 40 x 16 21.8 / 16.5).
constexpr int LINEAR_DB_ROWS = 1024, LINEAR_DB_ROWS_UNEVEN = 768;
// The same for fp32 and fp64 layers whose waves share k: a chunk of a strip takes 1.5 us there, 2.1 us of an uneven one.  us, in the launch and apart: fp32 1248 x 48 x 1488
// 11.8 / 16.2, 1200 x 128 x 448 11.4 / 15.1, 1536 x 112 x 64 9.2 / 10.1, 1296 x 64 x 320 9.8 / 9.5, 1648 x 176 x 272 12.7 / 11.9; uneven 1150 x 160 x 373 10.7 / 14.8, 1225 x 127 x 77
// 8.8 / 9.9, 1444 x 23 x 847 13.4 / 11.9, 1570 x 22 x 263 12.1 / 10.7; fp64 1280 x 96 x 512 13.9 / 15.7, 1399 x 689 x 151 27.0 / 30.9, 1648 x 272 x 464 32.5 / 28.9.
constexpr int LINEAR_DB_ROWS_WAVEKW = 1536, LINEAR_DB_ROWS_WAVEKW_UNEVEN = 1280;

// The plan that a product alone would follow
static Plan plan_alone(const GemmArgs& g, int dtype) {
    const Plan p = make_plan(1, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, 0, 0, dtype);
    if (p.fam == FAM_GENERIC || p.fam == FAM_TINY || p.ragged || (aligned16(g.A) && aligned16(g.B))) return p;
    return make_plan(1, g.m, g.k, g.n, g.a_rs, g.a_cs, g.b_rs, g.b_cs, g.c_rs, g.c_cs, 0, 0, dtype, false, false);
}

// Neither gradient is written over anything that the other product (or the bias gradient) reads: one launch after the other, dW over W was fine.
// (An absent gradient is at address 0, apart from everything.)
static bool gradients_apart(const GemmArgs& gx, const GemmArgs& gw, int dtype) {
    const int esz = (int)dtype_size(dtype);
    const Span dx = span_of(gx.C, gx.m, gx.n, gx.c_rs, gx.c_cs, esz), dw = span_of(gw.C, gw.m, gw.n, gw.c_rs, gw.c_cs, esz);
    const Span dy = span_of(gx.A, gx.m, gx.k, gx.a_rs, gx.a_cs, esz), w = span_of(gx.B, gx.k, gx.n, gx.b_rs, gx.b_cs, esz), x = span_of(gw.A, gw.m, gw.k, gw.a_rs, gw.a_cs, esz);
    return !(overlap(dx, dw) || overlap(dx, dy) || overlap(dx, x) || overlap(dw, dy) || overlap(dw, w));
}

// Nor does the bias gradient lie over an operand or a gradient of theirs
static bool bias_gradient_apart(const void* db, const GemmArgs& gx, const GemmArgs& gw, int dtype) {
    const int esz = (int)dtype_size(dtype);
    const Span b = span_of(db, 1, gx.k, 0, 1, esz), dx = span_of(gx.C, gx.m, gx.n, gx.c_rs, gx.c_cs, esz), dw = span_of(gw.C, gw.m, gw.n, gw.c_rs, gw.c_cs, esz);
    const Span dy = span_of(gx.A, gx.m, gx.k, gx.a_rs, gx.a_cs, esz), w = span_of(gx.B, gx.k, gx.n, gx.b_rs, gx.b_cs, esz), x = span_of(gw.A, gw.m, gw.k, gw.a_rs, gw.a_cs, esz);
    return !(overlap(b, dy) || overlap(b, w) || overlap(b, x) || overlap(b, dx) || overlap(b, dw));
}

// The tiles on which a product alone would share k among the waves or run as a tiny one; WKW_NONE: neither, or not with both operands k-contiguous
// (kc) or both free-index-contiguous
static WkwTile small_tile_alone(const GemmArgs& g, bool kc, int dtype) {
    const Plan p = plan_alone(g, dtype);
    const WkwTile tile = wavekw_takes(g, p, dtype);
    if (tile != WKW_NONE) return wkw_a_kc(g) == kc && wkw_b_kc(g) == kc ? tile : WKW_NONE;
    return p.fam == FAM_TINY ? WKW_TINY : WKW_NONE;
}

// Whether dX and dW of a 16-bit Linear layer go out as one launch: both on the 64 x 64 tile (an output of under half a CU count
// of 128 x 128 tiles) in the layouts of dense X and W, and neither gradient written over anything that the other product reads
// (one launch after the other, dW over W was fine).  Larger tiles fill a CU by themselves and gain nothing from company.
// dx_wavek: dX by itself would go to the kernel whose waves split k, and does so in the one launch too: the same bits either way.
// ragged: rows of either product are; then both take the ragged variants, which do the same with rows of whole vectors.
static bool linear_backward_pairs(const GemmArgs& gx, const GemmArgs& gw, int dtype, bool& edge, bool& dx_wavek, bool& ragged) {
    if (path_disabled("pair16")) return false;
    const Plan px = plan_alone(gx, dtype), pw = plan_alone(gw, dtype);
    if (pw.fam != FAM_MFMA16 || pw.bm != 64 || pw.bn != 64 || !pw.a_mc || !pw.b_mc) return false;
    bool dx_ragged = false;
    dx_wavek = gx.b_rs == 1 && px.fam != FAM_MFMA16_SKINNY && wavek16_takes(gx, px, dtype, dx_ragged);
    if (!dx_wavek && (px.fam != FAM_MFMA16 || px.bm != 64 || px.bn != 64 || px.a_mc || px.b_mc)) return false;
    ragged = pw.ragged || px.ragged || (dx_wavek && dx_ragged);
    edge = pw.edge || (px.edge && !dx_wavek);
    return gradients_apart(gx, gw, dtype);
}

}  // namespace rp

using namespace rp;

extern "C" {

int rp_hip_gemm_strided_batched(void* C, const void* A, const void* B, const void* bias,
                                int batch, int m, int k, int n,
                                long long a_bs, long long a_rs, long long a_cs,
                                long long b_bs, long long b_rs, long long b_cs,
                                long long c_bs, long long c_rs, long long c_cs,
                                int accumulate, int dtype) {
    if (!C || !A || !B || batch <= 0 || m <= 0 || k <= 0 || n <= 0) {
        set_error("rp_hip_gemm_strided_batched: null operand or non-positive extent (batch=%d m=%d k=%d n=%d)", batch, m, k, n);
        return -1;
    }
    if (!dtype_size(dtype)) { set_error("rp_hip_gemm_strided_batched: unsupported dtype %d", dtype); return -1; }
    // (Batch strides may have any sign: matrix z of an operand starts z strides from matrix 0, which lets one launch
    // cover separately allocated matrices of equal shape.  Row and column strides address inside a matrix.)
    if (a_rs < 0 || a_cs < 0 || b_rs < 0 || b_cs < 0 || c_rs < 0 || c_cs < 0) {
        set_error("rp_hip_gemm_strided_batched: negative row or column stride");
        return -1;
    }
    // the batch rides on a grid axis that holds at most 65535 blocks: longer batches go in chunks
    constexpr int MAX_BATCH = 65535;
    const long long esz = (long long)dtype_size(dtype);
    for (int b0 = 0; b0 < batch; b0 += MAX_BATCH) {
        const int nb = batch - b0 < MAX_BATCH ? batch - b0 : MAX_BATCH;
        GemmArgs g{(char*)C + b0 * c_bs * esz, (const char*)A + b0 * a_bs * esz, (const char*)B + b0 * b_bs * esz, bias,
                   nb, m, k, n, a_bs, a_rs, a_cs, b_bs, b_rs, b_cs, c_bs, c_rs, c_cs, accumulate};
        if (run_gemm(g, dtype) != 0) return -1;
    }
    return 0;
}

int rp_hip_gemm_strided_batched_noalloc(void* C, const void* A, const void* B, const void* bias,
                                        int batch, int m, int k, int n,
                                        long long a_bs, long long a_rs, long long a_cs,
                                        long long b_bs, long long b_rs, long long b_cs,
                                        long long c_bs, long long c_rs, long long c_cs,
                                        int accumulate, int dtype) {
    if (g_noalloc_base) { set_error("rp_hip_gemm_strided_batched_noalloc: re-entered"); return -1; }
    unsigned char* base = noalloc_scratch_of_current_device();
    if (!base) return -1;
    g_noalloc_base = base;
    g_noalloc_busy = false;
    g_noalloc_cleared = false;
    const int rc = rp_hip_gemm_strided_batched(C, A, B, bias, batch, m, k, n, a_bs, a_rs, a_cs, b_bs, b_rs, b_cs, c_bs, c_rs, c_cs, accumulate, dtype);
    g_noalloc_base = nullptr;
    g_noalloc_busy = false;
    return rc;
}

int matmul_kernel_device(void* C, const void* A, const void* B, int m, int k, int n, int dtype) {
    return rp_hip_gemm_strided_batched(C, A, B, nullptr, 1, m, k, n, 0, k, 1, 0, n, 1, 0, n, 1, 0, dtype);
}

int rp_hip_linear_backward(void* dx, void* dw, void* db, const void* dy, const void* x, const void* w, int m, int k, int n,
                           long long x_rs, long long x_cs, long long w_rs, long long w_cs,
                           long long dx_rs, long long dx_cs, long long dw_rs, long long dw_cs,
                           int accumulate_dx, int accumulate_dw, int accumulate_db, int dtype) {
    if (!dy || (dx && !w) || (dw && !x) || m <= 0 || k <= 0 || n <= 0 || !dtype_size(dtype)) {
        set_error("rp_hip_linear_backward: null operand, non-positive extent or unsupported dtype (m=%d k=%d n=%d)", m, k, n);
        return -1;
    }
    if (x_rs < 0 || x_cs < 0 || w_rs < 0 || w_cs < 0 || dx_rs < 0 || dx_cs < 0 || dw_rs < 0 || dw_cs < 0) { set_error("rp_hip_linear_backward: negative stride"); return -1; }
    // dx[m, k] = dy[m, n] . w^T (w [k, n] read with its strides swapped); dw[k, n] = x^T . dy (x [m, k] likewise)
    GemmArgs gx{dx, dy, w, nullptr, 1, m, n, k, 0, n, 1, 0, w_cs, w_rs, 0, dx_rs, dx_cs, accumulate_dx};
    GemmArgs gw{dw, x, dy, nullptr, 1, k, m, n, 0, x_cs, x_rs, 0, n, 1, 0, dw_rs, dw_cs, accumulate_dw};
    plain_k_strides(gx.m, gx.k, gx.n, gx.a_rs, gx.a_cs, gx.b_rs, gx.b_cs);
    plain_k_strides(gw.m, gw.k, gw.n, gw.a_rs, gw.a_cs, gw.b_rs, gw.b_cs);
    if (dtype == RP_DTYPE_FLOAT32 || dtype == RP_DTYPE_FLOAT64) {
        const WkwTile tx = dx ? small_tile_alone(gx, true, dtype) : WKW_TINY, tw = dw ? small_tile_alone(gw, false, dtype) : WKW_TINY;
        const bool apart = gradients_apart(gx, gw, dtype);
        if (dtype == RP_DTYPE_FLOAT32 && (dx || dw) && tx == WKW_TINY && tw == WKW_TINY && apart) {
            // small layer: one launch does all three, block for block what the separate launches would do
            const bool rides = db && bias_gradient_apart(db, gx, gw, dtype);
            if (!dx) gx.m = 0;
            if (!dw) gw.m = 0;
            if (launch_linear_backward_tiny(gx, gw, rides ? db : nullptr, dy, m, n, accumulate_db) != 0) return -1;
            return db && !rides ? rp_hip_reduce_rows(db, dy, m, n, accumulate_db, dtype) : 0;
        }
        // (many rounds of 16 x 16 tiles need the registers and the LDS that they have alone: three of them (us apart and in one launch: fp32 832 x 160 x 800 14.9 / 10.3,
        // 876 x 191 x 812 19.2 / 13.4), beside the 32 x 32 tiles of a long dW two (2659 x 49 x 3731 70.3 / 73.4, 1200 x 144 x 1408 24.7 / 26.1))
        const auto rounds16 = [&](const GemmArgs& g, WkwTile t) { return t == WKW_16X16 && (long long)((g.m + 15) / 16) * ((g.n + 15) / 16) > (tw == WKW_32X32 && m > 1024 ? 2 : 3) * cu_tiles(); };
        if (dx && dw && linear_backward_wavekw_takes(gx, gw, tx, tw, dtype) && (tx == tw || !(rounds16(gx, tx) || rounds16(gw, tw))) && apart) {
            report_kernel("linear_backward_wavek");
            const bool rides = db && m <= (n * dtype_size(dtype) % 64 ? LINEAR_DB_ROWS_WAVEKW_UNEVEN : LINEAR_DB_ROWS_WAVEKW) && bias_gradient_apart(db, gx, gw, dtype);
            if (launch_linear_backward_wavekw(gx, gw, tx, tw, rides ? db : nullptr, accumulate_db, dtype) != 0) return -1;
            return db && !rides ? rp_hip_reduce_rows(db, dy, m, n, accumulate_db, dtype) : 0;
        }
    }
    bool edge = false, dx_wavek = false, ragged = false;
    if ((dtype == RP_DTYPE_BFLOAT16 || dtype == RP_DTYPE_FLOAT16) && dx && dw && linear_backward_pairs(gx, gw, dtype, edge, dx_wavek, ragged)) {
        report_kernel("linear_backward16_64x64", ragged ? "linear_backward16_ragged" : nullptr);
        // The bias gradient rides along unless it would be written over something that is still read (one launch after the other
        // was fine), or its chain of chunks outlasts the products.
        const bool rides = db && m <= (n % 32 ? LINEAR_DB_ROWS_UNEVEN : LINEAR_DB_ROWS) && bias_gradient_apart(db, gx, gw, dtype);
        if (launch_linear_backward16(gx, gw, dx_wavek, rides ? db : nullptr, accumulate_db, edge, ragged, dtype) != 0) return -1;
        if (rides) return 0;
    } else {
        if (dx && run_gemm(gx, dtype) != 0) return -1;
        if (dw && run_gemm(gw, dtype) != 0) return -1;
    }
    if (db && rp_hip_reduce_rows(db, dy, m, n, accumulate_db, dtype) != 0) return -1;
    return 0;
}

const char* rp_hip_last_gemm_kernel(void) { return g_last_kernel; }
const char* rp_hip_last_gemm_launch(void) { return g_last_launch; }

const char* rp_hip_gemm_kernel_name(int batch, int m, int k, int n, long long a_rs, long long a_cs,
                                    long long b_rs, long long b_cs, long long c_rs, long long c_cs, int dtype) {
    if (batch <= 0 || m <= 0 || k <= 0 || n <= 0 || !dtype_size(dtype)) return "invalid";
    Plan p = make_plan(batch, m, k, n, a_rs, a_cs, b_rs, b_cs, c_rs, c_cs, 0, 0, dtype);
    return p.name;           // (mfma16_wavek, which stands in for two of the families where the pointers allow it, is reported by rp_hip_last_gemm_kernel)
}

}  // extern "C"
