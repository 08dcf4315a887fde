// fp32 / fp64 MFMA GEMM whose waves share k: what a workgroup does, for the kernel of one product (rp_gemm_wavekw.hip, which says what it is
// good for) and for the launch of all gradients of a Linear layer.
#pragma once
#include "rp_gemm.h"

namespace rp {

template <typename E> struct wkw_cfg;
template <> struct wkw_cfg<float> {
    static constexpr int KV = 4;                         // values of k in a 16-byte vector
    using acc_t = f32x4_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ constexpr int acc_row(int v, int kq) { return 4 * kq + v; }
};
template <> struct wkw_cfg<double> {
    static constexpr int KV = 2;
    using acc_t = f64x4_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ constexpr int acc_row(int v, int kq) { return 4 * v + kq; }
};

constexpr int WKW_CHUNKS = 2;                            // chunks of four vectors of k in a piece: a cache line of every row that has unit stride along k
template <typename E> constexpr int wkw_piece() { return WKW_CHUNKS * 4 * wkw_cfg<E>::KV; }
constexpr int WKW_ROW_PITCH = 128 + 32;                  // bytes of a row of a piece in LDS: the fragment reads run at full rate
constexpr int WKW_TILE_PITCH = 256 + 16;                 // values of a 16 x 16 partial tile in LDS: neighbouring tiles start 16 banks apart
constexpr bool wkw_staged(bool kc, int t) { return kc && t == 1; }
template <bool A_KC, bool B_KC, int TM, int TN>
constexpr size_t wkw_stage() { return (size_t)WKW_ROW_PITCH * 16 * ((wkw_staged(A_KC, TM) ? 1 : 0) + (wkw_staged(B_KC, TN) ? 1 : 0)); }       // bytes a wave
template <typename E, int TM, int TN, int NW>
constexpr bool wkw_halves() { return (size_t)NW * TM * TN * WKW_TILE_PITCH * sizeof(E) > 64 * 1024; }         // the upper half of the waves hands its sums to the lower half first
template <typename E, bool A_KC, bool B_KC, int TM, int TN, int NW>
constexpr size_t wkw_smem() {
    const size_t stages = NW * wkw_stage<A_KC, B_KC, TM, TN>(), parts = (size_t)(wkw_halves<E, TM, TN, NW>() ? NW / 2 : NW) * TM * TN * WKW_TILE_PITCH * sizeof(E);
    return stages > parts ? stages : parts;
}

__device__ __forceinline__ void wkw_wave_order() {       // keeps the compiler from moving a wave's LDS accesses across
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// N values in a row at byte `off` of a buffer.  (Vectors cast as a whole: arrays filled with memcpy were taken apart into bytes.)
template <typename E, int N> struct wkw_vec { typedef E type __attribute__((ext_vector_type(N))); };
template <typename E, int N> using wkw_vec_t = typename wkw_vec<E, N>::type;
template <typename E, int N>
__device__ __forceinline__ wkw_vec_t<E, N> wkw_fetch(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint32_t soff) {
    if constexpr (N * sizeof(E) == 4) return __builtin_bit_cast(wkw_vec_t<E, N>, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off, (int)soff, 0));
    else if constexpr (N * sizeof(E) == 8) return __builtin_bit_cast(wkw_vec_t<E, N>, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)off, (int)soff, 0));
    else return __builtin_bit_cast(wkw_vec_t<E, N>, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, (int)soff, 0));
}

// The fragments of a piece: T of 16 rows (of A; columns of B).  In MFMA step (c, j) lane (q, r) = (lane / 16, lane % 16) holds k = KV (4 c + q) + j.
template <typename E, int T>
struct WkwFragments { wkw_vec_t<E, wkw_cfg<E>::KV> v[WKW_CHUNKS][T]; };

// Byte offset of row `first + r` of an operand with unit stride along k, from the tile's first row (SEG: from the operand)
template <typename E, bool SEG>
__device__ __forceinline__ uint32_t wkw_row_offset(const GemmArgs& g, long long fs, int first, int extent, int r) {
    const int row = first + r < extent ? first + r : extent - 1;
    if constexpr (SEG) {
        const int seg = row / g.seg_n, c = row - seg * g.seg_n;
        return (uint32_t)((seg / g.seg_w * g.seg_sh + seg % g.seg_w * g.seg_sw + c * fs) * (long long)sizeof(E));
    }
    return (uint32_t)((row - first) * fs * (long long)sizeof(E));
}

// Pieces of one operand on their way, and where a lane finds its part of them.
// Unit stride along k, 16 rows: a load takes whole lines of eight rows, and LDS of the wave's own turns rows into fragments.
// SEG: B's k or n axis is a list of segments (GemmArgs::seg_*), for convolutions.
template <typename E, bool KC, int T, bool SEG>
struct WkwOperand {
    static_assert(KC && T == 1, "the others are below");
    static constexpr int KV = wkw_cfg<E>::KV, SZ = (int)sizeof(E);
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[2], lds_write, lds_read;                // bytes
    int k_lane;                                          // k of this lane's vectors, from the piece's start
    struct Piece { wkw_vec_t<E, KV> raw[2]; };

    // first: the tile's first row; rows past the last one read the last one
    __device__ __forceinline__ void init(const GemmArgs& g, const E* base, long long fs, long long ks, int first, int extent, int lane) {
        rsrc = buffer_rsrc(base + (SEG ? 0 : (long long)first * fs), 0x7fffffffll);
        k_lane = lane % 8 * KV;
#pragma unroll
        for (int i = 0; i < 2; i++) off[i] = wkw_row_offset<E, SEG>(g, fs, first, extent, 8 * i + lane / 8) + k_lane * SZ;
        lds_write = lane / 8 * WKW_ROW_PITCH + lane % 8 * 16;
        lds_read = lane % 16 * WKW_ROW_PITCH + lane / 16 * 16;
    }
    __device__ __forceinline__ void load(Piece& p, int piece) const {
#pragma unroll
        for (int i = 0; i < 2; i++) p.raw[i] = wkw_fetch<E, KV>(rsrc, off[i], piece * 128);
    }
    // a piece that k ends in: zeros from `left` values of k on
    __device__ __forceinline__ void load_end(Piece& p, int piece, int left) const {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < KV; e++) p.raw[i][e] = wkw_fetch<E, 1>(rsrc, k_lane + e < left ? off[i] + e * SZ + piece * 128u : BUFFER_OOB, 0)[0];
    }
    __device__ __forceinline__ void park(const Piece& p, unsigned char* stage) const {
#pragma unroll
        for (int i = 0; i < 2; i++) *(wkw_vec_t<E, KV>*)(stage + lds_write + i * 8 * WKW_ROW_PITCH) = p.raw[i];
    }
    static __device__ __forceinline__ E value(const Piece&, const WkwFragments<E, T>& f, int c, int t, int j) { return f.v[c][t][j]; }
    __device__ __forceinline__ void fragments(WkwFragments<E, T>& f, const unsigned char* stage) const {
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++) f.v[c][0] = *(const wkw_vec_t<E, KV>*)(stage + lds_read + c * 64);
    }
};

// Unit stride along k, more rows: fragment t holds rows 16 t + r, loaded as it is.
template <typename E, int T, bool SEG>
struct WkwOperandRows {
    static constexpr int KV = wkw_cfg<E>::KV, SZ = (int)sizeof(E);
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[T];                                     // bytes
    int k_lane;
    struct Piece { wkw_vec_t<E, KV> v[WKW_CHUNKS][T]; };

    __device__ __forceinline__ void init(const GemmArgs& g, const E* base, long long fs, long long ks, int first, int extent, int lane) {
        rsrc = buffer_rsrc(base + (SEG ? 0 : (long long)first * fs), 0x7fffffffll);
        k_lane = lane / 16 * KV;
#pragma unroll
        for (int t = 0; t < T; t++) off[t] = wkw_row_offset<E, SEG>(g, fs, first, extent, 16 * t + lane % 16) + k_lane * SZ;
    }
    __device__ __forceinline__ void load(Piece& p, int piece) const {
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++)
#pragma unroll
            for (int t = 0; t < T; t++) p.v[c][t] = wkw_fetch<E, KV>(rsrc, off[t], piece * 128 + c * 64);
    }
    __device__ __forceinline__ void load_end(Piece& p, int piece, int left) const {
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++)
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int e = 0; e < KV; e++)
                    p.v[c][t][e] = wkw_fetch<E, 1>(rsrc, c * 4 * KV + k_lane + e < left ? off[t] + e * SZ + piece * 128u + c * 64u : BUFFER_OOB, 0)[0];
    }
    __device__ __forceinline__ void park(const Piece&, unsigned char*) const {}
    static __device__ __forceinline__ E value(const Piece& p, const WkwFragments<E, T>&, int c, int t, int j) { return p.v[c][t][j]; }
    __device__ __forceinline__ void fragments(WkwFragments<E, T>&, const unsigned char*) const {}
};

// Unit stride along the free index: fragment t holds rows T r + t, so that a lane's T values of a k row are neighbours and 16 lanes load a
// stretch of it, which is a fragment as it is.
template <typename E, int T, bool SEG>
struct WkwOperand<E, false, T, SEG> {
    static constexpr int KV = wkw_cfg<E>::KV, SZ = (int)sizeof(E);
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[KV], k_bytes;                           // bytes; from one k to the next
    int k_lane;
    struct Piece { wkw_vec_t<E, T> row[WKW_CHUNKS][KV]; };

    int seg_k, seg_w;
    uint32_t seg_sh, seg_sw;                             // bytes

    // first: at most extent - 16 T
    __device__ __forceinline__ void init(const GemmArgs& g, const E* base, long long fs, long long ks, int first, int extent, int lane) {
        rsrc = buffer_rsrc(base + first, 0x7fffffffll);
        if constexpr (SEG) { seg_k = g.seg_k; seg_w = g.seg_w; seg_sh = (uint32_t)(g.seg_sh * SZ); seg_sw = (uint32_t)(g.seg_sw * SZ); }
        k_bytes = (uint32_t)ks * SZ;
        k_lane = lane / 16 * KV;
#pragma unroll
        for (int j = 0; j < KV; j++) off[j] = (uint32_t)(k_lane + j) * k_bytes + lane % 16 * T * SZ;
    }
    // a piece lies inside a segment (whole pieces long)
    __device__ __forceinline__ void load(Piece& p, int piece) const {
        uint32_t start = 0, k0 = (uint32_t)piece * wkw_piece<E>();
        if constexpr (SEG) {
            const uint32_t seg = k0 / (uint32_t)seg_k, row = seg / (uint32_t)seg_w;
            k0 -= seg * (uint32_t)seg_k;
            start = row * seg_sh + (seg - row * (uint32_t)seg_w) * seg_sw;
        }
        start += k0 * k_bytes;
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++)
#pragma unroll
            for (int j = 0; j < KV; j++) p.row[c][j] = wkw_fetch<E, T>(rsrc, off[j], start + (uint32_t)c * 4 * KV * k_bytes);
    }
    __device__ __forceinline__ void load_end(Piece& p, int piece, int left) const {
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++)
#pragma unroll
            for (int j = 0; j < KV; j++)
                p.row[c][j] = wkw_fetch<E, T>(rsrc, c * 4 * KV + k_lane + j < left ? off[j] + (uint32_t)(piece * WKW_CHUNKS + c) * 4 * KV * k_bytes : BUFFER_OOB, 0);
    }
    __device__ __forceinline__ void park(const Piece&, unsigned char*) const {}
    static __device__ __forceinline__ E value(const Piece& p, const WkwFragments<E, T>&, int c, int t, int j) { return p.row[c][j][t]; }
    __device__ __forceinline__ void fragments(WkwFragments<E, T>&, const unsigned char*) const {}
};

template <typename E, bool KC, int T, bool SEG>
using wkw_operand = std::conditional_t<KC && (T > 1), WkwOperandRows<E, T, SEG>, WkwOperand<E, KC, T == 1 || !KC ? T : 1, SEG>>;

// A 16 TM x 16 TN tile, number `block` of the schedule of `batch` matrices, by NW waves.  k goes in pieces, dealt to the waves in turn: a wave multiplies one piece out of
// registers while the next is on its way there, and the partial tiles meet in LDS, where they are added in a fixed order.
template <typename E, bool A_KC, bool B_KC, int TM, int TN, int NW, bool SEG = false>
__device__ __forceinline__ void gemm_wavekw_block(const GemmArgs& g, int tiles_m, int tiles_n, int block, int batch, unsigned char* lds) {
    using cfg = wkw_cfg<E>;
    using OpA = wkw_operand<E, A_KC, TM, false>;
    using OpB = wkw_operand<E, B_KC, TN, SEG>;
    constexpr int PK = wkw_piece<E>(), KV = cfg::KV;
    constexpr bool STAGED = wkw_staged(A_KC, TM) || wkw_staged(B_KC, TN);
    // block b runs on XCD b % 8: a run of matrices, and of tiles along the shorter side of an output, for each XCD, whose L2 then serves what they share.
    // (With a run of every matrix's tiles for each XCD, 250 matrices of one tile each were all on the first: 64 x 512 x 64 114 us, 25.)
    const int tiles = tiles_m * tiles_n, total = tiles * batch, per = (total + 7) / 8, at = block % 8 * per + block / 8;
    if (block / 8 >= per || at >= total) return;
    const int z = at / tiles, idx = at - z * tiles;
    const bool tall = tiles_m > tiles_n;
    const int m0 = (tall ? idx / tiles_n : idx % tiles_m) * 16 * TM, n0 = (tall ? idx % tiles_n : idx / tiles_m) * 16 * TN;
    // where a row of an operand is a row of k the last tile starts early, so that it ends with the operand; only its own part is stored
    const int ms = A_KC || m0 + 16 * TM <= g.m ? m0 : g.m - 16 * TM, ns = B_KC || n0 + 16 * TN <= g.n ? n0 : g.n - 16 * TN;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    OpA opa;
    OpB opb;
    opa.init(g, (const E*)g.A + (long long)z * g.a_bs, g.a_rs, g.a_cs, ms, g.m, lane);
    opb.init(g, (const E*)g.B + (long long)z * g.b_bs, g.b_cs, g.b_rs, ns, g.n, lane);
    unsigned char* const a_stage = lds + wave * wkw_stage<A_KC, B_KC, TM, TN>(), * const b_stage = a_stage + (wkw_staged(A_KC, TM) ? 16 * WKW_ROW_PITCH : 0);

    // Two pieces on their way at a time.  Sets of accumulators: where there are registers for them a piece's chunks, and pieces in turn, have their
    // own, so that k is summed in NW to 4 NW chains, which are added at the end.
    constexpr int BY_CHUNK = sizeof(E) == 4 && TM <= 2 && TN <= 2 ? WKW_CHUNKS : 1, SETS = BY_CHUNK * (TM * TN <= 2 ? 2 : 1);
    using acc_t = typename cfg::acc_t;
    acc_t sums[SETS][TM][TN];
#pragma unroll
    for (int d = 0; d < SETS; d++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) sums[d][i][j] = acc_t{0, 0, 0, 0};
    typename OpA::Piece a0, a1;
    typename OpB::Piece b0, b1;
    auto request = [&](typename OpA::Piece& a, typename OpB::Piece& b, int piece) {
        opa.load(a, piece);
        opb.load(b, piece);
    };
    auto multiply = [&](const typename OpA::Piece& a, const typename OpB::Piece& b, auto turn) {
        if constexpr (STAGED) {
            wkw_wave_order();                            // (a wave's LDS operations are executed in order)
            opa.park(a, a_stage);
            opb.park(b, b_stage);
            wkw_wave_order();
        }
        WkwFragments<E, TM> fa;
        WkwFragments<E, TN> fb;
        opa.fragments(fa, a_stage);
        opb.fragments(fb, b_stage);
#pragma unroll
        for (int c = 0; c < WKW_CHUNKS; c++)
#pragma unroll
            for (int s = 0; s < KV; s++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        acc_t& acc = sums[(decltype(turn)::value * BY_CHUNK + c % BY_CHUNK) % SETS][i][j];
                        acc = cfg::mma(OpA::value(a, fa, c, i, s), OpB::value(b, fb, c, j, s), acc);
                    }
    };
    const int whole = g.k / PK, mine = whole > wave ? (whole - wave - 1) / NW + 1 : 0;
    int p = wave, left = mine;                           // the next piece to multiply, and how many there are from it on
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // (requests without a condition inside the loop: the compiler's waits then count the loads exactly)
    if (left > 0) request(a0, b0, p);
    for (; left > 2; left -= 2, p += 2 * NW) {
        request(a1, b1, p + NW);
        multiply(a0, b0, I0{});
        request(a0, b0, p + 2 * NW);
        multiply(a1, b1, I1{});
    }
    if (left == 2) {
        request(a1, b1, p + NW);
        multiply(a0, b0, I0{});
        multiply(a1, b1, I1{});
    } else if (left == 1) {
        multiply(a0, b0, I0{});
    }
    if (g.k % PK != 0 && wave == whole % NW) {           // (the wave whose turn it is)
        opa.load_end(a0, whole, g.k - whole * PK);
        opb.load_end(b0, whole, g.k - whole * PK);
        multiply(a0, b0, I0{});
    }
    acc_t (&acc)[TM][TN] = sums[0];
#pragma unroll
    for (int d = 1; d < SETS; d++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] += sums[d][i][j];

    if constexpr (STAGED) __syncthreads();         // every wave is done with its stage
    E* const parts = (E*)lds;                            // [share][tile][register][lane]
    constexpr int SHARE = TM * TN * WKW_TILE_PITCH;
    constexpr int SHARES = wkw_halves<E, TM, TN, NW>() ? NW / 2 : NW;
    auto put = [&](E* to) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) to[(i * TN + j) * WKW_TILE_PITCH + v * 64 + lane] = acc[i][j][v];
    };
    if constexpr (SHARES < NW) {
        if (wave >= SHARES) put(parts + (wave - SHARES) * SHARE);
        __syncthreads();
        if (wave < SHARES) {
            const E* from = parts + wave * SHARE;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[i][j][v] += from[(i * TN + j) * WKW_TILE_PITCH + v * 64 + lane];
            put(parts + wave * SHARE);                   // (a wave writes where it alone has read)
        }
    } else {
        put(parts + wave * SHARE);
    }
    __syncthreads();
    const E* bias = (const E*)g.bias;
    E* C = (E*)g.C + (long long)z * g.c_bs;
    for (int e = t; e < 256 * TM * TN; e += 64 * NW) {
        const int row = e / (16 * TN), col = e % (16 * TN), gm = ms + row, gn = ns + col;
        const int i = A_KC ? row / 16 : row % TM, ri = A_KC ? row % 16 : row / TM, j = B_KC ? col / 16 : col % TN, ci = B_KC ? col % 16 : col / TN;
        const int at = (i * TN + j) * WKW_TILE_PITCH + (sizeof(E) == 4 ? (ri % 4) * 64 + (ri / 4) * 16 : (ri / 4) * 64 + (ri % 4) * 16) + ci;
        E sum = parts[at];
#pragma unroll
        for (int w = 1; w < SHARES; w++) sum += parts[w * SHARE + at];
        if (gm < m0 || gm >= g.m || gn < n0 || gn >= g.n) continue;
        if constexpr (SEG) {                             // folded output, bias per row: see GemmArgs
            int at_col = gn;
            if (g.c_fold_from > 0) {
                const int run = gn / g.c_fold_from, within = gn - run * g.c_fold_from;
                if (within >= g.c_fold_to) continue;
                at_col = run * g.c_fold_to + within;
            }
            C[gm * g.c_rs + at_col * g.c_cs] = finish<E>(sum, bias != nullptr, bias ? bias[g.bias_by_row ? gm : gn] : (E)0, false, (E)0);
            continue;
        }
        E* out = C + gm * g.c_rs + gn * g.c_cs;
        *out = finish<E>(sum, bias != nullptr, bias ? bias[gn] : (E)0, g.accumulate != 0, g.accumulate ? *out : (E)0);
    }
}

// Tiles of a product, and whether the operands can be addressed that way; WKW_NONE: not at all
// WKW_FEW_ROWS: 16 x 32 with chains of at most 32 values; WKW_TINY: the 16 x 16 tiles of rp_gemm_tiny.h, two a workgroup
enum WkwTile { WKW_NONE, WKW_16X16, WKW_16X32, WKW_32X32, WKW_16X64, WKW_64X64, WKW_FEW_ROWS, WKW_TINY };
WkwTile wavekw_tile(const GemmArgs& g, int dtype);
const char* wavekw_name(WkwTile tile, int dtype);                   // what rp_hip_last_gemm_launch says of it
int launch_wavekw(const GemmArgs& g, WkwTile tile, int dtype);      // fp32 / fp64 products that the waves of a workgroup share, see wavekw_takes
int launch_wavekw_segmented(const GemmArgs& g, WkwTile tile);       // fp32, A with unit stride along k, B in segments
// All gradients of a Linear layer in one launch, each product on the tiles that it would get alone; gx.A is dY [gx.m, gx.k], dense; db: gx.k column sums of dY, or null
bool linear_backward_wavekw_takes(const GemmArgs& gx, const GemmArgs& gw, WkwTile x, WkwTile w, int dtype);
int launch_linear_backward_wavekw(const GemmArgs& gx, const GemmArgs& gw, WkwTile x, WkwTile w, void* db, int accumulate_db, int dtype);
static inline bool wkw_a_kc(const GemmArgs& g) { return g.a_cs == 1; }
static inline bool wkw_b_kc(const GemmArgs& g) { return g.b_rs == 1 && (g.b_cs != 1 || g.n == 1); }

}  // namespace rp
