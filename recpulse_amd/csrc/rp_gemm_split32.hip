// fp32 GEMM on the bf16 matrix cores: every fp32 value as the exact sum of three bf16 values.
//
// The fp32 MFMA runs 128 multiply-adds per cycle and CU, the bf16 MFMA sixteen times as many.  x = h + m + l with h = bf16(x),
// m = bf16(x - h), l = x - h - m is exact (8 + 8 + 8 significant bits, each with its own sign, cover 24), so
//   a b = ah bh + (ah bm + am bh) + (am bm + ah bl + al bh) + [am bl + al bm + al bl]
// where the bracket is at most 2^-24 |a b| (|m| <= 2^-8 |h| and |l| <= 2^-17 |h|, so am bl and al bm reach 2^-25 each), as much as the
// rounding of a single fp32 product, and is left out: six bf16 MFMAs (whose products are exact in fp32) of 32 cycles per
// k-step of 16 stand in for eight fp32 MFMAs of 64.  The five small products go to an accumulator of their own, and the two
// meet once, in the epilogue: the large one then rounds once per 16 k instead of once per product or two.  2-norm error against
// 64 bits, this kernel / the fp32 MFMA kernel: N(0,1) values, k = 67 5.1e-8 / 1.5e-7, 256 9.0e-8 / 2.9e-7, 1024 1.9e-7 / 5.7e-7, 4096
// 4.0e-7 / 1.15e-6, the same in every layout; uniform values in [0, 1), k = 256 8.4e-8 / 2.2e-7, 4096 3.0e-7 / 8.4e-7; values spread over
// 2^+-30, k = 128 6.48e-8 / 6.46e-8, 4096 2.9e-7 / 3.3e-7.  Where a row has one significant term there is nothing to gain and the bracket
// shows: a diagonal matrix of N(0,1) times N(0,1) 2.60e-8 / 2.53e-8, the largest error of a value 1.67 x 2^-24 instead of 1.00.  (With
// am bl and al bm kept it is 1.00 again and no other figure moves by more than 1 %; 4096^3 then takes 870 us, 2048^3 150.)
//
// What the split cannot hold: infinities, NaN and values that round to bf16 infinity (their m and l become NaN, so every
// output they touch is NaN, here or in a finite dot product that overflowed), and values below 2^-110 whose last bits fall
// below the smallest bf16 subnormal (then what is left for l is no bf16 value).  Nor are the small products of results below
// 2^-110 held: they are subnormal, and each of the 6 k / 16 sums rounds to 2^-149 (up to k = 2^16 less than half an ulp of 2^-110).
// A wave that splits a value with such a rest says so in LDS; from that slab on the workgroup multiplies with fp32 MFMAs.  A tile
// whose result holds an infinity, a NaN or a tiny value is computed again that way from the first slab on.  So such inputs get the
// fp32 kernel's precision.  4096^3, one value of 1.2345 x 2^-115 per 128 rows, at the first, the middle and the last k: 1 200, 925 and
// 727 us, a sixteenth of all values 1 200 (725 without, 1 075 on the fp32 kernel; finding out at the end and computing such
// tiles again took 1 880); one infinity per 128 rows 1 820.  Looking for the smallest magnitude instead of a rest: 733 without.
// The check of the results costs 0.5 us: 1536 x 96 x 1536 16.3 -> 16.8 us, 2048^3 128 -> 131.
//
// Shape: 128 x 128 tile, 4 waves of 64 x 64, k slab 32.  A slab is fetched to registers as fp32 (16 values of either operand
// per thread), split there and written to LDS as rows of [32 h | 32 m | 32 l]; all four operand layouts leave the same
// rows, so the multiplying half is common to them.  Fragment reads per MFMA are half those of a plain bf16 kernel (twelve for
// 24 MFMAs).  LDS holds one slab (52 KB): two workgroups share a CU.  The next slab is requested at the start of this one's
// 48 MFMAs and split between those of the second half, two values after one or two MFMAs (splitting between the two barriers
// instead: 4096^3 788 us against 745, 2048^3 162 against 129).
//
// What bounds it: 52 % of the cycles are MFMA-busy, at a clock of 1.9 GHz and less that the power limit leaves.  4096^3: 725 -
// 800 us (890 back to back for long) where the fp32 MFMAs take 1 075 - 1 240; 2048^3 131 against 153; 3001 x 1027 x 2049 100 against 222.
#include "rp_gemm.h"

namespace rp {

namespace {

constexpr int S32_BK = 32;
constexpr int S32_PITCH = 3 * S32_BK + 8;           // 16-bit elements per LDS row: 16 rows of ds_read_b128 cover all banks once

// the products that are kept, as planes of A and B (0: h, 1: m, 2: l), the large one first
constexpr int S32_PA[6] = {0, 0, 1, 1, 0, 2}, S32_PB[6] = {0, 1, 0, 1, 2, 0};
constexpr int FP_NAN_INF_SUBNORMAL = 0x297;         // of v_cmp_class: both NaNs, both infinities, both signs of subnormal
constexpr int S32_MFMAS = 6 * 4;        // of a k-step of 16: four tiles of 32 x 32

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;

__device__ __forceinline__ uint32_t s32_pack(float a, float b) {
    const bf16x2_t v = {(__bf16)a, (__bf16)b};                        // one packed conversion, round to nearest even
    return __builtin_bit_cast(uint32_t, v);
}

// two values -> their h, m and l pairs.  lost collects the bits of what is left for l: it is a bf16 value, as it always is unless it
// falls below the bf16 subnormals, if its low half is zero.
__device__ __forceinline__ void s32_split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l, uint32_t& lost) {
    h = s32_pack(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xFFFF0000u);
    m = s32_pack(r0, r1);
    const float l0 = r0 - __uint_as_float(m << 16), l1 = r1 - __uint_as_float(m & 0xFFFF0000u);
    l = s32_pack(l0, l1);
    lost |= __float_as_uint(l0) | __float_as_uint(l1);
}

// One operand's slab traffic.  A thread holds four vectors of four values along the unit-stride axis.
//   KC (unit stride along k): vector i is row t / 8 + 32 i, k 4 (t % 8) .. + 3.
//   MC (unit stride along the free axis): vector i is k 4 (t % 8) + i, rows 4 (t / 8) .. + 3: a 4 x 4 block, transposed in
//   registers; eight lanes span the slab's k (64 bytes of an LDS row), a wave reads whole 128-byte lines of eight k rows at a time.
// EDGE: extents and row starts of any size (otherwise the tile and all slabs are whole).  A vector that straddles the end of its
// row is fetched `pull` elements further back, where it ends with the row, and shifted into place.
template <int ROWS, bool MC, bool EDGE>
struct S32Slab {
    static_assert(ROWS * S32_BK == 256 * 16, "16 values per thread");
    u32x4_t v[4];
    u32x2_t planes[4][3];         // rows' h, m and l
    int r0, kk0;                  // first free index and k of vector 0
    uint32_t goff[EDGE ? 4 : 1];  // byte offset of the vectors from the slab pointer
    int step;                     // bytes between vectors
    int pull;                     // MC: elements the vectors stick out of the free axis
    const char* slab;
    const char* end;
    long long slab_step;
    __device__ __forceinline__ void init(const float* base, long long free_stride, long long k_stride, int row0, int free_extent, int k0, int k, int t) {
        r0 = MC ? 4 * (t / 8) : t / 8;
        kk0 = 4 * (t % 8);
        slab = (const char*)(base + (long long)row0 * free_stride + (long long)k0 * k_stride);
        end = (const char*)(base + (long long)(free_extent - 1) * free_stride + (long long)(k - 1) * k_stride + 1);
        slab_step = (long long)S32_BK * k_stride * 4;
        step = (int)((MC ? k_stride : 32 * free_stride) * 4);
        pull = 0;
        if (EDGE && MC) {
            const int in = free_extent - row0 - r0;
            pull = in > 0 && in < 4 ? 4 - in : 0;
        }
#pragma unroll
        for (int i = 0; i < (EDGE ? 4 : 1); i++) {
            const int r = r0 + (MC ? 0 : 32 * i), kk = kk0 + (MC ? i : 0);
            goff[i] = (uint32_t)(((long long)r * free_stride + (long long)kk * k_stride) * 4) + (EDGE ? 16 : 0);
            if (EDGE && row0 + r >= free_extent) goff[i] = BUFFER_OOB;
        }
    }
    // the slab `slab` points at, of which kleft k are in range; then on to the next one
    __device__ __forceinline__ void load(int kleft) {
        if constexpr (!EDGE) {
            const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(slab, 0x7fffffffll);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)goff[0], i * step, 0);
        } else {
            const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(slab - 16, (long long)(end - slab) + 16);      // starts early: pulled-back offsets stay positive
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int in = kleft - kk0 - (MC ? i : 0);
                const int back = MC ? pull : (in > 0 && in < 4 ? 4 - in : 0);
                v[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, in > 0 ? (int)(goff[i] - 4 * back) : (int)BUFFER_OOB, 0, 0);
            }
        }
        slab += slab_step;
    }
    // straddling vectors into place (kleft: of the slab that was loaded)
    __device__ __forceinline__ void settle(int kleft) {
        if constexpr (EDGE) {
            const int in = kleft - kk0;
            const int back = MC ? pull : (in > 0 && in < 4 ? 4 - in : 0);
            if (__builtin_amdgcn_ballot_w64(back != 0) == 0) return;
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = __builtin_bit_cast(u32x4_t, __builtin_bit_cast(unsigned __int128, v[i]) >> (32 * back));
        }
    }
    __device__ __forceinline__ float at(int i, int e) const { return __uint_as_float(v[i][e]); }
    // unit u = 0 .. 7 of the split: two values of row u / 2 of the thread's four
    template <int U>
    __device__ __forceinline__ void split(uint32_t& lost) {
        constexpr int j = U / 2, p = U % 2;
        const float x0 = MC ? at(2 * p, j) : at(j, 2 * p), x1 = MC ? at(2 * p + 1, j) : at(j, 2 * p + 1);
        uint32_t h, m, l;
        s32_split2(x0, x1, h, m, l, lost);
        planes[j][0][p] = h; planes[j][1][p] = m; planes[j][2][p] = l;
    }
    __device__ __forceinline__ void split_all(uint32_t& lost) {
        static_for<0, 8>([&](auto u) { split<decltype(u)::value>(lost); });
    }
    __device__ __forceinline__ void store(uint16_t* lds) const {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint16_t* row = lds + (r0 + (MC ? j : 32 * j)) * S32_PITCH + kk0;
#pragma unroll
            for (int q = 0; q < 3; q++) *(u32x2_t*)(row + q * S32_BK) = planes[j][q];
        }
    }
    // the slab as fp32, k-major [32][ROWS + 4], for the fp32 MFMAs
    __device__ __forceinline__ void store_plain(float* lds) const {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (MC) *(u32x4_t*)(lds + (kk0 + i) * (ROWS + 4) + r0) = v[i];
            else
#pragma unroll
                for (int e = 0; e < 4; e++) lds[(kk0 + e) * (ROWS + 4) + r0 + 32 * i] = at(i, e);
        }
    }
};

}  // namespace

template <bool A_MC, bool B_MC, bool EDGE>
__global__ void __launch_bounds__(256, 2) gemm_split32_kernel(GemmArgs g, int tiles_m, int tiles_n) {
    constexpr int BM = 128, BN = 128, TM = 2, TN = 2;
    __shared__ __attribute__((aligned(16))) uint16_t lds[(BM + BN) * S32_PITCH];
    __shared__ int spare[64];
    __shared__ int odd_slab;             // the last slab that met a value which does not split
    static_assert(sizeof(lds) >= (size_t)S32_BK * (BM + 4 + BN + 4) * 4, "room for the fp32 slab");
    const TileCoord tc = schedule_tile(blockIdx.x, tiles_m, tiles_n);
    if (!tc.valid) return;
    const int z = blockIdx.y, m0 = tc.tm * BM, n0 = tc.tn * BN;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
    const int lf = lane & 31, lk = lane >> 5;
    const float* A = (const float*)g.A + (long long)z * g.a_bs;
    const float* B = (const float*)g.B + (long long)z * g.b_bs;
    uint16_t* const a_lds = lds;
    uint16_t* const b_lds = lds + BM * S32_PITCH;
    float* const a_plain = (float*)lds;
    float* const b_plain = a_plain + S32_BK * (BM + 4);

    f32x16_t big[TM][TN], small[TM][TN];
    auto clear = [&](f32x16_t (&acc)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
    };
    clear(big);
    clear(small);
    S32Slab<BM, A_MC, EDGE> sa;
    S32Slab<BN, B_MC, EDGE> sb;
    auto init = [&](int k0) {
        sa.init(A, g.a_rs, g.a_cs, m0, g.m, k0, g.k, t);
        sb.init(B, g.b_cs, g.b_rs, n0, g.n, k0, g.k, t);
    };
    auto request = [&](int kleft) { sa.load(kleft); sb.load(kleft); };
    auto settle = [&](int kleft) { sa.settle(kleft); sb.settle(kleft); };
    auto store = [&] { sa.store(a_lds); sb.store(b_lds); };
    // the slab in LDS as fp32 on the fp32 MFMAs
    auto multiply_plain = [&] {
        for (int kk = lk; kk < S32_BK; kk += 2) {
            float af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) af[i] = a_plain[kk * (BM + 4) + wm0 + 32 * i + lf];
#pragma unroll
            for (int j = 0; j < TN; j++) bf[j] = b_plain[kk * (BN + 4) + wn0 + 32 * j + lf];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) big[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], big[i][j], 0, 0, 0);
        }
    };

    // A slab is split, its waves say whether they met a value that does not split (`mark`), a barrier lets go of the slab
    // before it, its planes are stored, and after the next barrier all waves know (`odd`) how it is to be multiplied.
    uint32_t lost = 0;
    auto mark = [&](int slab) {
        ((lost & 0xFFFFu) != 0 ? &odd_slab : spare + lane)[0] = slab;         // (no branch here: with one, 2048^3 took 143 us instead of 130.5)
        lost = 0;
    };
    int odd;
    auto publish = [&] {
        __syncthreads();
        odd = odd_slab;
        store();
        __syncthreads();
        odd = __builtin_amdgcn_readfirstlane(odd);
    };
    // lane's fragment of MFMA tile i: row 32 i + lane % 32, k 8 (lane / 32) .. + 7 of a step of 16
    const uint16_t* const a_fr = a_lds + (wm0 + lf) * S32_PITCH + 8 * lk;
    const uint16_t* const b_fr = b_lds + (wn0 + lf) * S32_PITCH + 8 * lk;
    // one slab out of its planes; the next one is requested at its start and split between the MFMAs of its second half
    auto step = [&](int kleft, auto next_tag) {
        constexpr bool NEXT = decltype(next_tag)::value;
        if constexpr (NEXT) request(kleft - S32_BK);
        static_for<0, 2>([&](auto ksc) {
            constexpr int ks = decltype(ksc)::value;
            bf16x8_t af[TM][3], bf[TN][3];
#pragma unroll
            for (int p = 0; p < 3; p++) {
#pragma unroll
                for (int i = 0; i < TM; i++) af[i][p] = *(const bf16x8_t*)(a_fr + 32 * i * S32_PITCH + p * S32_BK + 16 * ks);
#pragma unroll
                for (int j = 0; j < TN; j++) bf[j][p] = *(const bf16x8_t*)(b_fr + 32 * j * S32_PITCH + p * S32_BK + 16 * ks);
            }
            if constexpr (NEXT && ks == 1) settle(kleft - S32_BK);
            static_for<0, S32_MFMAS>([&](auto qc) {
                constexpr int q = decltype(qc)::value, i = (q / TN) % TM, j = q % TN, prod = q / (TM * TN);
                f32x16_t& acc = prod == 0 ? big[i][j] : small[i][j];
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][S32_PA[prod]], bf[j][S32_PB[prod]], acc, 0, 0, 0);
                if constexpr (NEXT && ks == 1) {
                    static_for<16 * q / S32_MFMAS, 16 * (q + 1) / S32_MFMAS>([&](auto uc) {
                        constexpr int u = decltype(uc)::value;
                        if constexpr (u < 8) sa.template split<u>(lost);
                        else sb.template split<u - 8>(lost);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        });
    };

    init(0);
    request(g.k);
    if (t == 0) odd_slab = -1;
    settle(g.k);
    sa.split_all(lost);
    sb.split_all(lost);
    __syncthreads();
    mark(0);
    publish();
    int kleft = g.k, slab = 0;
    for (; kleft > S32_BK && odd != slab; kleft -= S32_BK) {
        step(kleft, std::true_type{});
        mark(++slab);
        publish();
    }
    if (odd != slab) {
        step(kleft, std::false_type{});
        kleft = 0;
    }
    // whether a result is one that the split cannot hold
    auto unsplittable = [&] {
        bool any = false;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    // (subnormal after 2^-16: below 2^-110)
                    any |= __builtin_amdgcn_classf(big[i][j][v] * 1.52587890625e-05f, FP_NAN_INF_SUBNORMAL);
                }
        return __syncthreads_or(any) != 0;
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) big[i][j][v] += small[i][j][v];
    if (unsplittable()) {                  // all of the tile again
        clear(big);
        kleft = g.k;
    }
    while (kleft > 0) {                    // what is left from the first odd slab on, or everything
        const bool whole = kleft == g.k;
        init(g.k - kleft);
        request(kleft);
        for (; kleft > 0; kleft -= S32_BK) {
            settle(kleft);
            sa.store_plain(a_plain);
            sb.store_plain(b_plain);
            __syncthreads();
            if (kleft > S32_BK) request(kleft - S32_BK);
            multiply_plain();
            __syncthreads();
        }
        if (!whole && unsplittable()) {
            clear(big);
            kleft = g.k;
        }
    }

    // straight from the accumulators: a store instruction is 32 adjacent columns of two rows
    float* C = (float*)g.C + (long long)z * g.c_bs;
    const float* bias = (const float*)g.bias;
    const bool has_bias = bias != nullptr, accum = g.accumulate != 0;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int gn = n0 + wn0 + 32 * j + lf;
        const bool col_ok = !EDGE || gn < g.n;
        const float bv = has_bias && col_ok ? bias[gn] : 0.f;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int gm = m0 + wm0 + 32 * i + 8 * (v / 4) + 4 * lk + (v % 4);
                if (EDGE && !(col_ok && gm < g.m)) continue;
                float* pc = C + (long long)gm * g.c_rs + (long long)gn * g.c_cs;
                *pc = finish<float>(big[i][j][v], has_bias, bv, accum, accum ? *pc : 0.f);
            }
    }
}

template <bool A_MC, bool B_MC>
static int launch_split32_layout(const GemmArgs& g, bool edge) {
    const int tiles_m = (g.m + 127) / 128, tiles_n = (g.n + 127) / 128;
    const dim3 grid(scheduled_grid(tiles_m, tiles_n), g.batch);
    if (edge) hipLaunchKernelGGL((gemm_split32_kernel<A_MC, B_MC, true>), grid, dim3(256), 0, current_stream(), g, tiles_m, tiles_n);
    else hipLaunchKernelGGL((gemm_split32_kernel<A_MC, B_MC, false>), grid, dim3(256), 0, current_stream(), g, tiles_m, tiles_n);
    return check_launch("gemm_split32_kernel") ? 0 : -1;
}

// Every fp32 product that the 128 x 128 tile is right for and whose k is not one or two slabs of whole vectors (those have a
// kernel that pipelines across tiles).  With the 64 x 64 tile a slab's split would take longer than its MFMAs.  Segmented
// operands and the convolution's epilogue options stay with the fp32 MFMA kernel, and so do short reductions of whole tiles
// that are at most one to a CU with both operands contiguous along their free axes (the weight gradient of a small batch), which
// need the 4 x 4 transposes here and none there: 512 x 128 x 4096 19.5 us here and 16.6 there, 512 x 256 x 4096 27.3 and 25.1.
bool split32_takes(const GemmArgs& g, const Plan& p) {
    const long long tiles = (long long)((g.m + 127) / 128) * ((g.n + 127) / 128) * g.batch;
    if (p.a_mc && p.b_mc && !p.ragged && !p.edge && g.k <= 256 && tiles <= device_cu_count()) return false;
    return p.bm == 128 && g.seg_k == 0 && g.seg_n == 0 && g.c_fold_from == 0 && !g.bias_by_row && !path_disabled("split32");
}

int launch_split32(const GemmArgs& g, const Plan& p) {
    const bool edge = p.ragged || g.m % 128 || g.n % 128 || g.k % S32_BK;
    if (!p.a_mc && p.b_mc) return launch_split32_layout<false, true>(g, edge);
    if (!p.a_mc && !p.b_mc) return launch_split32_layout<false, false>(g, edge);
    if (p.a_mc && p.b_mc) return launch_split32_layout<true, true>(g, edge);
    return launch_split32_layout<true, false>(g, edge);
}

}  // namespace rp
