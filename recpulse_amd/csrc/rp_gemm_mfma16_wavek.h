// bf16 / fp16 MFMA GEMM whose waves split k: what a workgroup does, for the kernel of one product (rp_gemm_mfma16_wavek.hip, which says
// what it is good for) and for the launch of all gradients of a Linear layer (rp_gemm_mfma16_64.hip).
#pragma once
#include "rp_gemm.h"

namespace rp {

template <typename T> struct wk_mma;
template <> struct wk_mma<bf16_t> {
    static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};
template <> struct wk_mma<f16_t> {
    static __device__ __forceinline__ f32x4_t run(u32x4_t a, u32x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
};

constexpr int WK_PIECE = 64;                     // elements of k: one cache line of a row

constexpr int WK_PITCH = WK_PIECE + 8;           // elements of a row in LDS: the 16 rows of a fragment start in 16 different groups of four banks

__device__ __forceinline__ void wk_wave_order() {            // keeps the compiler from moving a wave's LDS accesses across
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// B with unit stride along n (B_MC, TN = 4: a line of every k row) lies in LDS as it is in memory and is read transposed; k rows of a
// transposing read start 16 banks apart.
constexpr int WK_BPITCH = 64 + 32;
template <int TM, int TN, bool B_MC>
constexpr int wk_stage() { return 16 * TM * WK_PITCH + (B_MC ? WK_PIECE * WK_BPITCH : 16 * TN * WK_PITCH); }       // elements

template <int TM, int TN, int NW, bool B_MC, int WAVES = NW>
constexpr int wk_smem() {
    constexpr int stages = WAVES * wk_stage<TM, TN, B_MC>() * 2, parts = NW * TM * TN * 256 * 4;
    return stages > parts ? stages : parts;
}

// `v` with its elements (16 bits each) moved down by `pull` < 8
__device__ __forceinline__ u32x4_t wk_pull_shift(u32x4_t v, int pull) {
    return __builtin_bit_cast(u32x4_t, __builtin_bit_cast(unsigned __int128, v) >> (16 * pull));
}

// Tile `block` of the schedule, by WAVES waves: k goes in NW shares, NW / WAVES of them to a wave one after the other, so
// that the bits do not depend on how many waves there are.
// RAGGED: rows of any length that start at any element.  A vector that straddles the end of its row is loaded further back, so that it ends with
// the row, and shifted into place; at least eight elements along the unit-stride axis.
template <typename T, int TM, int TN, int NW, bool B_MC, int WAVES, bool RAGGED>
__device__ __forceinline__ void gemm_mfma16_wavek_block(const GemmArgs& g, int tiles_m, int tiles_n, int block, uint16_t* wk_lds) {
    constexpr int SHARES = NW / WAVES;
    static_assert(NW % WAVES == 0, "whole shares");
    constexpr int U = TM * TN == 1 ? 4 : 2, NB = B_MC ? WK_PIECE / 8 : 2 * TN;           // pieces at a time, loads of B a piece
    static_assert(!B_MC || TN == 4, "64 columns are a line");
    // block b runs on XCD b % 8: a run of tiles along the shorter side of the output for each XCD, whose L2 then serves what they share
    const int total = tiles_m * tiles_n, per = (total + 7) / 8, idx = block % 8 * per + block / 8;
    if (block / 8 >= per || idx >= total) return;
    const bool tall = tiles_m > tiles_n;
    const int m0 = (tall ? idx / tiles_n : idx % tiles_m) * 16 * TM, n0 = (tall ? idx % tiles_n : idx / tiles_m) * 16 * TN;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row = lane & 15, kq = (lane >> 4) * 8;                     // of a fragment
    const int load_row = lane >> 3, load_k = (lane & 7) * 8;             // of a load: eight rows' lines of a piece
    uint16_t* const stage = wk_lds + wave * wk_stage<TM, TN, B_MC>(), *const b_stage = stage + 16 * TM * WK_PITCH;

    // rows past the end and k past the end read zeros
    constexpr int BACK = RAGGED && B_MC ? 16 : 0;                        // B's descriptor starts this many bytes early, for vectors moved back
    const int rows_a = g.m - m0 < 16 * TM ? g.m - m0 : 16 * TM, rows_b = g.n - n0 < 16 * TN ? g.n - n0 : 16 * TN;
    const __amdgpu_buffer_rsrc_t a_rsrc = buffer_rsrc((const T*)g.A + m0 * g.a_rs, ((rows_a - 1) * g.a_rs + g.k) * 2);
    const __amdgpu_buffer_rsrc_t b_rsrc = B_MC ? buffer_rsrc((const char*)((const T*)g.B + n0) - BACK, ((g.k - 1) * g.b_rs + rows_b) * 2 + BACK)
                                               : buffer_rsrc((const T*)g.B + n0 * g.b_cs, ((rows_b - 1) * g.b_cs + g.k) * 2);
    uint32_t a_off[2 * TM], b_off[NB];
#pragma unroll
    for (int i = 0; i < 2 * TM; i++) a_off[i] = 8 * i + load_row < rows_a ? (uint32_t)(((8 * i + load_row) * g.a_rs + load_k) * 2) : BUFFER_OOB;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const bool live = (B_MC ? load_k : 8 * j + load_row) < rows_b;
        b_off[j] = live ? (uint32_t)(((8 * j + load_row) * (B_MC ? g.b_rs : g.b_cs) + load_k) * 2) + BACK : BUFFER_OOB;
    }
    // elements that this lane's vectors stick out of the columns of a tile at the edge
    const int b_pull = RAGGED && B_MC && rows_b > load_k && rows_b - load_k < 8 ? 8 - (rows_b - load_k) : 0;
    const uint32_t b_step = B_MC ? (uint32_t)g.b_rs * 2u : 2u;           // bytes from one k to the next

    // elements that this lane's vectors of piece kk stick out of k
    auto k_pull = [&](int kk) {
        const int in = g.k - kk - load_k;
        return in > 0 && in < 8 ? 8 - in : 0;
    };
    f32x4_t sums[SHARES][TM][TN];
    auto add_up = [&](f32x4_t (&acc)[TM][TN], int share) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        for (int k0 = share * WK_PIECE; k0 < g.k; k0 += NW * U * WK_PIECE) {
            u32x4_t a[U][2 * TM], b[U][NB];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int kk = k0 + u * NW * WK_PIECE;
                const bool live = kk + load_k < g.k;
                const uint32_t back = RAGGED ? 2u * k_pull(kk) : 0u;
#pragma unroll
                for (int i = 0; i < 2 * TM; i++) a[u][i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, (int)(live && a_off[i] != BUFFER_OOB ? a_off[i] + 2u * kk - back : BUFFER_OOB), 0, 0);
#pragma unroll
                for (int j = 0; j < NB; j++)                 // (unless RAGGED, k is a whole number of eights)
                    b[u][j] = __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, (int)((B_MC ? kk + 8 * j + (RAGGED ? load_row : 0) < g.k : live) && b_off[j] != BUFFER_OOB ? b_off[j] + b_step * kk - (B_MC ? 2u * b_pull : back) : BUFFER_OOB), 0, 0);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (SHARES > 1 && k0 + u * NW * WK_PIECE >= g.k) break;          // behind k: nothing to add (a wave with one share keeps its loop without branches)
                if constexpr (RAGGED) {
                    const int kk = k0 + u * NW * WK_PIECE;
                    if (kk < g.k && kk + WK_PIECE > g.k) {               // (wave-uniform)
                        const int pull = k_pull(kk);
#pragma unroll
                        for (int i = 0; i < 2 * TM; i++) a[u][i] = wk_pull_shift(a[u][i], pull);
                        if constexpr (!B_MC)
#pragma unroll
                            for (int j = 0; j < NB; j++) b[u][j] = wk_pull_shift(b[u][j], pull);
                    }
                    if (B_MC && rows_b < 64)
#pragma unroll
                        for (int j = 0; j < NB; j++) b[u][j] = wk_pull_shift(b[u][j], b_pull);
                }
                wk_wave_order();
#pragma unroll
                for (int i = 0; i < 2 * TM; i++) *(u32x4_t*)(stage + (8 * i + load_row) * WK_PITCH + load_k) = a[u][i];
#pragma unroll
                for (int j = 0; j < NB; j++) *(u32x4_t*)(b_stage + (8 * j + load_row) * (B_MC ? WK_BPITCH : WK_PITCH) + load_k) = b[u][j];
                wk_wave_order();
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    u32x4_t fa[TM], fb[TN];
#pragma unroll
                    for (int i = 0; i < TM; i++) fa[i] = *(const u32x4_t*)(stage + (16 * i + row) * WK_PITCH + 32 * h + kq);
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        if constexpr (B_MC) {        // 16 lanes read four k rows x 16 columns; each gets its column of the four
                            uint16_t* const at = b_stage + (32 * h + kq + (row >> 2)) * WK_BPITCH + 16 * j + 4 * (row & 3);
                            const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)at);
                            const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(at + 4 * WK_BPITCH));
                            fb[j] = __builtin_bit_cast(u32x4_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                        } else {
                            fb[j] = *(const u32x4_t*)(b_stage + (16 * j + row) * WK_PITCH + 32 * h + kq);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++) acc[i][j] = wk_mma<T>::run(fa[i], fb[j], acc[i][j]);
                }
            }
        }
    };
#pragma unroll
    for (int s = 0; s < SHARES; s++) add_up(sums[s], wave + s * WAVES);

    __syncthreads();                             // every wave is done with its stage
    float* const parts = (float*)wk_lds;         // [share][tile][row][column]
    // a lane holds column `row` and rows 4 (lane / 16) .. + 3 of its tiles
#pragma unroll
    for (int s = 0; s < SHARES; s++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) parts[((wave + s * WAVES) * TM * TN + i * TN + j) * 256 + (4 * (lane >> 4) + v) * 16 + row] = sums[s][i][j][v];
    __syncthreads();
    const T* bias = (const T*)g.bias;
    for (int e = t; e < 256 * TM * TN; e += 64 * WAVES) {
        const int part = e / 256, in = e % 256, gm = m0 + part / TN * 16 + in / 16, gn = n0 + part % TN * 16 + in % 16;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) sum += parts[w * TM * TN * 256 + e];
        if (gm >= g.m || gn >= g.n) continue;
        T* out = (T*)g.C + gm * g.c_rs + gn * g.c_cs;
        *out = finish<T>(sum, bias != nullptr, bias ? bias[gn] : T{}, g.accumulate != 0, g.accumulate ? *out : T{});
    }
}

// Tiles of a product with a k-contiguous B: the smallest that leaves a CU one workgroup; at 16 x 16, sixteen waves where they hold all of k
// at once (us, 8 and 16 waves: 64 x 4096 x 1024 6.2 / 5.7, 64 x 1024 x 1024 4.9 / 5.2, 8 x 6144 x 1536 6.7 / 7.8; 16 x 16 and 32 x 32 tiles
// 300 x 1536 x 300 5.2 / 6.0 with 4.8 at 32 x 16, 64 x 1024 x 4096 7.6 / 5.0)
enum WavekTile { WK_16X16_16, WK_16X16, WK_32X16, WK_32X32 };
static inline WavekTile wavek_tile(const GemmArgs& g) {
    const long long cus = device_cu_count() > 0 ? device_cu_count() : 256;
    const long long m16 = (g.m + 15) / 16, n16 = (g.n + 15) / 16, m32 = (g.m + 31) / 32;
    if (m16 * n16 <= cus) return g.k > 1024 && g.k <= 4096 ? WK_16X16_16 : WK_16X16;
    return m32 * n16 <= cus ? WK_32X16 : WK_32X32;
}

}  // namespace rp
