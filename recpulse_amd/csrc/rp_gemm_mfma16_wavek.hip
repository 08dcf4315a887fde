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

template <int TM, int TN, int NW, bool B_MC>
constexpr int wk_smem() {
    constexpr int stages = NW * wk_stage<TM, TN, B_MC>() * 2, parts = NW * TM * TN * 256 * 4;
    return stages > parts ? stages : parts;
}

template <typename T, int TM, int TN, int NW, bool B_MC>
__global__ void __launch_bounds__(64 * NW) gemm_mfma16_wavek_kernel(GemmArgs g, int tiles_m, int tiles_n) {
    constexpr int U = TM * TN == 1 ? 4 : 2, NB = B_MC ? WK_PIECE / 8 : 2 * TN;           // pieces at a time, loads of B a piece
    static_assert(!B_MC || TN == 4, "64 columns are a line");
    extern __shared__ __attribute__((aligned(16))) uint16_t wk_lds[];
    // block b runs on XCD b % 8: a run of tiles along the shorter side of the output for each XCD, whose L2 then serves what they share
    const int total = tiles_m * tiles_n, per = (total + 7) / 8, idx = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per || idx >= total) return;
    const bool tall = tiles_m > tiles_n;
    const int m0 = (tall ? idx / tiles_n : idx % tiles_m) * 16 * TM, n0 = (tall ? idx % tiles_n : idx / tiles_m) * 16 * TN;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row = lane & 15, kq = (lane >> 4) * 8;                     // of a fragment
    const int load_row = lane >> 3, load_k = (lane & 7) * 8;             // of a load: eight rows' lines of a piece
    uint16_t* const stage = wk_lds + wave * wk_stage<TM, TN, B_MC>(), *const b_stage = stage + 16 * TM * WK_PITCH;

    // rows past the end and k past the end read zeros
    const int rows_a = g.m - m0 < 16 * TM ? g.m - m0 : 16 * TM, rows_b = g.n - n0 < 16 * TN ? g.n - n0 : 16 * TN;
    const __amdgpu_buffer_rsrc_t a_rsrc = buffer_rsrc((const T*)g.A + m0 * g.a_rs, ((rows_a - 1) * g.a_rs + g.k) * 2);
    const __amdgpu_buffer_rsrc_t b_rsrc = B_MC ? buffer_rsrc((const T*)g.B + n0, ((g.k - 1) * g.b_rs + rows_b) * 2)
                                               : buffer_rsrc((const T*)g.B + n0 * g.b_cs, ((rows_b - 1) * g.b_cs + g.k) * 2);
    uint32_t a_off[2 * TM], b_off[NB];
#pragma unroll
    for (int i = 0; i < 2 * TM; i++) a_off[i] = 8 * i + load_row < rows_a ? (uint32_t)(((8 * i + load_row) * g.a_rs + load_k) * 2) : BUFFER_OOB;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const bool live = (B_MC ? load_k : 8 * j + load_row) < rows_b;
        b_off[j] = live ? (uint32_t)(((8 * j + load_row) * (B_MC ? g.b_rs : g.b_cs) + load_k) * 2) : BUFFER_OOB;
    }
    const uint32_t b_step = B_MC ? (uint32_t)g.b_rs * 2u : 2u;           // bytes from one k to the next

    f32x4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    for (int k0 = wave * WK_PIECE; k0 < g.k; k0 += NW * U * WK_PIECE) {
        u32x4_t a[U][2 * TM], b[U][NB];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int kk = k0 + u * NW * WK_PIECE;
            const bool live = kk + load_k < g.k;
#pragma unroll
            for (int i = 0; i < 2 * TM; i++) a[u][i] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, (int)(live ? a_off[i] + 2u * kk : BUFFER_OOB), 0, 0);
#pragma unroll
            for (int j = 0; j < NB; j++)                 // (k is a whole number of eights)
                b[u][j] = __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, (int)((B_MC ? kk + 8 * j < g.k : live) && b_off[j] != BUFFER_OOB ? b_off[j] + b_step * kk : BUFFER_OOB), 0, 0);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
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

    __syncthreads();                             // every wave is done with its stage
    float* const parts = (float*)wk_lds;         // [wave][tile][row][column]
    // a lane holds column `row` and rows 4 (lane / 16) .. + 3 of its tiles
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) parts[(wave * TM * TN + i * TN + j) * 256 + (4 * (lane >> 4) + v) * 16 + row] = acc[i][j][v];
    __syncthreads();
    const T* bias = (const T*)g.bias;
    for (int e = t; e < 256 * TM * TN; e += 64 * NW) {
        const int part = e / 256, in = e % 256, gm = m0 + part / TN * 16 + in / 16, gn = n0 + part % TN * 16 + in % 16;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) sum += parts[w * TM * TN * 256 + e];
        if (gm >= g.m || gn >= g.n) continue;
        T* out = (T*)g.C + gm * g.c_rs + gn * g.c_cs;
        *out = finish<T>(sum, bias != nullptr, bias ? bias[gn] : T{}, g.accumulate != 0, g.accumulate ? *out : T{});
    }
}

template <typename T, int TM, int TN, int NW, bool B_MC = false>
static int launch_wavek_t(const GemmArgs& g) {
    constexpr int smem = wk_smem<TM, TN, NW, B_MC>();
    const int tiles_m = (g.m + 16 * TM - 1) / (16 * TM), tiles_n = (g.n + 16 * TN - 1) / (16 * TN);
    auto kern = gemm_mfma16_wavek_kernel<T, TM, TN, NW, B_MC>;
    if (smem > 64 * 1024 && !check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem), "hipFuncSetAttribute")) return -1;
    hipLaunchKernelGGL(kern, dim3((unsigned)((tiles_m * tiles_n + 7) / 8 * 8)), dim3(64 * NW), smem, current_stream(), g, tiles_m, tiles_n);
    return check_launch("gemm_mfma16_wavek_kernel") ? 0 : -1;
}

template <typename T>
static int launch_wavek_type(const GemmArgs& g) {
    const long long cus = device_cu_count() > 0 ? device_cu_count() : 256;
    // B row-major: four waves where eight would leave some without a piece (us, four and eight: 7 x 608 x 152 4.9 / 5.3, 256 x 1024 x 256
    // 5.6 / 5.4; tiles of twice the rows 6.2 for 64 x 1024 x 4096, not 5.4)
    if (g.b_rs != 1) return g.k < 1024 ? launch_wavek_t<T, 1, 4, 4, true>(g) : launch_wavek_t<T, 1, 4, 8, true>(g);
    const long long m16 = (g.m + 15) / 16, n16 = (g.n + 15) / 16, m32 = (g.m + 31) / 32;
    // The smallest tile that leaves a CU one workgroup; at 16 x 16, sixteen waves where they hold all of k at once (us, 8 and 16
    // waves: 64 x 4096 x 1024 6.2 / 5.7, 64 x 1024 x 1024 4.9 / 5.2, 8 x 6144 x 1536 6.7 / 7.8; 16 x 16 and 32 x 32 tiles 300 x 1536 x 300 5.2 / 6.0 with
    // 4.8 at 32 x 16, 64 x 1024 x 4096 7.6 / 5.0)
    if (m16 * n16 <= cus) return g.k > 1024 && g.k <= 4096 ? launch_wavek_t<T, 1, 1, 16>(g) : launch_wavek_t<T, 1, 1, 8>(g);
    if (m32 * n16 <= cus) return launch_wavek_t<T, 2, 1, 8>(g);
    return launch_wavek_t<T, 2, 2, 8>(g);
}

int launch_mfma16_wavek(const GemmArgs& g, int dtype) { return dtype == RP_DTYPE_BFLOAT16 ? launch_wavek_type<bf16_t>(g) : launch_wavek_type<f16_t>(g); }

}  // namespace rp
