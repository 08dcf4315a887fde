// fp32 GEMM on 16 x 16 tiles: what four waves do, for the kernel of one product (rp_gemm_tiny.hip, which says what it is good for) and for the
// launches of all gradients of a Linear layer.
#pragma once
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

// One 16 x 16 tile of C_z (tile row tm, tile column tn) by four waves, threads 0 .. 255 of them being t; red: 3 x 256 floats of LDS of their own.
// Every wave of the workgroup comes here once.  Without `live` nothing is stored.
template <bool A_VEC, bool B_VEC>
__device__ __forceinline__ void tiny_tile(const GemmArgs& g, int z, int tm, int tn, float (*red)[256], int t, bool live = true) {
    const int lane = t & 63, wave = t >> 6;
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
    if (wave != 0 || !live) return;
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
__device__ __forceinline__ void tiny_tile_of(const GemmArgs& g, int tile, float (*red)[256], int t, bool live = true) {
    const int tiles_n = (g.n + 15) / 16;
    tiny_tile<A_VEC, B_VEC>(g, 0, tile / tiles_n, tile % tiles_n, red, t, live);
}

__device__ __forceinline__ void tiny_tile_any(const GemmArgs& g, bool a_vec, bool b_vec, int tile, float (*red)[256], int t, bool live = true) {
    if (a_vec && b_vec) tiny_tile_of<true, true>(g, tile, red, t, live);
    else if (a_vec) tiny_tile_of<true, false>(g, tile, red, t, live);
    else if (b_vec) tiny_tile_of<false, true>(g, tile, red, t, live);
    else tiny_tile_of<false, false>(g, tile, red, t, live);
}

// 16-byte loads along k need k to be the unit-stride axis; rows may start at any element
static inline bool tiny_a_vec(const GemmArgs& g) { return g.a_cs == 1; }
static inline bool tiny_b_vec(const GemmArgs& g) { return g.b_rs == 1; }

}  // namespace rp
