// Stride-1 "same" convolutions of 16-bit tensors straight from the image: no zero-bordered copy, no lowered matrix.
//
//   conv_taps16_kernel   out[n, c, p] = sum over taps and input channels of wt[c][tap][ci] . in[n, ci, p shifted by the tap]
//                        (the forward; with the weights transposed and reversed, the gradient of the input)
//   conv_dw16_kernel     dw[co, ci, tap] = sum over positions of dy[n, co, p] . x[n, ci, p shifted by the tap]
//
// Images are [n][channel][h][w].  Both kernels keep a strip of them in LDS as cells: cell (row, column) holds the channels
// of one position next to each other, with (kW - 1) / 2 zero columns on either side of a row.  A tap is then a fixed
// distance between cells, at any width and alignment of the image, and the channels of a cell are what a fragment of an
// MFMA wants next to each other.  Eight channels of four positions go through a thread's registers on the way.
#include "rp_gemm.h"

namespace rp {

template <typename T> struct cd_ops;
template <> struct cd_ops<bf16_t> {
    static __device__ __forceinline__ f32x16_t mma(s16x8_t a, s16x8_t b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    // two sums -> two bf16 in one word: adding 0x8000 carries into bit 16 exactly when the first dropped bit is set
    static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
        return __builtin_amdgcn_perm(__float_as_uint(hi) + 0x8000u, __float_as_uint(lo) + 0x8000u, 0x07060302u);
    }
    static __device__ __forceinline__ float low(uint32_t w) { return __uint_as_float(w << 16); }
    static __device__ __forceinline__ float high(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
};
template <> struct cd_ops<f16_t> {
    static __device__ __forceinline__ f32x16_t mma(s16x8_t a, s16x8_t b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack(float lo, float hi) { return (uint32_t)narrow_f16_bits(lo) | ((uint32_t)narrow_f16_bits(hi) << 16); }
    static __device__ __forceinline__ float low(uint32_t w) { f16_t x; x.bits = (uint16_t)w; return widen(x); }
    static __device__ __forceinline__ float high(uint32_t w) { f16_t x; x.bits = (uint16_t)(w >> 16); return widen(x); }
};

// Neighbouring positions of one channel, fetched as one group: eight or four that begin at a multiple of as many in a row
// (VW = 8, 4: 16 or 8 bytes, aligned), or any four of a plane (VW = 0).  In the last case the plane may begin at any element: the
// aligned words that hold the four are fetched (a load that begins between two words takes more than twice as long)
// and shifted into place; near the end of the plane of HW >= 4 positions the four last ones are, and what lies past it is zero.
// A load instruction takes a CU some 26 cycles however much of it is useful, so the widest one that fits is taken.
template <int VW> struct Group { using type = u32x2_t; static constexpr int N = 4; };
template <> struct Group<8> { using type = u32x4_t; static constexpr int N = 8; };
struct GroupPlace { int at; uint32_t past; };                // first position fetched, and bits to shift it down by
template <int VW>
__device__ __forceinline__ GroupPlace place_group(int p, int HW) {
    if (VW) return {p, 0u};
    const int at = p < HW - 4 ? p : HW - 4;
    return {at, 16u * (uint32_t)(p - at)};
}
template <int VW>
__device__ __forceinline__ typename Group<VW>::type load_group(const uint16_t* plane, GroupPlace f) {
    if constexpr (VW != 0) {
        return *(const typename Group<VW>::type*)(plane + f.at);
    } else {
        typedef uint32_t __attribute__((ext_vector_type(2), aligned(4))) words_t;
        const uintptr_t a = (uintptr_t)(plane + f.at);
        const uint32_t* q = (const uint32_t*)(a & ~(uintptr_t)3);
        const words_t w = *(const words_t*)q;
        uint32_t third = 0u;
        if (a & 2) third = q[2];                             // holds the last of the four
        const uint32_t sh = (uint32_t)(a & 2) * 8u;
        const uint64_t v = (uint64_t)__builtin_amdgcn_alignbit(w[1], w[0], sh) | (uint64_t)__builtin_amdgcn_alignbit(third, w[1], sh) << 32;
        return __builtin_bit_cast(u32x2_t, f.past < 64u ? v >> f.past : 0ull);
    }
}

// Position I of a group of eight channels, as the 16 bytes a cell holds
template <int I, typename V>
__device__ __forceinline__ u32x4_t gather_position(const V (&v)[8]) {
    constexpr uint32_t sel = I % 2 ? 0x07060302u : 0x05040100u;          // both high or both low halves
    u32x4_t c;
#pragma unroll
    for (int d = 0; d < 4; d++) c[d] = __builtin_amdgcn_perm(v[2 * d + 1][I / 2], v[2 * d][I / 2], sel);
    return c;
}

// Blocks that read the same part of an image go to one XCD side by side, and so do neighbouring parts: block b runs on XCD b % 8,
// every XCD owns a run of consecutive parts, and a part's `shared` blocks follow each other.  False: nothing left to do.
__device__ __forceinline__ bool shared_block(int block, int parts, int shared, int& part, int& which) {
    const int per = (parts + 7) / 8, slot = block / 8;
    part = block % 8 * per + slot / shared;
    which = slot % shared;
    return slot / shared < per && part < parts;
}
static unsigned shared_grid(int parts, int shared) { return 8u * (unsigned)((parts + 7) / 8) * (unsigned)shared; }

// ---- weights: [C_out][C_in][tap] -> [C_from / 32][tap][C_to][32], for the input gradient transposed and the taps reversed ----
struct ConvSort {
    uint16_t* wt;
    const uint16_t* w;
    int C_from, C_to, taps, total, for_input_grad;
    int first, blocks;                           // of CD_SORT values, beside other work: the first of these blocks, and how many (0: none)
};
constexpr int CD_SORT = 2048;
__device__ __forceinline__ uint16_t weight_by_tap(const ConvSort& s, int i) {
    const int row = i / 32, to = row % s.C_to, tap = row / s.C_to % s.taps, from = row / (s.C_to * s.taps) * 32 + i % 32;
    return s.for_input_grad ? s.w[((size_t)from * s.C_to + to) * s.taps + s.taps - 1 - tap] : s.w[((size_t)to * s.C_from + from) * s.taps + tap];
}
__global__ void __launch_bounds__(256) conv_weights_by_tap_kernel(ConvSort s) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < s.total) s.wt[i] = weight_by_tap(s, i);
}

// ---- weight gradient, second half ----
struct ConvFinish {
    void* dw;
    const float* part;                           // [split][tap][C_out][C_in]
    int splits, channels, taps;
    int first, blocks;                           // beside other work: the first of these blocks, and how many (0: none)
};
// dw[co][ci][tap] = sum over the splits, in their order (four runs of them side by side, then the runs in order), rounded once;
// 64 V neighbouring sums for 256 threads
template <typename T, int V>
__device__ __forceinline__ void conv_dw_finish(const ConvFinish& f, int unit, float (*runs)[64 * V]) {
    typedef float __attribute__((ext_vector_type(V))) sums_t;
    const int total = f.channels * f.taps, lane = threadIdx.x & 63, i = (unit * 64 + lane) * V, run = threadIdx.x >> 6;
    const int per = (f.splits + 3) / 4, s0 = run * per, s1 = s0 + per < f.splits ? s0 + per : f.splits;
    sums_t sum = (sums_t)(0.f);
    if (i < total) {
        int s = s0;
        for (; s + 8 <= s1; s += 8) {
            sums_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = *(const sums_t*)(f.part + (size_t)(s + u) * total + i);
#pragma unroll
            for (int u = 0; u < 8; u++) sum += v[u];
        }
        for (; s < s1; s++) sum += *(const sums_t*)(f.part + (size_t)s * total + i);
    }
    if (run > 0) *(sums_t*)(runs[run - 1] + lane * V) = sum;
    __syncthreads();
    if (run == 0 && i < total) {
#pragma unroll
        for (int r = 0; r < 3; r++) sum += *(const sums_t*)(runs[r] + lane * V);
#pragma unroll
        for (int e = 0; e < V; e++) {
            const int tap = (i + e) / f.channels, c = i + e - tap * f.channels;          // c = co * C_in + ci
            ((T*)f.dw)[(size_t)c * f.taps + tap] = narrow<T>(sum[e]);
        }
    }
}

// ---- forward / input gradient ----
constexpr int CD_CO = 64;                        // output channels of a workgroup
constexpr int CD_CK = 32;                        // input channels in LDS at a time
constexpr int CD_STRIP = 512;                    // positions of the strip, at most: one group of eight or two of four per thread
constexpr int CD_PITCH = CD_CK + 8;              // elements of a cell: 80 bytes, so 16 lanes on neighbouring cells read from all 64 banks

struct ConvTapsArgs {
    void* out;
    const void* in;
    const void* wt;
    const void* bias;
    int batch, C_from, C_to, H, W, kH;
    int positions;                               // per workgroup (at most NPOS): whole rows where that wastes little of a tile
    int cells;                                   // room for the strip with its borders
    int groups;                                  // of positions
    int by_channel;                              // wt is [C_to][C_from][tap], as the caller keeps weights (3 x 3 taps only)
    ConvFinish finish;                           // the last blocks add up a weight gradient
};

// A workgroup computes 64 channels of `positions` consecutive positions (over all samples), four waves side by side: NPOS = 256 gives
// a wave 64 positions x 64 channels, NPOS = 64 (few positions in all) 32 x 32.  Per 32 input channels the strip of the image
// goes to LDS once; the weights follow tap row by tap row through two LDS stages, the next row's being fetched while one is
// multiplied (3 x 3: all nine taps at once, ROWS = 3).  Two workgroups share a CU, so one's fetches run under the other's products;
// what bounds it is the chain of a workgroup's own phases (of 31 000 cycles at 64 channels 8 000 are products, the rest is
// issuing loads, waiting for the first of them, and the epilogue), with 23 % of the MFMA cycles used.
// us, forward, from zero-bordered planes and here: bf16 64 x 64 x 56 x 56 -> 64 3 x 3 55 / 32, 34 x 128 x 56 x 56 -> 64 58 / 30, 2 x 64 x 28 x 28 -> 64 12.8 / 6.6,
// 32 x 256 x 7 x 7 -> 256 5 x 5 83 / 45.
template <typename T, int KW, int ROWS, int VW, int NPOS>
__global__ void __launch_bounds__(256, 2) conv_taps16_kernel(ConvTapsArgs g) {
    constexpr int WN = NPOS == 256 ? 4 : 2, WM = 4 / WN;                 // waves along positions and channels
    constexpr int TP = NPOS / WN / 32, TC = CD_CO / WM / 32;             // 32 x 32 tiles of a wave
    constexpr int NW = ROWS * KW, W_STAGE = NW * CD_CO * CD_PITCH;       // taps in LDS at a time
    constexpr int OP = NPOS + 8;                                         // elements of a staged output row
    extern __shared__ __attribute__((aligned(16))) uint16_t cd_smem[];
    uint16_t* cells = cd_smem;
    uint16_t* wts = cd_smem + (size_t)g.cells * CD_PITCH;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wn = wave % WN, wm = wave / WN;
    if (g.finish.blocks > 0 && (int)blockIdx.x >= g.finish.first) {
        for (int u = (int)blockIdx.x - g.finish.first; u * 256 < g.finish.channels * g.finish.taps; u += g.finish.blocks) {
            conv_dw_finish<T, 4>(g.finish, u, (float (*)[256])cd_smem);
            __syncthreads();
        }
        return;
    }
    const int H = g.H, W = g.W, HW = H * W, total = g.batch * HW, ph = g.kH / 2, Wc = W + KW - 1, taps = g.kH * KW;
    int group, c_tile;
    if (!shared_block(blockIdx.x, g.groups, (g.C_to + CD_CO - 1) / CD_CO, group, c_tile)) return;
    const int q0 = group * g.positions, q1 = q0 + g.positions < total ? q0 + g.positions : total;
    const int co0 = c_tile * CD_CO;
    // Samples n_lo .. n_hi have rows here.  LDS holds, sample by sample, the image rows that the output rows reach.
    const int n_lo = q0 / HW, n_hi = (q1 - 1) / HW;
    const int r_first = (q0 - n_lo * HW) / W, r_last = (q1 - 1 - n_hi * HW) / W;
    const int cells_first = ((n_hi > n_lo ? H - 1 : r_last) - r_first + g.kH) * Wc, cells_whole = (H + g.kH - 1) * Wc;
    auto first_cell = [&](int s) { return s == n_lo ? -r_first * Wc : cells_first + (s - n_lo - 1) * cells_whole; };      // of sample s's output row 0, tap (0, 0)

    const T* bias = (const T*)g.bias;
    int a_at[TP];                                // this lane's positions: cell of tap (0, 0), then its octet of channels
#pragma unroll
    for (int j = 0; j < TP; j++) {
        int q = q0 + wn * (NPOS / WN) + j * 32 + (lane & 31);
        q = q < q1 ? q : q1 - 1;                 // past the end: some position that exists, whose result is not stored
        const int s = q / HW, p = q - s * HW, r = p / W;
        a_at[j] = (first_cell(s) + r * Wc + p - r * W) * CD_PITCH + (lane >> 5) * 8;
    }
    const int b_at = (wm * (CD_CO / WM) + (lane & 31)) * CD_PITCH + (lane >> 5) * 8;

    f32x16_t acc[TP][TC];
#pragma unroll
    for (int j = 0; j < TP; j++)
#pragma unroll
        for (int i = 0; i < TC; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][i][v] = 0.f;

    // weights of (channels c0 .., ROWS tap rows from kh): one 16-byte piece per thread and tap
    u32x4_t wr[NW];
    const int w_co = t >> 2, w_piece = t & 3;
    const bool w_live = co0 + w_co < g.C_to;
    const uint16_t* w_src = (const uint16_t*)g.wt + (w_live ? co0 + w_co : 0) * 32 + w_piece * 8;
    static_assert(CD_CK == 32, "the weights are sorted by 32 channels");
    // ROWS > 1: nine taps of eight channels are nine pieces either way; weights by channel are sorted on their way to LDS
    const bool by_channel = ROWS > 1 && g.by_channel;
    auto load_weights = [&](int c0, int kh) {
        if (by_channel) {
            const uint16_t* src = (const uint16_t*)g.wt + ((size_t)(w_live ? co0 + w_co : 0) * g.C_from + c0 + w_piece * 8) * NW;
#pragma unroll
            for (int i = 0; i < NW; i++) {
                wr[i] = (u32x4_t){0u, 0u, 0u, 0u};
                if (w_live) wr[i] = *(const u32x4_t*)(src + i * 8);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NW; i++) {
            wr[i] = (u32x4_t){0u, 0u, 0u, 0u};
            if (w_live) wr[i] = *(const u32x4_t*)(w_src + ((size_t)c0 * taps + (size_t)(kh * KW + i) * 32) * g.C_to);
        }
    };
    auto store_weights = [&](uint16_t* stage) {
        if (by_channel) {
            static_for<0, NW>([&](auto tapc) {
                constexpr int tap = decltype(tapc)::value;
                u32x4_t piece;
                static_for<0, 4>([&](auto dc) {
                    constexpr int d = decltype(dc)::value, lo = 2 * d * NW + tap, hi = lo + NW;          // element of channels 2d, 2d + 1
                    constexpr uint32_t sel = (uint32_t)(lo % 2 ? 0x0302 : 0x0100) | (uint32_t)(hi % 2 ? 0x0706 : 0x0504) << 16;
                    if constexpr (hi < NW * 8) piece[d] = __builtin_amdgcn_perm(wr[hi / 8][hi / 2 % 4], wr[lo / 8][lo / 2 % 4], sel);
                });
                *(u32x4_t*)(stage + (tap * CD_CO + w_co) * CD_PITCH + w_piece * 8) = piece;
            });
            return;
        }
#pragma unroll
        for (int i = 0; i < NW; i++) *(u32x4_t*)(stage + (i * CD_CO + w_co) * CD_PITCH + w_piece * 8) = wr[i];
    };

    load_weights(0, 0);

    // The strip of 32 channels: a thread's units are (octet of channels, group of neighbouring positions of a sample).  Where they are
    // fetched from and which cells they go to is the same for every 32 channels.
    constexpr int GN = Group<VW>::N, UNITS = CD_STRIP / (64 * GN), NC = VW ? 1 : 4;
    const int s_octet = t & 3;
    GroupPlace from[UNITS];
    const uint16_t* plane[UNITS];
    int cell[UNITS][NC];                         // element of the unit's octet in the cell of a position (the others follow it unless VW = 0); negative: none
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        int group = (t >> 2) + 64 * u;
        plane[u] = nullptr;
        from[u] = {0, 0u};
#pragma unroll
        for (int e = 0; e < NC; e++) cell[u][e] = -1;
        for (int s = n_lo; s <= n_hi; s++) {
            const int r_lo = s == n_lo ? r_first : 0, r_hi = s == n_hi ? r_last : H - 1;                   // output rows of this sample
            const int i_lo = r_lo - ph > 0 ? r_lo - ph : 0, i_hi = r_hi + ph < H - 1 ? r_hi + ph : H - 1;  // image rows they reach
            const int end = (i_hi + 1) * W, groups = (end - i_lo * W + GN - 1) / GN;
            if (group >= 0 && group < groups) {
                const int p = i_lo * W + group * GN;
                plane[u] = (const uint16_t*)g.in + ((size_t)s * g.C_from + s_octet * 8) * HW;
                from[u] = place_group<VW>(p, HW);
                const int cell0 = first_cell(s) + ph * Wc + KW / 2;              // of image position (0, 0)
                int r = p / W, w = p - r * W;
#pragma unroll
                for (int e = 0; e < NC; e++) {
                    if (p + e < end) cell[u][e] = (cell0 + r * Wc + w) * CD_PITCH + s_octet * 8;
                    if (++w == W) { w = 0; r++; }
                }
            }
            group -= groups;
        }
    }
    typename Group<VW>::type strip[UNITS][8];
    auto fetch_strip = [&](int c0) {
#pragma unroll
        for (int u = 0; u < UNITS; u++)
            if (cell[u][0] >= 0) {
                const uint16_t* src = plane[u] + (size_t)c0 * HW;
#pragma unroll
                for (int c = 0; c < 8; c++) strip[u][c] = load_group<VW>(src + (size_t)c * HW, from[u]);
            }
    };
    auto put_strip = [&]() {
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            if constexpr (VW != 0) {
                if (cell[u][0] >= 0)
                    static_for<0, GN>([&](auto ec) { *(u32x4_t*)(cells + cell[u][0] + decltype(ec)::value * CD_PITCH) = gather_position<decltype(ec)::value>(strip[u]); });
            } else {
                static_for<0, 4>([&](auto ec) {
                    constexpr int e = decltype(ec)::value;
                    if (cell[u][e] >= 0) *(u32x4_t*)(cells + cell[u][e]) = gather_position<e>(strip[u]);
                });
            }
        }
    };

    fetch_strip(0);
    for (int i = t; i < g.cells * (CD_PITCH / 8); i += 256) *(u32x4_t*)(cells + i * 8) = (u32x4_t){0u, 0u, 0u, 0u};     // borders stay zero
    __syncthreads();
    auto multiply = [&](const uint16_t* ws, const uint16_t* xs) {       // one tap row
#pragma unroll
        for (int kw = 0; kw < KW; kw++)
#pragma unroll
            for (int ks = 0; ks < CD_CK / 16; ks++) {
                s16x8_t a[TP], b[TC];
#pragma unroll
                for (int j = 0; j < TP; j++) a[j] = *(const s16x8_t*)(xs + a_at[j] + kw * CD_PITCH + ks * 16);
#pragma unroll
                for (int i = 0; i < TC; i++) b[i] = *(const s16x8_t*)(ws + b_at + (kw * CD_CO + i * 32) * CD_PITCH + ks * 16);
#pragma unroll
                for (int j = 0; j < TP; j++)
#pragma unroll
                    for (int i = 0; i < TC; i++) acc[j][i] = cd_ops<T>::mma(a[j], b[i], acc[j][i]);      // rows: positions, columns: channels
            }
    };
    int buf = 0;
    for (int c0 = 0; c0 < g.C_from; c0 += CD_CK) {
        const bool more = c0 + CD_CK < g.C_from;
        put_strip();
        store_weights(wts + buf * W_STAGE);
        if constexpr (ROWS > 1) {                // every tap's weights are there
            __syncthreads();
            if (more) {
                fetch_strip(c0 + CD_CK);
                load_weights(c0 + CD_CK, 0);
            }
#pragma unroll
            for (int kh = 0; kh < ROWS; kh++) multiply(wts + kh * KW * CD_CO * CD_PITCH, cells + kh * Wc * CD_PITCH);
        } else {
            if (more) fetch_strip(c0 + CD_CK);
            for (int kh = 0; kh < g.kH; kh++) {
                __syncthreads();                 // the strip and this tap row's weights are in LDS; nobody reads the other stage any more
                const bool row_left = kh + 1 < g.kH;
                if (row_left || more) load_weights(row_left ? c0 : c0 + CD_CK, row_left ? kh + 1 : 0);
                multiply(wts + buf * W_STAGE, cells + kh * Wc * CD_PITCH);
                buf ^= 1;
                if (row_left) store_weights(wts + buf * W_STAGE);
            }
        }
        __syncthreads();                         // everyone is done with the strip
    }

    // ---- epilogue: a lane holds one channel and four neighbouring positions per quad; rows of a channel leave whole ----
    uint16_t* rows = cd_smem;
    auto stage_rows = [&](auto biased) {
#pragma unroll
        for (int i = 0; i < TC; i++) {
            const int c = wm * (CD_CO / WM) + i * 32 + (lane & 31);
            const float add = decltype(biased)::value && co0 + c < g.C_to ? widen(bias[co0 + c]) : 0.f;
#pragma unroll
            for (int j = 0; j < TP; j++)
#pragma unroll
                for (int v = 0; v < 16; v += 4) {
                    u32x2_t y = {cd_ops<T>::pack(acc[j][i][v], acc[j][i][v + 1]), cd_ops<T>::pack(acc[j][i][v + 2], acc[j][i][v + 3])};
                    if constexpr (decltype(biased)::value)             // one rounding per operation
                        y = (u32x2_t){cd_ops<T>::pack(cd_ops<T>::low(y[0]) + add, cd_ops<T>::high(y[0]) + add), cd_ops<T>::pack(cd_ops<T>::low(y[1]) + add, cd_ops<T>::high(y[1]) + add)};
                    *(u32x2_t*)(rows + c * OP + wn * (NPOS / WN) + j * 32 + 2 * v + 4 * (lane >> 5)) = y;
                }
        }
    };
    if (bias) stage_rows(std::true_type{});
    else stage_rows(std::false_type{});
    __syncthreads();
    const bool wide = VW && HW % 8 == 0 && g.positions % 8 == 0 && ((uintptr_t)g.out & 15) == 0;
    for (int u = t; u < CD_CO * (NPOS / 8); u += 256) {
        const int c = u / (NPOS / 8), o = (u % (NPOS / 8)) * 8, q = q0 + o;
        if (co0 + c >= g.C_to || q >= q1) continue;
        const u32x4_t y = *(const u32x4_t*)(rows + c * OP + o);
        int s = q / HW, p = q - s * HW;
        if (wide) {                              // eight positions of one sample, 16-byte aligned
            *(u32x4_t*)((uint16_t*)g.out + ((size_t)s * g.C_to + co0 + c) * HW + p) = y;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e += VW ? 4 : 1) {
                if (q + e < q1) {
                    uint16_t* dst = (uint16_t*)g.out + ((size_t)s * g.C_to + co0 + c) * HW + p;
                    if constexpr (VW != 0) *(u32x2_t*)dst = (u32x2_t){y[e / 2], y[e / 2 + 1]};
                    else *dst = (uint16_t)(y[e / 2] >> (16 * (e % 2)));
                }
                p += VW ? 4 : 1;
                if (p >= HW) { p -= HW; s++; }
            }
        }
    }
}

// ---- weight gradient ----
constexpr int CW_POS = 128;                      // positions of a strip, at most: whole rows, each rounded up to whole fours
constexpr int CW_XP = 64 + 32;                   // elements of a cell of 64 channels: k rows of a transposing read start 16 banks apart
constexpr int CW_DP = CW_POS + 8;                // elements of a row of dy

struct ConvDwArgs {
    float* part;                                 // [split][tap][C_out][C_in]
    const void* dy;
    const void* x;
    int batch, C_in, C_out, H, W, kH;
    int rows;                                    // image rows of a strip
    int strips, per_split;                       // strips of the whole batch (over all samples), and of one split
    int c_in_tiles, splits;
    ConvSort sort;                               // the last blocks sort the weights of an input gradient
};

// A workgroup owns 64 x 64 channels of one tap row and walks the strips of its split; the sums stay in registers.  k is the
// position: dy is k-contiguous as it lies in memory; x lies in LDS as cells, read transposed.  The waves split the channels of x
// in halves and the k steps into odd and even ones (fewer fragment bytes per MFMA than a quarter of the outputs each),
// which are added at the end.  The next strip is fetched into registers while one is multiplied.  Bound by issuing loads (a load
// takes a CU 26 cycles, a strip 64 of them); the tap rows of a strip run side by side on one XCD, whose L2 then serves two of the three.
// us, from zero-bordered planes and here: bf16 64 x 64 x 56 x 56 -> 64 3 x 3 77 / 36, 32 x 256 x 7 x 7 -> 256 5 x 5 117 / 51, 4 x 128 x 56 x 56 -> 128 3 x 3 40 / 26.
template <typename T, int KW, int VW>
__global__ void __launch_bounds__(256, 2) conv_dw16_kernel(ConvDwArgs g) {
    extern __shared__ __attribute__((aligned(16))) uint16_t cd_smem[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = wave & 1, parity = wave >> 1;
    if (g.sort.blocks > 0 && (int)blockIdx.x >= g.sort.first) {
        const int first = ((int)blockIdx.x - g.sort.first) * CD_SORT + t;
#pragma unroll
        for (int i = 0; i < CD_SORT / 256; i++)
            if (first + 256 * i < g.sort.total) g.sort.wt[first + 256 * i] = weight_by_tap(g.sort, first + 256 * i);
        return;
    }
    const int H = g.H, W = g.W, HW = H * W, Wc = W + KW - 1, Wk = (W + 3) & ~3, npos = g.rows * Wk, steps = (npos + 15) / 16;
    const int cells = g.rows * Wc + KW;          // the last KW cells stay zero
    uint16_t* xs = cd_smem;
    uint16_t* ds = cd_smem + (size_t)cells * CW_XP;
    const int tiles = g.c_in_tiles * ((g.C_out + 63) / 64);
    int part, kh;                                // the tap rows of a part read the same rows of the images
    if (!shared_block(blockIdx.x, g.splits * tiles, g.kH, part, kh)) return;
    const int split = part / tiles, tile = part % tiles, co0 = (tile / g.c_in_tiles) * 64, ci0 = (tile % g.c_in_tiles) * 64;
    const int strip0 = split * g.per_split, strip1 = strip0 + g.per_split < g.strips ? strip0 + g.per_split : g.strips;
    const int all_rows = g.batch * H, shift = kh - g.kH / 2;

    // fetching x: thread = (octet of channels, group of positions of a row); fetching dy: (group, every DC-th channel)
    constexpr int GN = Group<VW>::N, DG = CW_POS / GN, DC = 256 / DG, DN = 64 / DC;
    const int x_octet = t & 7, x_pos = (t >> 3) * GN, x_row = x_pos / Wk, x_col = x_pos - x_row * Wk;
    const int d_co = t / DG, d_pos = (t % DG) * GN, d_row = d_pos / Wk, d_col = d_pos - d_row * Wk;
    const int x_cell = (x_row * Wc + x_col + KW / 2) * CW_XP + x_octet * 8;
    const int x_chan = ci0 + x_octet * 8;
    const uint64_t d_keep = W - d_col >= 4 ? ~0ull : (1ull << (16 * (W - d_col))) - 1;          // VW = 0: positions past the row's end are zeros
    using group_t = typename Group<VW>::type;
    group_t xv[8], dv[DN];
    auto fetch = [&](int strip) {
        {
            const int row = strip * g.rows + x_row, s = row / H, h = row - s * H + shift;
            const bool live = x_pos < npos && row < all_rows && h >= 0 && h < H;
            const uint16_t* plane = (const uint16_t*)g.x + ((size_t)s * g.C_in + x_chan) * HW;
            const GroupPlace f = place_group<VW>(h * W + x_col, HW);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                xv[c] = group_t{};
                if (live && x_chan + c < g.C_in) xv[c] = load_group<VW>(plane + (size_t)c * HW, f);
            }
        }
        const int row = strip * g.rows + d_row, s = row / H, h = row - s * H;
        const bool live = d_pos < npos && row < all_rows;
        const uint16_t* plane = (const uint16_t*)g.dy + ((size_t)s * g.C_out + co0 + d_co) * HW;
        const GroupPlace f = place_group<VW>(h * W + d_col, HW);
#pragma unroll
        for (int c = 0; c < DN; c++) {
            dv[c] = group_t{};
            if (live && co0 + d_co + DC * c < g.C_out) dv[c] = load_group<VW>(plane + (size_t)(DC * c) * HW, f);
        }
    };
    auto put = [&]() {
        static_for<0, GN>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            if (x_pos < npos && (VW || x_col + e < W)) *(u32x4_t*)(xs + x_cell + e * CW_XP) = gather_position<e>(xv);          // (rows outside the image: zeros)
        });
#pragma unroll
        for (int c = 0; c < DN; c++) {
            if constexpr (VW == 0) dv[c] = __builtin_bit_cast(u32x2_t, __builtin_bit_cast(uint64_t, dv[c]) & d_keep);
            *(group_t*)(ds + (d_co + DC * c) * CW_DP + d_pos) = dv[c];       // (positions past the strip: zeros)
        }
    };

    // fragments: dy rows are k-contiguous; of x, the transposing read of 16 lanes covers four k rows (cells) x 16 channels
    const int d_at = (lane & 31) * CW_DP + (lane >> 5) * 8;
    const int grp = lane >> 4, s16 = lane & 15;
    int x_at[4][2];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int p = (parity + 2 * i) * 16 + 8 * (grp >> 1) + 4 * h + (s16 >> 2), r = p / Wk, w = p - r * Wk;
            const int cell = p < npos && w < W ? r * Wc + w : cells - KW;
            x_at[i][h] = cell * CW_XP + half * 32 + 16 * (grp & 1) + 4 * (s16 & 3);
        }

    f32x16_t acc[2][KW];
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int kw = 0; kw < KW; kw++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[m][kw][v] = 0.f;

    fetch(strip0);
    for (int i = t; i < cells * (CW_XP / 8); i += 256) *(u32x4_t*)(xs + i * 8) = (u32x4_t){0u, 0u, 0u, 0u};
    for (int strip = strip0; strip < strip1; strip++) {
        __syncthreads();                         // everyone is done with the strip before
        put();
        __syncthreads();
        if (strip + 1 < strip1) fetch(strip + 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int step = parity + 2 * i;
            if (step < steps) {                  // (the same for all lanes of the wave)
                s16x8_t a[2];
#pragma unroll
                for (int m = 0; m < 2; m++) a[m] = *(const s16x8_t*)(ds + d_at + m * 32 * CW_DP + step * 16);
#pragma unroll
                for (int kw = 0; kw < KW; kw++) {
                    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(xs + x_at[i][0] + kw * CW_XP));
                    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3)))*)(xs + x_at[i][1] + kw * CW_XP));
                    const s16x8_t b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                    for (int m = 0; m < 2; m++) acc[m][kw] = cd_ops<T>::mma(a[m], b, acc[m][kw]);      // rows: channels of dy, columns: channels of x
                }
            }
        }
    }

    // odd k steps + even ones, then the split's sums leave as they are
    float* sums = (float*)cd_smem;
    const int ci = ci0 + half * 32 + (lane & 31);
#pragma unroll
    for (int m = 0; m < 2; m++) {
        __syncthreads();
        if (parity == 1) {
#pragma unroll
            for (int kw = 0; kw < KW; kw++)
#pragma unroll
                for (int v = 0; v < 16; v++) sums[((half * KW + kw) * 16 + v) * 64 + lane] = acc[m][kw][v];
        }
        __syncthreads();
        if (parity == 0) {
#pragma unroll
            for (int kw = 0; kw < KW; kw++) {
                float* dst = g.part + ((size_t)(split * g.kH + kh) * KW + kw) * g.C_out * g.C_in;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int co = co0 + m * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
                    if (co < g.C_out && ci < g.C_in) dst[(size_t)co * g.C_in + ci] = acc[m][kw][v] + sums[((half * KW + kw) * 16 + v) * 64 + lane];
                }
            }
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256) conv_dw_finish_kernel(ConvFinish f) {
    __shared__ float runs[3][64];
    conv_dw_finish<T, 1>(f, blockIdx.x, runs);
}

// ---- host side ----
static int positions_whole_rows(int npos, int W) {
    const int whole = npos / W * W;              // whole rows: fewer image rows per output row; an eighth of the tile may idle for it
    return whole * 8 >= npos * 7 ? whole : npos;
}

static long long strip_cells(int positions, int batch, int H, int W, int kH, int kW) {
    const long long hw = (long long)H * W;
    const long long rows = positions % W == 0 ? positions / W : (positions + W - 2) / W + 1;
    long long samples = hw % positions == 0 ? 1 : (positions + hw - 2) / hw + 1;
    if (samples > batch) samples = batch;
    return (rows + samples * (kH - 1)) * (W + kW - 1);
}

constexpr size_t CD_LDS = 160 * 1024;            // of a CU
static int cus_of_device() { return device_cu_count() > 0 ? device_cu_count() : 256; }
// Workgroups of the weight gradient in all, two per CU: more of them leave more partial sums to be written and added (us at 384,
// 512 and 768: 64 x 64 x 56 x 56 3 x 3 38.8 / 36.2 / 44.6, 16 x 256 x 14 x 14 35.5 / 34.9 / 48.7, 20 x 64 x 50 x 50 38.2 / 36.9 / 48.1).
static int dw_blocks() { return 2 * cus_of_device(); }

static size_t taps_smem(int npos, long long cells, int kH, int kW) {
    const int staged = kH == 3 && kW == 3 ? 9 : 2 * kW;                  // all taps once, or a tap row twice
    const size_t loop = (size_t)cells * CD_PITCH * 2 + (size_t)staged * CD_CO * CD_PITCH * 2, epi = (size_t)CD_CO * (npos + 8) * 2;
    return loop > epi ? loop : epi;
}

// Positions of a workgroup: as many as its tile has, whole rows where that wastes little, some rows fewer where two workgroups
// fit a CU then.
static int positions_per_group(int npos, int batch, int H, int W, int kH, int kW) {
    const int most = positions_whole_rows(npos, W);
    for (int p = most; p % W == 0 && p * 8 >= npos * 7; p -= W)
        if (taps_smem(npos, strip_cells(p, batch, H, W, kH, kW), kH, kW) <= CD_LDS / 2) return p;
    return most;
}

static int dw_rows(int W) { return CW_POS / ((W + 3) / 4 * 4); }

static size_t dw_smem(int W, int kW) {
    const size_t loop = ((size_t)dw_rows(W) * (W + kW - 1) + kW) * CW_XP * 2 + (size_t)64 * CW_DP * 2, sums = (size_t)2 * kW * 16 * 64 * 4;
    return loop > sums ? loop : sums;
}

// the widest group that rows of W positions of both images consist of, aligned (VW of the kernels)
static int group_width(int W, const void* a, const void* b) {
    const uintptr_t p = (uintptr_t)a | (uintptr_t)b;
    return W % 8 == 0 && (p & 15) == 0 ? 8 : (W % 4 == 0 && (p & 7) == 0 ? 4 : 0);
}

static int taps_npos(int batch, int C_to, int H, int W) {
    const long long total = (long long)batch * H * W, at256 = (total + 255) / 256 * ((C_to + CD_CO - 1) / CD_CO);
    return at256 >= cus_of_device() ? 256 : 64;
}

bool conv_taps16_takes(int batch, int C_from, int C_to, int H, int W, int kH, int kW, int dtype) {
    if (path_disabled("convdirect") || (dtype != RP_DTYPE_BFLOAT16 && dtype != RP_DTYPE_FLOAT16)) return false;
    if ((kW != 3 && kW != 5) || kH % 2 == 0 || C_from % CD_CK || C_from <= 0 || C_to <= 0 || C_to > (1 << 20)) return false;
    if ((long long)batch * H * W >= (1ll << 30) || (long long)C_from * C_to * kH * kW >= (1ll << 30)) return false;
    if ((long long)H * W < 4) return false;
    const long long total = (long long)batch * H * W;
    const int npos = taps_npos(batch, C_to, H, W), positions = positions_per_group(npos, batch, H, W, kH, kW);
    const long long cells = strip_cells(positions, batch, H, W, kH, kW), rows = cells / (W + kW - 1);
    const long long samples = W % 8 == 0 ? 0 : (positions + (long long)H * W - 2) / ((long long)H * W) + 1;       // that end inside a group
    const size_t smem = taps_smem(npos, cells, kH, kW);
    // 64 positions a workgroup, more than two rounds of the CUs: the planes are faster where the strip and the weights leave a CU one
    // workgroup at a time (5 x 5, us, here and there: 12 x 192 x 39 x 39 -> 128 96 / 72, 5 x 256 x 45 x 38 -> 256 126 / 107, 22 x 192 x 39 x 39
    // -> 64 94 / 83; two rounds 7 x 256 x 33 x 33 -> 192 83 / 95, one 4 x 256 x 38 x 38 -> 128 47 / 65), and where the strip is six and more
    // times its positions (3 x 3: 2 x 192 x 96 x 96 -> 128 45 / 31, 5 x 192 x 96 x 96 -> 64 50 / 38, 11 x 192 x 75 x 75 -> 64 85 / 73;
    // 13 x 64 x 42 x 67 -> 64 23 / 25).
    const bool many = (total + positions - 1) / positions * ((C_to + CD_CO - 1) / CD_CO) > 2 * cus_of_device();
    if (npos == 64 && many && (smem > CD_LDS / 2 || (W > 64 && C_from > 64))) return false;
    return rows * W + 7 * samples <= CD_STRIP && smem <= CD_LDS;
}

template <typename T, int KW, int ROWS, int VW, int NPOS>
static int launch_taps_t(const ConvTapsArgs& g) {
    const size_t smem = taps_smem(NPOS, g.cells, g.kH, KW);
    auto kern = conv_taps16_kernel<T, KW, ROWS, VW, NPOS>;
    if (smem > 64 * 1024 && !check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem), "hipFuncSetAttribute")) return -1;
    hipLaunchKernelGGL(kern, dim3(shared_grid(g.groups, (g.C_to + CD_CO - 1) / CD_CO) + (unsigned)g.finish.blocks), dim3(256), smem, current_stream(), g);
    return check_launch("conv_taps16_kernel") ? 0 : -1;
}

template <typename T, int KW, int ROWS>
static int launch_taps_k(const ConvTapsArgs& g, int npos, int vw) {
    if (npos == 256) return vw == 8 ? launch_taps_t<T, KW, ROWS, 8, 256>(g) : vw == 4 ? launch_taps_t<T, KW, ROWS, 4, 256>(g) : launch_taps_t<T, KW, ROWS, 0, 256>(g);
    return vw >= 4 ? launch_taps_t<T, KW, ROWS, 4, 64>(g) : launch_taps_t<T, KW, ROWS, 0, 64>(g);
}

static int launch_taps(const ConvTapsArgs& g, int npos, int kW, int dtype) {
    const bool bf = dtype == RP_DTYPE_BFLOAT16;
    const int vw = group_width(g.W, g.in, g.out);
    if (kW == 3 && g.kH == 3) return bf ? launch_taps_k<bf16_t, 3, 3>(g, npos, vw) : launch_taps_k<f16_t, 3, 3>(g, npos, vw);
    if (kW == 3) return bf ? launch_taps_k<bf16_t, 3, 1>(g, npos, vw) : launch_taps_k<f16_t, 3, 1>(g, npos, vw);
    return bf ? launch_taps_k<bf16_t, 5, 1>(g, npos, vw) : launch_taps_k<f16_t, 5, 1>(g, npos, vw);
}

static ConvTapsArgs taps_args(void* out, const void* in, const void* bias, int batch, int C_from, int C_to, int H, int W, int kH, int kW, int npos) {
    const int positions = positions_per_group(npos, batch, H, W, kH, kW), groups = (int)(((long long)batch * H * W + positions - 1) / positions);
    return ConvTapsArgs{out, in, nullptr, bias, batch, C_from, C_to, H, W, kH, positions, (int)strip_cells(positions, batch, H, W, kH, kW), groups, 0, ConvFinish{}};
}

static bool ranges_apart(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
    return (const char*)a + a_bytes <= (const char*)b || (const char*)b + b_bytes <= (const char*)a;
}

// out[batch, C_to, H, W] from in[batch, C_from, H, W] and w [C_out, C_in, kH, kW] (for_input_grad: C_from = C_out); bias per output channel or null
int launch_conv_taps16(void* out, const void* in, const void* w, const void* bias, int batch, int C_from, int C_to, int H, int W, int kH, int kW, bool for_input_grad, int dtype) {
    const int taps = kH * kW, total = C_from * C_to * taps, npos = taps_npos(batch, C_to, H, W);
    ConvTapsArgs g = taps_args(out, in, bias, batch, C_from, C_to, H, W, kH, kW, npos);
    // Workgroups that sort the weights themselves save a launch and take longer each (us, sorted by a launch and in the workgroups: 49
    // of them 11.4 / 8.9, 196 24 / 21, 784 26 / 30): as long as there is not more than one per CU.
    // An output over the weights: a workgroup reads them for every 32 channels while others already store, so they are copied first.
    const bool apart = ranges_apart(out, (size_t)batch * C_to * H * W * 2, w, (size_t)total * 2);
    g.by_channel = kH == 3 && kW == 3 && !for_input_grad && apart && ((uintptr_t)w & 15) == 0 && (long long)g.groups * ((C_to + CD_CO - 1) / CD_CO) <= cus_of_device();
    void* wt = nullptr;
    int rc = 0;
    if (!g.by_channel) {
        if (rp_hip_malloc(&wt, (size_t)total * 2) != 0) return -1;
        const ConvSort sort{(uint16_t*)wt, (const uint16_t*)w, C_from, C_to, taps, total, for_input_grad ? 1 : 0, 0, 0};
        hipLaunchKernelGGL(conv_weights_by_tap_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, current_stream(), sort);
        rc = check_launch("conv_weights_by_tap_kernel") ? 0 : -1;
    }
    g.wt = g.by_channel ? w : wt;
    if (rc == 0) rc = launch_taps(g, npos, kW, dtype);
    report_kernel(npos == 256 ? "conv_taps16_256x64" : "conv_taps16_64x64");
    if (wt) rp_hip_free(wt);                     // back to the pool while the kernels are still queued: safe for later work on this stream
    return rc;
}

bool conv_dw16_takes(int batch, int C_in, int C_out, int H, int W, int kH, int kW, int dtype) {
    if (path_disabled("convdirect") || (dtype != RP_DTYPE_BFLOAT16 && dtype != RP_DTYPE_FLOAT16)) return false;
    if ((kW != 3 && kW != 5) || kH % 2 == 0 || W > CW_POS) return false;
    if ((long long)batch * H * W >= (1ll << 30) || (long long)C_in * C_out * kH * kW >= (1ll << 28)) return false;
    // 5 x 5 taps on rows of arbitrary width: the words fetched for every tap row of every 64 x 64 channels cost more than the
    // padded planes, except for the narrowest images (us, here and there: 6 x 192 x 41 x 41 50 / 43, 21 x 64 x 18 x 18 29 / 25, 32 x 256 x 7 x 7 51 / 117)
    if (kW == 5 && W % 4 != 0 && W > 8) return false;
    // The same words make three taps a row slower than the planes where every workgroup walks several strips of many channels (3 x 3, us,
    // here and there, tiles of 64 x 64 channels times strips of the batch: 10 x 128 x 75 x 75 -> 256 6000 of them 232 / 124, 12 x 192 x 53 x 53
    // -> 256 3816 156 / 121, 9 x 256 x 33 x 33 -> 256 1584 81 / 66, 4 x 192 x 41 x 41 -> 256 984 53 / 43; 27 x 64 x 35 x 23 -> 256 756 51 / 58,
    // 31 x 192 x 15 x 15 -> 256 708 43 / 55; one tile, 64 strips and 2486, 18 / 34 and 110 / 133)
    const long long tiles = (long long)((C_in + 63) / 64) * ((C_out + 63) / 64), strips = ((long long)batch * H + dw_rows(W) - 1) / dw_rows(W);
    if (W % 4 != 0 && tiles > 1 && tiles * strips > 800) return false;
    return (long long)H * W >= 4 && dw_smem(W, kW) <= CD_LDS;
}

template <typename T, int KW, int VW>
static int launch_dw_t(const ConvDwArgs& g) {
    const size_t smem = dw_smem(g.W, KW);
    auto kern = conv_dw16_kernel<T, KW, VW>;
    if (smem > 64 * 1024 && !check_hip(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem), "hipFuncSetAttribute")) return -1;
    hipLaunchKernelGGL(kern, dim3(shared_grid(g.splits * g.c_in_tiles * ((g.C_out + 63) / 64), g.kH) + (unsigned)g.sort.blocks), dim3(256), smem, current_stream(), g);
    return check_launch("conv_dw16_kernel") ? 0 : -1;
}

static int launch_dw(const ConvDwArgs& g, int kW, int dtype) {
    const bool bf = dtype == RP_DTYPE_BFLOAT16;
    const int vw = group_width(g.W, g.dy, g.x);
    if (kW == 3) {
        if (vw == 8) return bf ? launch_dw_t<bf16_t, 3, 8>(g) : launch_dw_t<f16_t, 3, 8>(g);
        if (vw == 4) return bf ? launch_dw_t<bf16_t, 3, 4>(g) : launch_dw_t<f16_t, 3, 4>(g);
        return bf ? launch_dw_t<bf16_t, 3, 0>(g) : launch_dw_t<f16_t, 3, 0>(g);
    }
    if (vw >= 4) return bf ? launch_dw_t<bf16_t, 5, 4>(g) : launch_dw_t<f16_t, 5, 4>(g);           // (its accumulators leave no room for groups of eight)
    return bf ? launch_dw_t<bf16_t, 5, 0>(g) : launch_dw_t<f16_t, 5, 0>(g);
}

static ConvDwArgs dw_args(const void* dy, const void* x, int batch, int C_in, int C_out, int H, int W, int kH) {
    const int rows = dw_rows(W);
    const int strips = (int)(((long long)batch * H + rows - 1) / rows);
    const int tiles = ((C_in + 63) / 64) * ((C_out + 63) / 64);
    int splits = dw_blocks() / (tiles * kH);
    splits = splits < 1 ? 1 : (splits > strips ? strips : splits);
    const int per_split = (strips + splits - 1) / splits;
    splits = (strips + per_split - 1) / per_split;
    return ConvDwArgs{nullptr, dy, x, batch, C_in, C_out, H, W, kH, rows, strips, per_split, (C_in + 63) / 64, splits, ConvSort{}};
}
static size_t dw_part_bytes(const ConvDwArgs& g, int kW) { return (size_t)g.splits * g.C_in * g.C_out * g.kH * kW * sizeof(float); }

// dw [C_out, C_in, kH, kW] from dy [batch, C_out, H, W] and x [batch, C_in, H, W]
int launch_conv_dw16(void* dw, const void* dy, const void* x, int batch, int C_in, int C_out, int H, int W, int kH, int kW, int dtype) {
    ConvDwArgs g = dw_args(dy, x, batch, C_in, C_out, H, W, kH);
    void* part = nullptr;
    if (rp_hip_malloc(&part, dw_part_bytes(g, kW)) != 0) return -1;
    g.part = (float*)part;
    int rc = launch_dw(g, kW, dtype);
    if (rc == 0) {
        const ConvFinish f{dw, g.part, g.splits, C_out * C_in, kH * kW, 0, 0};
        const dim3 grid((unsigned)(((long long)f.channels * f.taps + 63) / 64));
        if (dtype == RP_DTYPE_BFLOAT16) hipLaunchKernelGGL(conv_dw_finish_kernel<bf16_t>, grid, dim3(256), 0, current_stream(), f);
        else hipLaunchKernelGGL(conv_dw_finish_kernel<f16_t>, grid, dim3(256), 0, current_stream(), f);
        rc = check_launch("conv_dw_finish_kernel") ? 0 : -1;
    }
    report_kernel("conv_dw16");
    rp_hip_free(part);
    return rc;
}

// Both gradients, each as above (the same bits), in two launches of four: the weights of dX are sorted beside the partial sums of dW, which are
// added up beside dX.  Behind one another a launch costs 4.7 us whatever it does, and both of these small ones are done before the large ones' last
// workgroups are.  us, forward, both gradients and bias gradient, four launches and two: bf16 64 x 64 x 56 x 56 -> 64 3 x 3 99.8 / 93.9, 5 x 64 x 28 x 28 -> 256
// 59.4 / 49.9, 11 x 64 x 28 x 28 -> 64 5 x 5 62.3 / 50.3, f16 14 x 64 x 14 x 14 -> 64 3 x 3 42.8 / 34.6; 53 x 128 x 38 x 38 -> 128 194.6 / 195.8.
// (The sorting blocks last: dW's leave some places of the chip's 512 free, and in front of them they took 1.4 us more.)
// Sums are added four to a thread here, not one: a workgroup holds the LDS of the one beside it, which leaves few of them on a CU.
// False: not taken (a gradient over what the other reads, or no memory for both at once).
bool launch_conv_gradients16(void* dx, void* dw, const void* dy, const void* x, const void* w, int batch, int C_in, int C_out, int H, int W, int kH, int kW, int dtype, int& rc) {
    const int taps = kH * kW, total = C_in * C_out * taps;
    const size_t w_bytes = (size_t)total * 2, hw = (size_t)H * W * 2;
    // dW is stored while dX is read from dY and stored; x is read before dX is stored
    if (!ranges_apart(dw, w_bytes, dy, (size_t)batch * C_out * hw) || !ranges_apart(dw, w_bytes, dx, (size_t)batch * C_in * hw) ||
        !ranges_apart(dx, (size_t)batch * C_in * hw, x, (size_t)batch * C_in * hw)) return false;
    ConvDwArgs gw = dw_args(dy, x, batch, C_in, C_out, H, W, kH);
    const int npos = taps_npos(batch, C_in, H, W);
    ConvTapsArgs gx = taps_args(dx, dy, nullptr, batch, C_out, C_in, H, W, kH, kW, npos);
    void *wt = nullptr, *part = nullptr;
    if (rp_hip_malloc(&part, dw_part_bytes(gw, kW)) != 0) return false;
    if (rp_hip_malloc(&wt, w_bytes) != 0) { rp_hip_free(part); return false; }
    gw.part = (float*)part;
    gw.sort = ConvSort{(uint16_t*)wt, (const uint16_t*)w, C_out, C_in, taps, total, 1, (int)shared_grid(gw.splits * gw.c_in_tiles * ((C_out + 63) / 64), kH), (total + CD_SORT - 1) / CD_SORT};
    gx.wt = wt;
    const int units = (total + 255) / 256, most = 4 * cus_of_device();          // (C_out is whole 32s: total is whole fours)
    gx.finish = ConvFinish{dw, gw.part, gw.splits, C_out * C_in, taps, (int)shared_grid(gx.groups, (C_in + CD_CO - 1) / CD_CO), units < most ? units : most};
    rc = launch_dw(gw, kW, dtype);
    if (rc == 0) rc = launch_taps(gx, npos, kW, dtype);
    report_kernel("conv_dw16", "conv_gradients16");
    rp_hip_free(part);
    rp_hip_free(wt);
    return true;
}

}  // namespace rp
