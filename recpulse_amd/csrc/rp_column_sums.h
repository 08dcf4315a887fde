// Column sums of a dense [rows, cols] matrix (the bias gradient of a Linear layer), shared by rp_hip_reduce_rows and the
// one-launch backward of small layers so that both leave the same bits.
//
// The order is fixed.  Up to 256 rows are added top to bottom in the accumulate type, the reference's own order
// (ops/ops.c:7027-7086).  More rows are cut into chunks of 256 and those into runs of 64: the rows of a run, the runs of a
// chunk and the chunks are each added top to bottom (the error bound is that of a sum of 68 + rows / 256 terms instead
// of one of rows terms, and four waves add at a time).
//
// What bounds it is not the arithmetic but how many loads are in flight: a thread that walks its column with
// sixteen loads at a time spends a memory round trip per sixteen rows (1024 x 1024 in bf16 took 23 us).  The threads
// of a workgroup therefore fetch a tile of WIDTH bytes times ROWS rows at once, 16 bytes per load and all of them in flight together,
// park it in LDS, and the rows are added out of LDS, a column per lane.
#pragma once
#include "rp_common.h"

#include <cstring>

namespace rp {

constexpr int COLSUM_CHUNK = 256, COLSUM_RUN = 64;

// PADDED: a row's gap after every run, so that lanes of different runs read different LDS banks.
template <typename T, int WIDTH, int ROWS, int THREADS = 256, bool PADDED = false>
struct ColumnTile {
    static constexpr int COLS = WIDTH / (int)sizeof(T), VEC = 16 / (int)sizeof(T);
    static constexpr int VPR = WIDTH / 16, RPP = THREADS / VPR, NV = ROWS / RPP;     // vectors per row, rows per pass of the threads, passes
    static constexpr size_t BYTES = (size_t)WIDTH * (ROWS + (PADDED ? ROWS / COLSUM_RUN : 0));
    static __device__ __forceinline__ int row_offset(int row) { return (row + (PADDED ? row / COLSUM_RUN : 0)) * COLS; }
    typedef __attribute__((ext_vector_type(4))) unsigned int vec_t;
    vec_t v[NV];
    // rows from r0 on (zeros from r1 on), columns from c0 on
    __device__ __forceinline__ void load(const T* grad, int r0, int r1, int c0, int cols, int t) {
        const int c = c0 + (t % VPR) * VEC;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int r = r0 + t / VPR + RPP * i;
            v[i] = vec_t{0, 0, 0, 0};
            if (r >= r1) continue;
            const T* p = grad + (size_t)r * cols + c;
            if (c + VEC <= cols) memcpy(&v[i], p, 16);           // at any alignment of whole elements
            else {
                T e[VEC];
                memset(e, 0, 16);
#pragma unroll
                for (int k = 0; k < VEC; k++) if (c + k < cols) e[k] = p[k];
                memcpy(&v[i], e, 16);
            }
        }
    }
    __device__ __forceinline__ void store(T* lds, int t) const {
#pragma unroll
        for (int i = 0; i < NV; i++) *(vec_t*)(lds + row_offset(t / VPR + RPP * i) + (t % VPR) * VEC) = v[i];
    }
    // s + the first n rows from lds on (of one run, if padded), top to bottom, sixteen rows read ahead of the ones being added (adding the zeros
    // past the last row changes nothing: s is never -0)
    static __device__ __forceinline__ typename traits<T>::acc add(typename traits<T>::acc s, const T* lds, int col, int n) {
        constexpr int U = 16;
        static_assert(ROWS % U == 0, "whole groups of rows");
        T x[U], next[U];
#pragma unroll
        for (int u = 0; u < U; u++) x[u] = lds[u * COLS + col];
        for (int r = 0; r < n; r += U) {
            const int ahead = r + U < n ? r + U : r;
#pragma unroll
            for (int u = 0; u < U; u++) next[u] = lds[(ahead + u) * COLS + col];
#pragma unroll
            for (int u = 0; u < U; u++) s += widen(x[u]);
#pragma unroll
            for (int u = 0; u < U; u++) x[u] = next[u];
        }
        return s;
    }
};

// Column sums of one strip of 64 bytes' worth of columns by a workgroup, in the order above: a chunk
// of 256 rows at a time in LDS, its four runs added side by side, the next chunk on its way to registers meanwhile.
struct BiasGradient {
    void* out;
    int cols, accumulate;
    int blocks;              // workgroups it takes (0: no bias gradient)
};
template <typename T, int THREADS>
struct StripSums {
    using A = typename traits<T>::acc;
    using Tile = ColumnTile<T, 64, COLSUM_CHUNK, THREADS, true>;
    static constexpr int COLS = Tile::COLS, RUNS = COLSUM_CHUNK / COLSUM_RUN;
    static constexpr size_t LDS = Tile::BYTES + RUNS * COLS * sizeof(A);
    static __device__ void run(T* out, const T* grad, int rows, int cols, int accumulate, int strip, unsigned char* lds) {
        T* tile = (T*)lds;
        A* parts = (A*)(lds + Tile::BYTES);              // [run][column]
        const int t = threadIdx.x, run = t / COLS, col = t % COLS, c0 = strip * COLS;
        Tile regs;
        regs.load(grad, 0, rows, c0, cols, t);
        A s = 0;
        for (int r = 0; r < rows; r += COLSUM_CHUNK) {
            regs.store(tile, t);
            __syncthreads();
            if (r + COLSUM_CHUNK < rows) regs.load(grad, r + COLSUM_CHUNK, rows, c0, cols, t);
            if (rows <= COLSUM_CHUNK) {                  // one chunk: all of its rows top to bottom
                if (t < COLS)
                    for (int q = 0; q * COLSUM_RUN < rows; q++)
                        s = Tile::add(s, tile + Tile::row_offset(q * COLSUM_RUN), col, rows - q * COLSUM_RUN < COLSUM_RUN ? rows - q * COLSUM_RUN : COLSUM_RUN);
            } else {
                if (t < RUNS * COLS) {
                    const int n = rows - r - run * COLSUM_RUN;
                    parts[t] = n > 0 ? Tile::add(0, tile + Tile::row_offset(run * COLSUM_RUN), col, n < COLSUM_RUN ? n : COLSUM_RUN) : (A)0;
                }
                __syncthreads();
                if (t < COLS) {
                    A c = parts[t];
#pragma unroll
                    for (int q = 1; q < RUNS; q++) c += parts[q * COLS + t];
                    s += c;
                }
            }
            __syncthreads();
        }
        const int j = c0 + t;
        if (t >= COLS || j >= cols) return;
        T y = narrow<T>(s);
        if (accumulate) y = narrow<T>(widen(out[j]) + widen(y));
        out[j] = y;
    }
};

}  // namespace rp
