// FP64 GEMM tiles on the CDNA matrix cores (v_mfma_f64_16x16x4f64).
//
// One 16x16 tile of C = A B (row-major, A: M x K, B: K x N) per 256-thread
// block: wave w of the block accumulates the products over its quarter of K
// (a multiple of 4), 16 MFMA steps of K=4 per round with all of the round's
// operand loads issued first.  The operands of the solvers that use this
// (a few hundred rows, some MB) stay in L2, so each lane loads its
// elements straight from there: A[r0 + l%16][k + l/16] and
// B[k + l/16][c0 + l%16] for lane l.  Register v (0..3) of lane l's
// accumulator holds C[r0 + 4*v + l/16][c0 + l%16] (measured on gfx950 with a
// known-answer tile).  Elements outside the matrix
// load as 0, so partial tiles and any K are exact.  The caller adds the four
// waves' accumulators in a fixed order, so results do not depend on timing.
#pragma once
#include <hip/hip_runtime.h>

namespace pic {

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ inline v4d dgemm_tile_mfma(int M, int N, int K, const double *__restrict__ A,
                                      const double *__restrict__ B, int r0, int c0) {
    constexpr int U = 16;   // MFMA steps per round
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int kq = lane >> 4;
    const int ar = r0 + (lane & 15), bc = c0 + (lane & 15);
    const bool arow = ar < M, bcol = bc < N;
    const double *__restrict__ Ap = A + (size_t)(arow ? ar : 0) * K;
    // quarter of K for this wave, in steps of 4
    const int steps = (K + 3) / 4;
    const int per = (steps + 3) / 4;
    const int kbeg = 4 * min(steps, wv * per), kend = 4 * min(steps, (wv + 1) * per);
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = kbeg; k0 < kend; k0 += 4 * U) {
        double a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 4 * u + kq;
            const bool in = k < kend && k < K;
            a[u] = (arow && in) ? Ap[k] : 0.0;
            b[u] = (bcol && in) ? B[(size_t)k * N + bc] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
    }
    return acc;
}

// The same for a 32x32 tile: acc[2 i + j] is the 16x16 tile at row 16 i and
// column 16 j, each sum in the order of dgemm_tile_mfma.  Every operand
// element loaded serves two tiles.
__device__ inline void dgemm_tile_mfma2(int M, int N, int K, const double *__restrict__ A,
                                        const double *__restrict__ B, int r0, int c0, v4d acc[4]) {
    constexpr int U = 8;   // MFMA steps per round
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int kq = lane >> 4;
    const int ar = r0 + (lane & 15), bc = c0 + (lane & 15);
    const bool arow0 = ar < M, arow1 = ar + 16 < M, bcol0 = bc < N, bcol1 = bc + 16 < N;
    const double *__restrict__ A0 = A + (size_t)(arow0 ? ar : 0) * K;
    const double *__restrict__ A1 = A + (size_t)(arow1 ? ar + 16 : 0) * K;
    const int steps = (K + 3) / 4;
    const int per = (steps + 3) / 4;
    const int kbeg = 4 * min(steps, wv * per), kend = 4 * min(steps, (wv + 1) * per);
#pragma unroll
    for (int h = 0; h < 4; ++h) acc[h] = v4d{0.0, 0.0, 0.0, 0.0};
    for (int k0 = kbeg; k0 < kend; k0 += 4 * U) {
        double a0[U], a1[U], b0[U], b1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 4 * u + kq;
            const bool in = k < kend && k < K;
            const double *__restrict__ Bk = B + (size_t)(in ? k : 0) * N;
            a0[u] = (arow0 && in) ? A0[k] : 0.0;
            a1[u] = (arow1 && in) ? A1[k] : 0.0;
            b0[u] = (bcol0 && in) ? Bk[bc] : 0.0;
            b1[u] = (bcol1 && in) ? Bk[bc + 16] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[u], b0[u], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[u], b1[u], acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[u], b0[u], acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[u], b1[u], acc[3], 0, 0, 0);
        }
    }
}

}  // namespace pic
