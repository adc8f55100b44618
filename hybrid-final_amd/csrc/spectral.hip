// Field solve for separable operators: FP64 fast-Poisson inverse inside FP64
// iterative refinement.
//
// When the unknowns form a rectangle with uniform coefficients (every CCP
// deck with electrodes on two opposite walls), the field operator is
// A = cx Tx (x) I + I (x) cy Ty + shift I and
//     A^-1 R = Vx [ (Vx^-1 R Vy^-T) ./ (cx lx_a + cy ly_b + shift) ] Vy^T,
// i.e. four small dense products and an elementwise scale.  Each refinement
// cycle is
//     r = b - A x   (FP64 stencil, deterministic reduction of ||r||, ||b||)
//     x += A^-1 r   (FP64 products)
// and the solve stops on ||b - A x|| <= tol ||b||.  When the operator equals
// the separable model exactly, one cycle reaches ~1e-14 from any start; the
// cycle count is capped by the caller.  The launch sequence is fixed
// (graph-capturable); a solve that has converged skips the rest of it.
//
// At these sizes (n <= ~1000 per side) the solve is bound by the number of
// dependent launches (4 to 5 us each up to 128^2) and by load latency, not by
// FLOPs: each product is one launch, one 16x16 output tile per block on the
// FP64 matrix cores with K split over its 4 waves, so a 256^2 problem runs 289
// blocks of 4 waves from L2-resident operands.  The convergence test before a
// cycle is made by the first product's launch (block 0, beside its tile) and
// the one after the last cycle by later kernels of the step: a cycle is five
// launches, and the solve of an exact model with the fields that follow it
// six where separate norm, potential and field launches made ten.
#include <hip/hip_runtime.h>

#include "dgemm_mfma.h"
#include "multi.h"
#include "pic_kernels.h"
#include "spec_norm.h"

namespace pic {

namespace {

constexpr int GT = 16;   // GEMM output tile edge

// r = b - A x in FP64; per-block partial sums of r.r and b.b.  The first
// residual of a solve resets the solve state.
template <typename RB>
struct ResidJob {
    PcgOperator A;
    const RB *b;
    const double *x;
    double *r, *partials;
    SpecState *s;
    int first;
};

template <typename RB>
__device__ __forceinline__ void residual64_body(const ResidJob<RB> &J, int bx) {
    const PcgOperator &A = J.A;
    const double *x = J.x;
    SpecState *s = J.s;
    if (J.first) {
        if (bx == 0 && threadIdx.x == 0) { s->done = 0; s->outer = 0; s->rel = 0.0; s->status = 0; }
    } else if (s->done) {
        return;
    }
    __shared__ double sh[2 * RES_BLOCK];
    const int i = bx * RES_BLOCK + threadIdx.x;
    double rr = 0.0, bb = 0.0;
    if (i < A.N) {
        const int o = 5 * i;
        double ax = A.vald[o] * x[A.col[o]];
        ax += A.vald[o + 1] * x[A.col[o + 1]];
        ax += A.vald[o + 2] * x[A.col[o + 2]];
        ax += A.vald[o + 3] * x[A.col[o + 3]];
        ax += A.vald[o + 4] * x[A.col[o + 4]];
        const double bi = (double)J.b[i];
        const double ri = bi - ax;
        if (J.r) J.r[i] = ri;
        rr = ri * ri;
        bb = bi * bi;
    }
    block_sum2<RES_BLOCK>(rr, bb, sh);
    if (threadIdx.x == 0) {
        J.partials[2 * bx] = rr;
        J.partials[2 * bx + 1] = bb;
    }
}

template <typename RB>
__global__ __launch_bounds__(RES_BLOCK) void k_residual64(ResidJob<RB> J) { residual64_body<RB>(J, blockIdx.x); }
template <typename RB>
__global__ __launch_bounds__(RES_BLOCK) void k_residual64_m(const ResidJob<RB> *J, const uint32_t *map) {
    int lb;
    const ResidJob<RB> &a = multi_record(J, map, lb);
    residual64_body<RB>(a, lb);
}

// one block: the convergence decision after the last cycle (staged solves)
__global__ __launch_bounds__(RES_BLOCK) void k_spec_finalize(SpecFinal F) {
    __shared__ double sh[2 * RES_BLOCK];
    if (F.s->done) return;
    double rr, bb;
    sum_partials(F.partials, F.nblk, rr, bb, sh);
    if (threadIdx.x == 0) spec_decide(rr, bb, F.tol, 1, F.s, F.res);
}

// C = A B (row-major, A: M x K, B: K x N) in FP64 on the matrix cores
// (dgemm_tile_mfma), one 16x16 output tile per 256-thread block with K split
// over its 4 waves.  MODE 0: store; MODE 1: store C .* scale; MODE 2:
// x64 += C; MODE 3: store, and block 0 makes the cycle's convergence test.
struct GemmJob {
    int M, N, K;
    const double *A, *B;
    double *C;
    const double *scale;
    double *x64;
    SpecFinal F;
    int gx;   // blocks along x of the job's own grid
};

template <int MODE>
__device__ __forceinline__ void dgemm_body(const GemmJob &J, int bx, int by) {
    const int M = J.M, N = J.N, K = J.K;
    const double *__restrict__ A = J.A;
    const double *__restrict__ B = J.B;
    double *__restrict__ C = J.C;
    const double *__restrict__ scale = J.scale;
    double *__restrict__ x64 = J.x64;

    // MODE 3 decides in this launch; the others read what an earlier one wrote
    if (MODE != 3 && J.F.s->done) return;
    __shared__ double part[4][256];
    const int r0 = by * GT, c0 = bx * GT;
    const v4d acc = dgemm_tile_mfma(M, N, K, A, B, r0, c0);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int v = 0; v < 4; ++v) part[wv][lane * 4 + v] = acc[v];
    __syncthreads();
    // thread t adds the four waves' accumulator slot t (lane t/4, register t%4)
    const int t = threadIdx.x;
    const int l = t >> 2, v = t & 3;
    const double sum = ((part[0][t] + part[1][t]) + part[2][t]) + part[3][t];
    const int r = r0 + 4 * v + (l >> 4), c = c0 + (l & 15);
    if (r < M && c < N) {
        const size_t o = (size_t)r * N + c;
        if (MODE == 1) C[o] = sum * scale[o];
        else if (MODE == 2) x64[o] += sum;
        else C[o] = sum;
    }
    if (MODE == 3 && bx == 0 && by == 0) {
        __syncthreads();
        double rr, bb;
        sum_partials(J.F.partials, J.F.nblk, rr, bb, &part[0][0]);
        if (threadIdx.x == 0 && !J.F.s->done) spec_decide(rr, bb, J.F.tol, 0, J.F.s, J.F.res);
    }
}

template <int MODE>
__global__ __launch_bounds__(256) void k_dgemm(GemmJob J) { dgemm_body<MODE>(J, blockIdx.x, blockIdx.y); }
template <int MODE>
__global__ __launch_bounds__(256) void k_dgemm_m(const GemmJob *J, const uint32_t *map) {
    int lb;
    const GemmJob &a = multi_record(J, map, lb);
    dgemm_body<MODE>(a, lb % a.gx, lb / a.gx);
}

template <typename RB>
void launch_resid(const ResidJob<RB> &J, hipStream_t st) {
    const int nblk = (J.A.N + RES_BLOCK - 1) / RES_BLOCK;
    if (Recorder *rec = launch_recorder()) rec->add(&launch_m<ResidJob<RB>, k_residual64_m<RB>, RES_BLOCK>, J, nblk);
    else hipLaunchKernelGGL(k_residual64<RB>, dim3(nblk), dim3(RES_BLOCK), 0, st, J);
}

}  // namespace

template <typename RB>
SpecFinal spectral_solve(const PcgOperator &A, const SpecDev &sp, const RB *b, double *x, double tol, int max_cycles,
                         SpecState *state, double *partials, PcgResult *res, hipStream_t st) {
    const int nblk = (A.N + RES_BLOCK - 1) / RES_BLOCK;
    Recorder *rec = launch_recorder();
    const SpecFinal F{(const double *)partials, nblk, tol, state, res};
    for (int k = 0; k < max_cycles; ++k) {
        launch_resid<RB>(ResidJob<RB>{A, b, (const double *)x, sp.r, partials, state, k == 0}, st);
        // T1 = Vx^-1 R ; T2 = (T1 Vy^-T) .* dinv ; T1 = Vx T2 ; x += T1 Vy^T
        const dim3 g((sp.ny + GT - 1) / GT, (sp.nx + GT - 1) / GT);
        const dim3 blk(GT * GT);
        const int gx = (int)g.x;
        const GemmJob J0{sp.nx, sp.ny, sp.nx, sp.Vxi, (const double *)sp.r, sp.T1, nullptr, nullptr, F, gx};
        const GemmJob J1{sp.nx, sp.ny, sp.ny, (const double *)sp.T1, sp.VyiT, sp.T2, sp.dinv, nullptr, F, gx};
        const GemmJob J2{sp.nx, sp.ny, sp.nx, sp.Vx, (const double *)sp.T2, sp.T1, nullptr, nullptr, F, gx};
        const GemmJob J3{sp.nx, sp.ny, sp.ny, (const double *)sp.T1, sp.VyT, nullptr, nullptr, x, F, gx};
        if (rec) {
            const int nb = (int)(g.x * g.y);
            rec->add(&launch_m<GemmJob, k_dgemm_m<3>, 256>, J0, nb);
            rec->add(&launch_m<GemmJob, k_dgemm_m<1>, 256>, J1, nb);
            rec->add(&launch_m<GemmJob, k_dgemm_m<0>, 256>, J2, nb);
            rec->add(&launch_m<GemmJob, k_dgemm_m<2>, 256>, J3, nb);
        } else {
            hipLaunchKernelGGL(k_dgemm<3>, g, blk, 0, st, J0);
            hipLaunchKernelGGL(k_dgemm<1>, g, blk, 0, st, J1);
            hipLaunchKernelGGL(k_dgemm<0>, g, blk, 0, st, J2);
            hipLaunchKernelGGL(k_dgemm<2>, g, blk, 0, st, J3);
        }
    }
    return F;
}

template <typename RB>
void spectral_finish(const PcgOperator &A, const RB *b, const double *x, const SpecFinal &F, hipStream_t st) {
    launch_resid<RB>(ResidJob<RB>{A, b, x, nullptr, const_cast<double *>(F.partials), F.s, 0}, st);
    hipLaunchKernelGGL(k_spec_finalize, dim3(1), dim3(RES_BLOCK), 0, st, F);
}

#define INST(RB)                                                                                                      \
    template SpecFinal spectral_solve<RB>(const PcgOperator &, const SpecDev &, const RB *, double *, double, int,    \
                                          SpecState *, double *, PcgResult *, hipStream_t);                           \
    template void spectral_finish<RB>(const PcgOperator &, const RB *, const double *, const SpecFinal &, hipStream_t);
INST(float)
INST(double)
#undef INST

}  // namespace pic
