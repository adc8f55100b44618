// The stopping rule of the separable field solve: fixed-order sums of the
// residual's per-block partials and what follows from them.
#pragma once
#include <hip/hip_runtime.h>

#include "pic_kernels.h"

namespace pic {

constexpr int RES_BLOCK = 256;   // threads per block of the kernels that form or sum residuals

// sums (a, b) over a block of BS threads with a fixed tree; every thread gets
// both.  sh: 2 * BS doubles.
template <int BS>
__device__ inline void block_sum2(double &a, double &b, double *sh) {
    const int t = threadIdx.x;
    sh[t] = a;
    sh[BS + t] = b;
    __syncthreads();
    for (int off = BS / 2; off > 0; off >>= 1) {
        if (t < off) {
            sh[t] += sh[t + off];
            sh[BS + t] += sh[BS + t + off];
        }
        __syncthreads();
    }
    a = sh[0];
    b = sh[BS];
    __syncthreads();
}

// ||r||^2 and ||b||^2 from nblk pairs of partials, by a block of RES_BLOCK threads
__device__ inline void sum_partials(const double *partials, int nblk, double &rr, double &bb, double *sh) {
    rr = bb = 0.0;
    for (int b = threadIdx.x; b < nblk; b += RES_BLOCK) {
        rr += partials[2 * b];
        bb += partials[2 * b + 1];
    }
    block_sum2<RES_BLOCK>(rr, bb, sh);
}

// what one thread does with a cycle's norms: converged (or out of cycles) ends
// the solve and writes its result, otherwise the cycle counts
__device__ inline bool spec_converged(double rr, double bb, double tol) {
    return bb > 0.0 ? rr <= tol * tol * bb : rr <= 1e-300;
}
__device__ inline void spec_decide(double rr, double bb, double tol, int last, SpecState *s, PcgResult *res) {
    const double rel = bb > 0.0 ? sqrt(rr / bb) : sqrt(rr);
    // a zero right-hand side after a non-zero one leaves the last solution's
    // rounding, which no relative test can pass
    const bool conv = spec_converged(rr, bb, tol) || (last && bb == 0.0 && rr < 1e300);
    s->rel = rel;
    if (conv || last) {
        s->done = 1;
        s->status = conv ? 0 : 1;
        res->iters = s->outer;
        res->outer = s->outer;
        res->rel_res = rel;
        res->status = s->status;
    } else {
        s->outer += 1;
    }
}

}  // namespace pic
