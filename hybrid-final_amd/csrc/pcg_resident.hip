// Field solve: Jacobi-preconditioned conjugate gradients whose vectors live
// in registers, one persistent kernel per solve.
//
// Each thread owns RPT rows of the operator: their coefficients, r, p, s = A p
// and x stay in its registers for the whole solve, and only z = M^-1 r goes to
// LDS, where the stencil reads it.  The recurrence is the one-reduction form
// of the method (Chronopoulos and Gear, 1989: w = A z gives both dot products
// of an iteration at once), so an iteration is one stencil sweep and one sum.
// It needs a symmetric operator.  The field operator is one up to the mirror
// rows of Neumann walls, which count their outer neighbour twice: with row
// weights W (2 inside, 1 on such a wall) W A is symmetric, so the dot products
// are taken with W.  The stopping rule is the plain norm.
//
// Up to 4096 unknowns one block solves alone and never leaves its CU: an
// iteration costs two block barriers.  Larger operators take a few blocks.
// They exchange the z values that other blocks' rows read (ghosts) and the
// partial sums through tagged words: a 64-bit word carries 32 bits of data
// and the exchange's number, is written with one store and is polled by its
// readers until the number is the one they wait for.  The data is its own
// flag: there is no barrier, no fence and no cache write-back, and every
// block sums all partials in the same order, so the result does not depend on
// timing.  Sweeps and sums alternate, and each kind switches between two sets
// of words: a block that writes a set again has completed a sum that every
// block joined after it had read that set.
//
// What bounds it: a chain of block barriers, a wave reduction and a division
// (one block: 1.5 us per iteration up to 2048 FP64 rows, 3.2 us at 4096, where
// two waves per SIMD walk eight rows each) and the two latencies of an
// exchange across the chip (several blocks: 3.5-3.9 us for 12 000 rows, 5.4 us
// for 65 000).  With the vectors in memory and fenced grid barriers an
// iteration took 14 us at 4095 rows and 14 us at 11 868.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "pcg_resident.h"

namespace pic {

namespace {

constexpr int NSUM = 3;   // values summed per exchange
typedef unsigned long long u64;

struct ResidentArgs {
    int N, rows;              // unknowns, rows per block
    const double *offd, *diagd, *mdiagd;   // 4N couplings, N diagonal, N its inverse
    const float *mdiagf;
    const uint16_t *lcol;     // 4N: index of the coupling's column in the block's z (own rows, then ghosts)
    const float *weight;      // N: W
    const uint8_t *pub;       // N: 1 when another block reads the row's z
    const int *ghost_start;   // per block
    const int *ghost;         // global rows of each block's ghosts
    u64 *halo;                // 2 sets x N x 2 tagged words
    u64 *part;                // 2 sets x blocks x NSUM x 2 tagged words
    ResidentState *st;
    u64 spin_limit;           // wait limit, in ticks of the 100 MHz constant clock
};

// sum over a 64-lane wave in a fixed order, result in every lane (the
// row shifts and broadcasts of the vector ALU, no LDS)
__device__ inline double wave_sum64(double v) {
#define PIC_DPP_ADD(ctrl, mask)                                                                                        \
    {                                                                                                                  \
        const long long b = __double_as_longlong(v);                                                                   \
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, ctrl, mask, 0xf, false);                                 \
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, mask, 0xf, false);                         \
        v += __longlong_as_double((long long)(((u64)(uint32_t)hi << 32) | (uint32_t)lo));                              \
    }
    PIC_DPP_ADD(0x111, 0xf)   // row_shr:1
    PIC_DPP_ADD(0x112, 0xf)   // row_shr:2
    PIC_DPP_ADD(0x114, 0xf)   // row_shr:4
    PIC_DPP_ADD(0x118, 0xf)   // row_shr:8
    PIC_DPP_ADD(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
    PIC_DPP_ADD(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef PIC_DPP_ADD
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double((long long)(((u64)(uint32_t)hi << 32) | (uint32_t)lo));
}

__device__ inline void tagged_store(u64 *w, uint32_t tag, uint32_t data) {
    __hip_atomic_store(w, ((u64)tag << 32) | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One block's view of the exchanges.  `dead` is set once a wait has run out
// of time (here or in another block, which raises st->abort): the block then
// stops waiting and leaves at the next sum.
struct Exchange {
    u64 *halo, *part;
    ResidentState *st;
    u64 spin_limit;
    uint32_t base;   // this solve's tags
    uint32_t seq = 0;
    int N, nblk;
    __device__ uint32_t tag() const { return base | (seq & 0xfffffu); }
    __device__ uint32_t half() const { return (seq >> 1) & 1; }   // sweeps and sums alternate
    __device__ bool poll(const u64 *w, uint32_t &data) const {
        const uint32_t want = tag();
        u64 v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)(v >> 32) != want) {
            const u64 t0 = __builtin_amdgcn_s_memrealtime();
            for (int n = 1;; ++n) {
                // the limit first: with a limit of zero no word may be waited for
                if (__builtin_amdgcn_s_memrealtime() - t0 >= spin_limit) {
                    __hip_atomic_store(&st->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return false;
                }
                if ((n & 63) == 0 && __hip_atomic_load(&st->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                    return false;
                v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)(v >> 32) == want) break;
            }
        }
        data = (uint32_t)v;
        return true;
    }
};

template <typename V> struct Words;
template <> struct Words<double> {
    static constexpr int n = 2;
    static __device__ uint32_t get(double v, int k) { return (uint32_t)((u64)__double_as_longlong(v) >> (32 * k)); }
};
template <> struct Words<float> {
    static constexpr int n = 1;
    static __device__ uint32_t get(float v, int) { return __float_as_uint(v); }
};

__device__ inline double fma_v(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float fma_v(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// With eight rows of doubles the registers are full: what is cheap to form
// again (unpacked addresses, weights, z) is formed at each use instead of
// being kept, which would spill (5.3 us per iteration of 4095 rows).
template <int RPT, typename T>
__device__ inline void keep_apart(T &v) {
    if (RPT == 8) asm volatile("" : "+v"(v));
}

// A block's rows of one precision: the couplings and the LDS indices of their
// columns (two to a register), in registers.  Row j of thread t is
// row0 + j * BS + t.
template <typename V, int BS, int RPT, bool GRID>
struct Rows {
    V off[RPT][4];
    uint32_t at[RPT][2];
    __device__ void load(const ResidentArgs &A, int row0, int n) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int l = j * BS + (int)threadIdx.x;
            const size_t i = (size_t)(row0 + (l < n ? l : 0));
            const uint2 c = ((const uint2 *)A.lcol)[i];
            at[j][0] = l < n ? c.x : 0u;
            at[j][1] = l < n ? c.y : 0u;
#pragma unroll
            for (int e = 0; e < 4; ++e) off[j][e] = l < n ? (V)A.offd[4 * i + e] : (V)0;
        }
    }
    // y = c + (off-diagonal part of A) z over the block's rows, z handed out
    // through LDS and, between blocks, the tagged words; c is the diagonal's
    // part (r itself where z = r / diagonal)
    __device__ void sweep(const ResidentArgs &A, Exchange &X, const uint8_t (&pub)[RPT], const V (&z)[RPT],
                          const V (&c)[RPT], V (&y)[RPT], V *zs, int row0, int n, bool &dead) {
        constexpr int W = Words<V>::n;
        u64 *set = nullptr;
        if (GRID) {
            ++X.seq;
            set = X.halo + (size_t)X.half() * X.N * 2;
        }
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int l = j * BS + (int)threadIdx.x;
            if (l < n) zs[l] = z[j];
            if (GRID && pub[j]) {
#pragma unroll
                for (int k = 0; k < W; ++k)
                    tagged_store(set + (size_t)(row0 + l) * 2 + k, X.tag(), Words<V>::get(z[j], k));
            }
        }
        if (GRID) {
            const int g0 = A.ghost_start[blockIdx.x], ng = A.ghost_start[blockIdx.x + 1] - g0;
            uint32_t *words = (uint32_t *)(zs + n);
            for (int q = threadIdx.x; q < ng * W; q += BS) {
                uint32_t d = 0;
                if (!dead && !X.poll(set + (size_t)A.ghost[g0 + q / W] * 2 + q % W, d)) dead = true;
                words[q] = d;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            uint32_t a0 = at[j][0], a1 = at[j][1];
            keep_apart<RPT>(a0);
            keep_apart<RPT>(a1);
            V s = fma_v(off[j][0], zs[a0 & 0xffffu], c[j]);
            s = fma_v(off[j][1], zs[a0 >> 16], s);
            s = fma_v(off[j][2], zs[a1 & 0xffffu], s);
            s = fma_v(off[j][3], zs[a1 >> 16], s);
            y[j] = s;
        }
    }
};

// sums v[] over all threads of all blocks, the same bits everywhere; false
// when the solve is being abandoned
template <int BS, bool GRID>
__device__ inline bool sum_all(Exchange &X, double (&v)[NSUM], double *sh, uint32_t &phase, bool dead) {
    constexpr int NW = BS / 64;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double *mine = sh + (size_t)(phase & 1) * NW * NSUM;
    ++phase;
#pragma unroll
    for (int q = 0; q < NSUM; ++q) {
        const double s = wave_sum64(v[q]);
        if (lane == 0) mine[wv * NSUM + q] = s;
    }
    __syncthreads();
    if (!GRID) {
#pragma unroll
        for (int q = 0; q < NSUM; ++q) {
            double s = mine[q];
#pragma unroll
            for (int w = 1; w < NW; ++w) s += mine[w * NSUM + q];
            v[q] = s;
        }
        return true;
    }
    ++X.seq;
    u64 *set = X.part + (size_t)X.half() * X.nblk * NSUM * 2;
    if (threadIdx.x < NSUM) {
        double s = mine[threadIdx.x];
        for (int w = 1; w < NW; ++w) s += mine[w * NSUM + threadIdx.x];
        for (int k = 0; k < 2; ++k)
            tagged_store(set + ((size_t)blockIdx.x * NSUM + threadIdx.x) * 2 + k, X.tag(), Words<double>::get(s, k));
    }
    uint32_t *got = (uint32_t *)(sh + 2 * NW * NSUM);   // blocks x NSUM doubles
    for (int q = threadIdx.x; q < X.nblk * NSUM * 2; q += BS) {
        uint32_t d = 0;
        if (!dead && !X.poll(set + q, d)) dead = true;
        got[q] = d;
    }
    if (__syncthreads_or(dead)) return false;
    const double *all = (const double *)got;
#pragma unroll
    for (int q = 0; q < NSUM; ++q) {
        double s = 0.0;
        for (int b = lane; b < X.nblk; b += 64) s += all[b * NSUM + q];
        v[q] = wave_sum64(s);
    }
    // `got` is rewritten only after the next sweep's barrier
    return true;
}

template <int BS>
__device__ inline Exchange open_exchange(const ResidentArgs &A) {
    Exchange X;
    X.halo = A.halo; X.part = A.part; X.st = A.st; X.spin_limit = A.spin_limit;
    X.base = A.st->solve << 20;
    X.N = A.N; X.nblk = (int)gridDim.x;
    return X;
}

__device__ inline void close_solve(const ResidentArgs &A, PcgResult *res, int it, int outer, double rel, int status) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        res->iters = it;
        res->outer = outer;
        res->rel_res = rel;
        res->status = status;
        A.st->solve += 1;   // every block has read it: each took part in a sum
    }
}
__device__ inline void abandon(const ResidentArgs &A, PcgResult *res) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        res->status = 3;
        A.st->solve += 1;
    }
}

// ------------------------------------------------------------ plain FP64
template <int BS, int RPT, bool GRID>
__global__ __launch_bounds__(BS) void k_resident_plain(ResidentArgs A, const double *b, double *x, double tol, int maxit,
                                                       PcgResult *res) {
    extern __shared__ double lds[];
    constexpr int NW = BS / 64;
    double *sh = lds, *zs = lds + 2 * NW * NSUM + (GRID ? (int)gridDim.x * NSUM : 0);
    const int row0 = blockIdx.x * A.rows, n = min(A.rows, A.N - row0);
    Exchange X = open_exchange<BS>(A);
    Rows<double, BS, RPT, GRID> op;
    op.load(A, row0, n);
    uint8_t pub[RPT];
    float wt[RPT];
    double md[RPT], r[RPT], z[RPT], w[RPT], p[RPT], s[RPT], xv[RPT];
    uint32_t phase = 0;
    bool dead = false;
    double bb_mine = 0.0;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int l = j * BS + (int)threadIdx.x;
        const bool in = l < n;
        pub[j] = GRID && in ? A.pub[row0 + l] : 0;
        wt[j] = in ? A.weight[row0 + l] : 0.0f;
        md[j] = in ? A.mdiagd[row0 + l] : 0.0;
        r[j] = in ? b[row0 + l] : 0.0;
        xv[j] = in ? x[row0 + l] : 0.0;
        p[j] = 0.0; s[j] = 0.0;
        z[j] = in ? A.diagd[row0 + l] * xv[j] : 0.0;
        bb_mine += r[j] * r[j];
    }
    op.sweep(A, X, pub, xv, z, w, zs, row0, n, dead);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        r[j] -= w[j];
        z[j] = md[j] * r[j];
    }
    // a sum between two sweeps: z in LDS is rewritten only after every thread has read it
    double v[NSUM] = {bb_mine, 0.0, 0.0};
    if (!sum_all<BS, GRID>(X, v, sh, phase, dead)) { abandon(A, res); return; }
    const double bb = v[0], tol2 = tol * tol * bb;
    double inv_gamma = 0.0, pq = 0.0, rr = 0.0;   // of the iteration before: 1 / (r . z), p . A p
    int it = 0, status = 0;
    if (bb == 0.0) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) xv[j] = 0.0;
    } else {
        for (;;) {
            op.sweep(A, X, pub, z, r, w, zs, row0, n, dead);
            v[0] = v[1] = v[2] = 0.0;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                float wj = wt[j];
                keep_apart<RPT>(wj);
                keep_apart<RPT>(md[j]);
                const double wz = (double)wj * (md[j] * r[j]);
                v[0] = fma_v(r[j], wz, v[0]);
                v[1] = fma_v(w[j], wz, v[1]);
                v[2] = fma_v(r[j], r[j], v[2]);
            }
            if (!sum_all<BS, GRID>(X, v, sh, phase, dead)) { abandon(A, res); return; }
            rr = v[2];
            if (rr <= tol2) break;
            if (it >= maxit) { status = 1; break; }
            const double beta = v[0] * inv_gamma;
            pq = v[1] - beta * beta * pq;
            const double alpha = pq != 0.0 ? v[0] / pq : 0.0;
            inv_gamma = v[0] != 0.0 ? 1.0 / v[0] : 0.0;
            ++it;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                keep_apart<RPT>(md[j]);
                p[j] = fma_v(beta, p[j], md[j] * r[j]);
                s[j] = fma_v(beta, s[j], w[j]);
                xv[j] = fma_v(alpha, p[j], xv[j]);
                r[j] = fma_v(-alpha, s[j], r[j]);
                z[j] = md[j] * r[j];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int l = j * BS + (int)threadIdx.x;
        if (l < n) x[row0 + l] = xv[j];
    }
    close_solve(A, res, it, 1, bb > 0.0 ? sqrt(rr / bb) : 0.0, status);
}

// ------------------------------------------------------------ FP32 inside FP64 refinement
template <int BS, int RPT, bool GRID>
__global__ __launch_bounds__(BS) void k_resident_refined(ResidentArgs A, const float *b, double *x, double tol,
                                                         double inner_tol, int maxit, PcgResult *res) {
    extern __shared__ double lds[];
    constexpr int NW = BS / 64;
    double *sh = lds, *zs = lds + 2 * NW * NSUM + (GRID ? (int)gridDim.x * NSUM : 0);
    const int row0 = blockIdx.x * A.rows, n = min(A.rows, A.N - row0);
    Exchange X = open_exchange<BS>(A);
    Rows<float, BS, RPT, GRID> op;
    op.load(A, row0, n);
    uint8_t pub[RPT];
    float md[RPT], wt[RPT];
    double xv[RPT], bv[RPT];
    uint32_t phase = 0;
    bool dead = false;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int l = j * BS + (int)threadIdx.x;
        const bool in = l < n;
        pub[j] = GRID && in ? A.pub[row0 + l] : 0;
        wt[j] = in ? A.weight[row0 + l] : 0.0f;
        md[j] = in ? A.mdiagf[row0 + l] : 0.0f;
        bv[j] = in ? (double)b[row0 + l] : 0.0;
        xv[j] = in ? x[row0 + l] : 0.0;
    }
    int it = 0, outer = 0, status = 0;
    double bb = 0.0, rr64 = 0.0;
    for (;;) {
        // FP64 residual of the current iterate
        double v[NSUM] = {0.0, 0.0, 0.0};
        float r[RPT];
        {
            double y[RPT], c[RPT];
            Rows<double, BS, RPT, GRID> op64;
            op64.load(A, row0, n);
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int l = j * BS + (int)threadIdx.x;
                c[j] = l < n ? A.diagd[row0 + l] * xv[j] : 0.0;
            }
            op64.sweep(A, X, pub, xv, c, y, zs, row0, n, dead);
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const double ri = bv[j] - y[j];
                r[j] = (float)ri;
                v[0] += ri * ri;
                v[1] += bv[j] * bv[j];
                v[2] += (double)r[j] * (double)r[j];
            }
        }
        if (!sum_all<BS, GRID>(X, v, sh, phase, dead)) { abandon(A, res); return; }
        rr64 = v[0];
        bb = v[1];
        if (bb == 0.0) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) xv[j] = 0.0;
            rr64 = 0.0;
            break;
        }
        if (rr64 <= tol * tol * bb) break;
        if (it >= maxit) { status = 1; break; }
        ++outer;
        // inner FP32 solve of A d = r from d = 0; dot products in FP64
        const double stop2 = inner_tol * inner_tol * v[2];
        float z[RPT], w[RPT], p[RPT], s[RPT], d[RPT];
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            z[j] = md[j] * r[j];
            p[j] = 0.0f; s[j] = 0.0f; d[j] = 0.0f;
        }
        double inv_gamma = 0.0, pq = 0.0;
        for (int k = 0;; ++k) {
            op.sweep(A, X, pub, z, r, w, (float *)zs, row0, n, dead);
            v[0] = v[1] = v[2] = 0.0;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const double wz = (double)(wt[j] * z[j]);   // W is a power of two: exact
                v[0] += (double)r[j] * wz;
                v[1] += (double)w[j] * wz;
                v[2] += (double)r[j] * (double)r[j];
            }
            if (!sum_all<BS, GRID>(X, v, sh, phase, dead)) { abandon(A, res); return; }
            if (k > 0 && (v[2] <= stop2 || it >= maxit)) break;
            const double beta = v[0] * inv_gamma;
            pq = v[1] - beta * beta * pq;
            const double alpha = pq != 0.0 ? v[0] / pq : 0.0;
            inv_gamma = v[0] != 0.0 ? 1.0 / v[0] : 0.0;
            ++it;
            const float af = (float)alpha, bf = (float)beta;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                p[j] = fma_v(bf, p[j], z[j]);
                s[j] = fma_v(bf, s[j], w[j]);
                d[j] = fma_v(af, p[j], d[j]);
                r[j] = fma_v(-af, s[j], r[j]);
                z[j] = md[j] * r[j];
            }
        }
#pragma unroll
        for (int j = 0; j < RPT; ++j) xv[j] += (double)d[j];
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int l = j * BS + (int)threadIdx.x;
        if (l < n) x[row0 + l] = xv[j];
    }
    close_solve(A, res, it, outer, bb > 0.0 ? sqrt(rr64 / bb) : 0.0, status);
}

__global__ void k_resident_reset(ResidentState *st) {
    if (threadIdx.x == 0) st->abort = 0;
}

template <typename T>
int put(T **dst, const std::vector<T> &v, hipStream_t s) {
    if (hipMalloc((void **)dst, std::max<size_t>(1, v.size()) * sizeof(T)) != hipSuccess) return -40;
    if (v.empty()) return 0;
    if (hipMemcpyAsync(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s) != hipSuccess) return -40;
    return hipStreamSynchronize(s) == hipSuccess ? 0 : -40;
}

}  // namespace

// Launch shape.  One block holds 512 threads x 8 rows; above that, 1024 rows
// per block while that makes at most 64 blocks (a sum reads every block's
// partials), then 2048 (the most that fits the registers beside the exchanges)
// up to half the CUs, so that two cases' solves fit the device together.  want_blocks > 0 fixes the grid (256
// threads per block); `split` asks for a grid even where one block would do.
static bool resident_shape(int N, int ncu, int want_blocks, bool split, int &bs, int &rpt, int &nblk) {
    auto fit = [&](int rows) { int r = 1; while (r * bs < rows) r *= 2; return r; };
    if (want_blocks > 0 || split) {
        bs = 256;
        const int need = (N + bs - 1) / bs;
        nblk = want_blocks > 0 ? std::min(want_blocks, need) : need;
        nblk = std::max(1, std::min(nblk, ncu));
        rpt = fit((N + nblk - 1) / nblk);
        return rpt <= 8;
    }
    bs = 512;
    if (N <= 4096) {
        nblk = 1;
        rpt = fit(N);
        return true;
    }
    for (rpt = 2; rpt <= 4; rpt *= 2) {
        nblk = (N + bs * rpt - 1) / (bs * rpt);
        if (nblk <= (rpt == 2 ? std::min(64, ncu / 2) : ncu / 2)) return true;
    }
    return false;
}

// Row weights that make W A symmetric, powers of two (see the top): spread
// from the first row of each connected part along the couplings.  False when
// the operator has none.
static bool row_weights(int N, const int *col, const double *val, std::vector<float> &w) {
    w.assign(N, 0.0f);
    std::vector<int> todo;
    for (int first = 0; first < N; ++first) {
        if (w[first] != 0.0f) continue;
        w[first] = 1.0f;
        todo.push_back(first);
        while (!todo.empty()) {
            const int i = todo.back();
            todo.pop_back();
            for (int e = 0; e < 5; ++e) {
                const int j = col[5 * (size_t)i + e];
                const double aij = val[5 * (size_t)i + e];
                if (j == i || aij == 0.0) continue;
                double aji = 0.0;
                for (int f = 0; f < 5; ++f)
                    if (col[5 * (size_t)j + f] == i) aji += val[5 * (size_t)j + f];
                if (!(aij / aji > 1e-3 && aij / aji < 1e3)) return false;
                int ex = 0;
                const double m = frexp(aij / aji, &ex);   // the ratio as m 2^ex, m in [0.5, 1)
                const double k = m < 0.75 ? 0.5 : 1.0;    // the power of two next to it
                if (fabs(m - k) > 1e-4) return false;
                const float wj = (float)ldexp((double)w[i] * k, ex);
                if (w[j] == 0.0f) {
                    w[j] = wj;
                    todo.push_back(j);
                } else if (w[j] != wj) {
                    return false;
                }
            }
        }
    }
    return true;
}

PcgResident *pcg_resident_create(int N, const int *col, const double *val, int ncu, int want_blocks, bool split, hipStream_t s, int *err) {
    *err = 0;
    int bs = 0, rpt = 0, nblk = 0;
    if (N < 1 || !resident_shape(N, ncu, want_blocks, split, bs, rpt, nblk)) return nullptr;
    std::vector<float> weight;
    if (!row_weights(N, col, val, weight)) return nullptr;
    const int rows = (N + nblk - 1) / nblk;
    nblk = (N + rows - 1) / rows;
    // columns outside a block's rows become ghosts behind its own rows
    std::vector<uint16_t> lcol(4 * (size_t)N);
    std::vector<double> off(4 * (size_t)N, 0.0), diag(N, 0.0);
    for (int i = 0; i < N; ++i)
        for (int e = 0; e < 5; ++e)
            if (col[5 * (size_t)i + e] == i) diag[i] += val[5 * (size_t)i + e];
    std::vector<uint8_t> pub(N, 0);
    std::vector<int> gstart(nblk + 1, 0), ghost;
    size_t most = 0;
    for (int b = 0; b < nblk; ++b) {
        const int r0 = b * rows, r1 = std::min(N, r0 + rows), n = r1 - r0;
        std::vector<int> g;
        for (size_t q = 5 * (size_t)r0; q < 5 * (size_t)r1; ++q)
            if (col[q] < r0 || col[q] >= r1) g.push_back(col[q]);
        std::sort(g.begin(), g.end());
        g.erase(std::unique(g.begin(), g.end()), g.end());
        if (n + g.size() > 65535) return nullptr;
        for (int i = r0; i < r1; ++i) {
            int k = 0;
            for (int e = 0; e < 5; ++e) {
                const int c = col[5 * (size_t)i + e];
                if (c == i) continue;   // the diagonal, and the padding of short rows
                if (k == 4) return nullptr;
                off[4 * (size_t)i + k] = val[5 * (size_t)i + e];
                lcol[4 * (size_t)i + k++] =
                    (uint16_t)(c >= r0 && c < r1 ? c - r0 : n + (std::lower_bound(g.begin(), g.end(), c) - g.begin()));
            }
            for (; k < 4; ++k) lcol[4 * (size_t)i + k] = (uint16_t)(i - r0);
        }
        for (int c : g) pub[c] = 1;
        ghost.insert(ghost.end(), g.begin(), g.end());
        gstart[b + 1] = (int)ghost.size();
        most = std::max(most, n + g.size());
    }
    const bool grid = nblk > 1 || bs == 256;   // the kernels with exchanges
    const size_t lds = (2 * (size_t)(bs / 64) * NSUM + (grid ? (size_t)nblk * NSUM : 0) + most) * sizeof(double);
    if (lds > 63 * 1024) return nullptr;   // more ghosts than a block's LDS takes without asking for more
    PcgResident *w = new PcgResident();
    w->N = N; w->bs = bs; w->rpt = rpt; w->nblk = nblk; w->rows = rows; w->lds = lds;
    int e = put(&w->lcol, lcol, s);
    if (!e) e = put(&w->off, off, s);
    if (!e) e = put(&w->diag, diag, s);
    if (!e) e = put(&w->weight, weight, s);
    if (!e) e = put(&w->pub, pub, s);
    if (!e) e = put(&w->ghost_start, gstart, s);
    if (!e) e = put(&w->ghost, ghost, s);
    // the words start with no solve's tags
    if (!e && grid) e = put(&w->halo, std::vector<unsigned long long>(4 * (size_t)N, 0), s);
    if (!e && grid) e = put(&w->part, std::vector<unsigned long long>(4 * (size_t)nblk * NSUM, 0), s);
    if (!e) e = put(&w->st, std::vector<ResidentState>(1, ResidentState{1u, 0u}), s);
    if (e) {
        *err = e;
        pcg_resident_destroy(w);
        return nullptr;
    }
    return w;
}

void pcg_resident_destroy(PcgResident *w) {
    if (!w) return;
    void *bufs[] = {w->lcol, w->off, w->diag, w->weight, w->pub, w->ghost_start, w->ghost, w->halo, w->part, w->st};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    delete w;
}

hipError_t pcg_resident_reset(PcgResident *w, hipStream_t s) {
    hipLaunchKernelGGL(k_resident_reset, dim3(1), dim3(64), 0, s, w->st);
    return hipGetLastError();
}

static ResidentArgs args_of(const PcgResident *w, const PcgOperator &A, unsigned long long spin_limit) {
    ResidentArgs a{};
    a.N = w->N; a.rows = w->rows;
    a.offd = w->off; a.diagd = w->diag; a.mdiagd = A.mdiagd; a.mdiagf = A.mdiagf;
    a.lcol = w->lcol; a.weight = w->weight; a.pub = w->pub; a.ghost_start = w->ghost_start; a.ghost = w->ghost;
    a.halo = w->halo; a.part = w->part; a.st = w->st;
    a.spin_limit = spin_limit;
    return a;
}

// one block needs no exchange; a grid runs the tagged one
#define PIC_RESIDENT(kernel, ...)                                                                                      \
    do {                                                                                                               \
        const dim3 g(w->nblk), t(w->bs);                                                                               \
        const bool grid = w->nblk > 1;                                                                                 \
        if (w->bs == 512) {                                                                                            \
            if (!grid && w->rpt == 1) hipLaunchKernelGGL((kernel<512, 1, false>), g, t, w->lds, s, __VA_ARGS__);   \
            else if (!grid && w->rpt == 2) hipLaunchKernelGGL((kernel<512, 2, false>), g, t, w->lds, s, __VA_ARGS__); \
            else if (!grid && w->rpt == 4) hipLaunchKernelGGL((kernel<512, 4, false>), g, t, w->lds, s, __VA_ARGS__); \
            else if (!grid) hipLaunchKernelGGL((kernel<512, 8, false>), g, t, w->lds, s, __VA_ARGS__);             \
            else if (w->rpt == 2) hipLaunchKernelGGL((kernel<512, 2, true>), g, t, w->lds, s, __VA_ARGS__);        \
            else hipLaunchKernelGGL((kernel<512, 4, true>), g, t, w->lds, s, __VA_ARGS__);                         \
        } else {                                                                                                       \
            if (w->rpt == 1) hipLaunchKernelGGL((kernel<256, 1, true>), g, t, w->lds, s, __VA_ARGS__);             \
            else if (w->rpt == 2) hipLaunchKernelGGL((kernel<256, 2, true>), g, t, w->lds, s, __VA_ARGS__);        \
            else if (w->rpt == 4) hipLaunchKernelGGL((kernel<256, 4, true>), g, t, w->lds, s, __VA_ARGS__);        \
            else hipLaunchKernelGGL((kernel<256, 8, true>), g, t, w->lds, s, __VA_ARGS__);                         \
        }                                                                                                              \
        return hipGetLastError();                                                                                      \
    } while (0)

hipError_t pcg_resident_plain(PcgResident *w, const PcgOperator &A, const double *b, double *x, double tol, int maxit,
                              unsigned long long spin_limit, PcgResult *res, hipStream_t s) {
    PIC_RESIDENT(k_resident_plain, args_of(w, A, spin_limit), b, x, tol, maxit, res);
}

hipError_t pcg_resident_refined(PcgResident *w, const PcgOperator &A, const float *b, double *x, double tol,
                                double inner_tol, int maxit, unsigned long long spin_limit, PcgResult *res,
                                hipStream_t s) {
    PIC_RESIDENT(k_resident_refined, args_of(w, A, spin_limit), b, x, tol, inner_tol, maxit, res);
}

}  // namespace pic
