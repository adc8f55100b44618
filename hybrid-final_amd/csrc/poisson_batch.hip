// Batched 5-point Poisson solves on one GPU (many independent problems of
// different sizes in one launch sequence).
//
// Problem p has nx x ny unknowns on a unit-spacing grid with each side
// Neumann (mirror) or Dirichlet (0), operator A = Tx (x) I + I (x) Ty with
// Tx, Ty the 1-D second-difference matrices (interior rows [-1 2 -1], a
// Neumann end row [2 -2], a Dirichlet end row [2 -1]); unknown (a, b) is at
// a * ny + b of the problem's block.  Every such operator is separable, so
// each problem is solved with the exact FP64 fast-Poisson inverse
//     x = Vx [ (Vx^-1 R Vy^-T) ./ (lx_a + ly_b) ] Vy^T
// (four GEMMs per problem, all problems batched into one launch each,
// closed-form eigenbases), wrapped in FP64 iterative refinement that stops
// on ||b - A x|| <= tol ||b|| per problem.  The eigenbasis inverses come from
// weighted orthogonality (T = D^-1 S with S symmetric, D = 1/2 on Neumann end
// rows), so no matrix is inverted numerically.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <mutex>
#include <cstdio>
#include <cmath>
#include <cstring>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/picmcc.h"
#include "dgemm_mfma.h"

namespace pic {
namespace {

constexpr int BT = 256;   // threads of a GEMM or residual block
constexpr int RB = BT;    // unknowns of a residual block
// blocks of a refinement cycle's launches, which loop over the work: as many
// as the card holds at once
constexpr int LATER_BLOCKS = 1024;
// GEMM output tiles are 32 x 32, which halves the operand loads per product,
// where that leaves two blocks for each of the 256 CUs and the sums are at
// least 160 long on average over the tiles; else 16 x 16, as short sums are
// bound by the blocks' latency and not by their loads.  A solve with small
// tiles against large ones, in us: 24 problems of 40..120 a side (203 large
// tiles) 106 and 105, 40 of 48..150 (427) 102 and 113, 64 of 48..224 (1060, sums
// of 118) 153 and 158, 60 of 130 (1342) 155 and 162, 60 of 185 (2160) 278 and
// 245, 20 of 335 (2420) 458 and 355, 2 of 620 (761) 316 and 241, 1 of 900
// (841) 437 and 361.
constexpr int LARGE_TILES = 512, LARGE_SUM = 160;

struct GemmTask {          // one output tile of one problem's GEMM
    int prob, r0, c0, pad;
};
struct ProbDev {           // device view of one problem
    int nx, ny;
    long long off;         // offset of its unknowns in the flat vectors
    int bc[4];             // left(a=0), right(a=nx-1), bottom(b=0), top(b=ny-1): 0 Neumann, 1 Dirichlet
    const double *Vx, *Vxi, *VyT, *VyiT, *dinv;
};

// A x for unknown (a, b) of problem q
__device__ inline double apply_A(const ProbDev &q, const double *x, int a, int b) {
    const double *u = x + q.off;
    const int nx = q.nx, ny = q.ny;
    const double c = u[(size_t)a * ny + b];
    double ax = 4.0 * c;
    // x direction
    if (a > 0 && a < nx - 1) ax -= u[(size_t)(a - 1) * ny + b] + u[(size_t)(a + 1) * ny + b];
    else if (nx == 1) ax -= (q.bc[0] == 0 ? c : 0.0) + (q.bc[1] == 0 ? c : 0.0);
    else if (a == 0) ax -= (q.bc[0] == 0 ? 2.0 : 1.0) * u[(size_t)1 * ny + b];
    else ax -= (q.bc[1] == 0 ? 2.0 : 1.0) * u[(size_t)(nx - 2) * ny + b];
    // y direction
    if (b > 0 && b < ny - 1) ax -= u[(size_t)a * ny + b - 1] + u[(size_t)a * ny + b + 1];
    else if (ny == 1) ax -= (q.bc[2] == 0 ? c : 0.0) + (q.bc[3] == 0 ? c : 0.0);
    else if (b == 0) ax -= (q.bc[2] == 0 ? 2.0 : 1.0) * u[(size_t)a * ny + 1];
    else ax -= (q.bc[3] == 0 ? 2.0 : 1.0) * u[(size_t)a * ny + ny - 2];
    return ax;
}

// sum of v over the block's 4 waves (every thread of wave 0 gets it), fixed order
__device__ inline double block_sum(double v, double *sh) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return v;
}

// r = b - A x per block of one problem; per-block partial sums of r.r, b.b.
// FIRST: the solve's start, x = 0 with r = b, read in place by the first
// product, so only the sums and the zeros are written.  Bound by launch and
// memory latency (7 MB: 8 us with an LDS tree over the block, 6 with shuffles).
template <bool FIRST>
__global__ __launch_bounds__(RB) void k_pb_residual(const ProbDev *P, const int2 *blocks, int nblk, const double *b,
                                                    double *x, double *r, double *part, const int *done, int *left,
                                                    int nprob) {
    if (FIRST) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *left = nprob;
    } else if (*left == 0) {
        return;
    }
    __shared__ double sh[BT / 64];
    for (int k = blockIdx.x; k < nblk; k += gridDim.x) {   // one pass if FIRST
        const int2 bl = blocks[k];   // (problem, first unknown of the block within the problem)
        if (!FIRST && done[bl.x]) continue;
        const ProbDev q = P[bl.x];
        double rr = 0.0, bb = 0.0;
        const int i = bl.y + (int)threadIdx.x;
        if (i < q.nx * q.ny) {
            const double bi = b[q.off + i];
            double ri = bi;
            if (FIRST) {
                x[q.off + i] = 0.0;
            } else {
                ri = bi - apply_A(q, x, i / q.ny, i % q.ny);
                r[q.off + i] = ri;
            }
            rr = ri * ri;
            bb = bi * bi;
        }
        rr = block_sum(rr, sh);
        bb = block_sum(bb, sh);
        if (threadIdx.x == 0) { part[2 * k] = rr; part[2 * k + 1] = bb; }
    }
}

// done[] of a problem: 0 in work, 1 converged, 2 out of cycles
// Per problem, one wave: fixed-order sum of its blocks' partials and the
// convergence decision.  A thread a problem took 21 us for 196 partials, a
// serial chain of loads; a wave takes 3.
__global__ __launch_bounds__(64) void k_pb_finalize(const int *bstart, const double *part, double tol, int first,
                                                    int last, int *done, int *left, double *rel) {
    const int p = blockIdx.x;
    if (!first && (*left == 0 || done[p])) return;
    double rr = 0.0, bb = 0.0;
    for (int k = bstart[p] + (int)threadIdx.x; k < bstart[p + 1]; k += 64) {
        rr += part[2 * k];
        bb += part[2 * k + 1];
    }
    for (int o = 32; o > 0; o >>= 1) {
        rr += __shfl_xor(rr, o);
        bb += __shfl_xor(bb, o);
    }
    if (threadIdx.x != 0) return;
    const bool conv = bb > 0.0 ? rr <= tol * tol * bb : rr <= 1e-300;
    rel[p] = bb > 0.0 ? sqrt(rr / bb) : sqrt(rr);
    const int d = conv ? 1 : last ? 2 : 0;
    done[p] = d;
    if (d) atomicSub(left, 1);
}

// batched C = A B per problem, one tile of 16 S a side per block on the FP64
// matrix cores (dgemm_tile_mfma, K split over the block's 4 waves); MODE
// selects the operands:
// 0: T1 = Vx^-1 R, 1: T2 = (T1 Vy^-T) .* dinv, 2: T1 = Vx T2, 3: x += T1 Vy^T.
// Bound by the operand loads from L2, or by a block's chain of loads where the
// sums are short.  The first cycle's launch has a block per tile; the later
// ones, which usually find nothing left, loop over the tiles from fewer blocks.
template <int MODE, int S>
__global__ __launch_bounds__(BT) void k_pb_gemm(const ProbDev *P, const GemmTask *tasks, int ntask, const double *R,
                                                double *T1, double *T2, double *x, const int *done, const int *left) {
    if (*left == 0) return;
    __shared__ double part[4][S * S * 256];
    for (int k = blockIdx.x; k < ntask; k += gridDim.x) {
        const GemmTask tk = tasks[k];
        if (done[tk.prob]) continue;   // uniform over the block
        const ProbDev q = P[tk.prob];
        const int M = q.nx, N = q.ny;
        const int K = (MODE == 0 || MODE == 2) ? q.nx : q.ny;
        const double *A = MODE == 0 ? q.Vxi : MODE == 1 ? T1 + q.off : MODE == 2 ? q.Vx : T1 + q.off;
        const double *B = MODE == 0 ? R + q.off : MODE == 1 ? q.VyiT : MODE == 2 ? T2 + q.off : q.VyT;
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        if constexpr (S == 1) {
            const v4d acc = dgemm_tile_mfma(M, N, K, A, B, tk.r0, tk.c0);
#pragma unroll
            for (int j = 0; j < 4; ++j) part[wv][lane * 4 + j] = acc[j];
        } else {
            v4d acc[4];
            dgemm_tile_mfma2(M, N, K, A, B, tk.r0, tk.c0, acc);
#pragma unroll
            for (int h = 0; h < 4; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) part[wv][h * 256 + lane * 4 + j] = acc[h][j];
        }
        __syncthreads();
        // thread t adds the four waves' accumulator slot t (lane t/4, register t%4)
        const int t = threadIdx.x, l = t >> 2;
#pragma unroll
        for (int h = 0; h < S * S; ++h) {
            const int e = h * 256 + t;
            const double v = ((part[0][e] + part[1][e]) + part[2][e]) + part[3][e];
            const int r = tk.r0 + 16 * (h / S) + 4 * (t & 3) + (l >> 4), c = tk.c0 + 16 * (h % S) + (l & 15);
            if (r >= M || c >= N) continue;
            const size_t o = (size_t)q.off + (size_t)r * N + c;
            if (MODE == 0) T1[o] = v;
            else if (MODE == 1) T2[o] = v * q.dinv[(size_t)r * N + c];
            else if (MODE == 2) T1[o] = v;
            else x[o] += v;
        }
        __syncthreads();   // the slots are read before the next tile's are written
    }
}

// closed-form eigenbasis of the n x n second difference with the given ends
// (0 Neumann, 1 Dirichlet): V (columns = eigenvectors), lambda, and V^-1
// from the D-weighted orthogonality of the eigenvectors
void eigen_1d(int n, int left, int right, std::vector<double> &V, std::vector<double> &Vi, std::vector<double> &lam) {
    const double PI = 3.14159265358979323846;
    V.assign((size_t)n * n, 0.0);
    Vi.assign((size_t)n * n, 0.0);
    lam.assign(n, 0.0);
    for (int k = 0; k < n; ++k) {
        double th;
        if (left == 0 && right == 0) th = n > 1 ? PI * k / (n - 1) : 0.0;
        else if (left == 1 && right == 1) th = PI * (k + 1) / (n + 1);
        else th = PI * (2 * k + 1) / (2.0 * n);
        for (int a = 0; a < n; ++a) {
            double v;
            if (left == 0 && right == 0) v = std::cos(th * a);
            else if (left == 1 && right == 1) v = std::sin(th * (a + 1));
            else if (left == 0) v = std::cos(th * a);
            else v = std::cos(th * (n - 1 - a));
            V[(size_t)a * n + k] = v;
        }
        lam[k] = 2.0 - 2.0 * std::cos(th);
        if (n == 1) lam[k] = (left == 0 ? 0.0 : 1.0) + (right == 0 ? 0.0 : 1.0);
    }
    // weights: 1/2 on a Neumann end row (n > 1), 1 elsewhere
    std::vector<double> w(n, 1.0);
    if (n > 1) {
        if (left == 0) w[0] = 0.5;
        if (right == 0) w[n - 1] = 0.5;
    }
    for (int k = 0; k < n; ++k) {
        double d = 0.0;
        for (int a = 0; a < n; ++a) d += w[a] * V[(size_t)a * n + k] * V[(size_t)a * n + k];
        for (int a = 0; a < n; ++a) Vi[(size_t)k * n + a] = w[a] * V[(size_t)a * n + k] / d;
    }
}

}  // namespace
}  // namespace pic

using namespace pic;

struct pic_pbatch {
    int nprob = 0;
    long long N = 0;
    int dev = 0;
    hipStream_t st = nullptr;
    std::vector<ProbDev> host;
    std::vector<long long> offs;
    ProbDev *P = nullptr;
    GemmTask *tasks = nullptr;
    int ntask = 0, tile = 16;
    int2 *blocks = nullptr;
    int nblk = 0;
    int *bstart = nullptr;
    double *b = nullptr, *x = nullptr, *r = nullptr, *T1 = nullptr, *T2 = nullptr, *part = nullptr, *rel = nullptr;
    int *done = nullptr, *left = nullptr;   // left: problems still in work
    std::vector<void *> owned;
    std::string err;
};

static thread_local std::string g_pb_err;

#define PBCHK(x)                                                                                                       \
    do {                                                                                                               \
        hipError_t e_ = (x);                                                                                           \
        if (e_ != hipSuccess) {                                                                                        \
            g_pb_err = std::string("HIP error: ") + hipGetErrorString(e_) + " at " #x;                                \
            return -1;                                                                                                 \
        }                                                                                                              \
    } while (0)

template <typename T>
static hipError_t pb_upload(pic_pbatch *B, T **p, const std::vector<T> &v) {
    hipError_t e = hipMalloc((void **)p, std::max<size_t>(1, v.size()) * sizeof(T));
    if (e != hipSuccess) return e;
    B->owned.push_back(*p);
    if (v.empty()) return hipSuccess;
    e = hipMemcpyAsync(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, B->st);
    if (e == hipSuccess) e = hipStreamSynchronize(B->st);
    return e;
}
template <typename T>
static hipError_t pb_alloc(pic_pbatch *B, T **p, size_t n) {
    hipError_t e = hipMalloc((void **)p, std::max<size_t>(1, n) * sizeof(T));
    if (e == hipSuccess) B->owned.push_back(*p);
    return e;
}

static int pb_destroy(pic_pbatch *B) {
    if (!B) return 0;
    if (B->st) {
        const hipError_t e = hipStreamSynchronize(B->st);
        if (e != hipSuccess) fprintf(stderr, "picmcc: Poisson batch teardown: %s\n", hipGetErrorString(e));
    }
    for (void *p : B->owned) (void)hipFree(p);
    if (B->st) (void)hipStreamDestroy(B->st);
    delete B;
    return 0;
}

// Host-side tables of a batch: the problems, their GEMM tiles and residual
// blocks, and the matrices each problem reads (eigenbases shared between
// problems with the same size and ends, and each problem's 1/(lx + ly)).
// ProbDev's matrix pointers are filled by bind() once the matrices are on
// the device.
struct PbPlan {
    std::vector<ProbDev> probs;
    std::vector<std::vector<double>> mats;
    std::vector<std::array<int, 5>> refs;   // per problem: Vx, Vxi, VyT, VyiT, dinv (indices into mats)
    std::vector<GemmTask> tasks;
    std::vector<int2> blocks;
    std::vector<int> bstart;
    int tile = 16;
    long long N = 0;
    void bind(const std::vector<const double *> &dev) {
        for (size_t p = 0; p < probs.size(); ++p) {
            probs[p].Vx = dev[refs[p][0]];
            probs[p].Vxi = dev[refs[p][1]];
            probs[p].VyT = dev[refs[p][2]];
            probs[p].VyiT = dev[refs[p][3]];
            probs[p].dinv = dev[refs[p][4]];
        }
    }
};

static int pb_plan(int nprob, const int *nx, const int *ny, const int *bc, PbPlan &pl) {
    if (nprob <= 0 || !nx || !ny || !bc) { g_pb_err = "invalid arguments"; return -2; }
    for (int p = 0; p < nprob; ++p) {
        if (nx[p] < 1 || ny[p] < 1) { g_pb_err = "problem sizes must be positive"; return -2; }
        const int *c = bc + 4 * p;
        for (int s = 0; s < 4; ++s)
            if (c[s] != 0 && c[s] != 1) { g_pb_err = "boundary codes are 0 (Neumann) or 1 (Dirichlet)"; return -2; }
        if (!(c[0] || c[1] || c[2] || c[3])) { g_pb_err = "a pure Neumann problem is singular"; return -2; }
    }
    std::map<std::tuple<int, int, int, int>, std::pair<int, int>> cache;   // (axis, n, ends) -> (V, Vi)
    auto basis = [&](int axis, int n, int l, int r, int &iv, int &ivi, std::vector<double> &lam) {
        std::vector<double> v, vi;
        eigen_1d(n, l, r, v, vi, lam);
        const auto key = std::make_tuple(axis, n, l, r);
        const auto it = cache.find(key);
        if (it != cache.end()) { iv = it->second.first; ivi = it->second.second; return; }
        if (axis == 1) {   // the y bases are used as V^T and (V^-1)^T
            std::vector<double> vt((size_t)n * n), vit((size_t)n * n);
            for (int i = 0; i < n; ++i)
                for (int j = 0; j < n; ++j) { vt[(size_t)i * n + j] = v[(size_t)j * n + i]; vit[(size_t)i * n + j] = vi[(size_t)j * n + i]; }
            v.swap(vt);
            vi.swap(vit);
        }
        iv = (int)pl.mats.size();
        pl.mats.push_back(std::move(v));
        ivi = (int)pl.mats.size();
        pl.mats.push_back(std::move(vi));
        cache[key] = {iv, ivi};
    };
    long long large = 0, sums = 0;
    for (int p = 0; p < nprob; ++p) {
        const long long t = (long long)((nx[p] + 31) / 32) * ((ny[p] + 31) / 32);
        large += t;
        sums += t * (((long long)nx[p] + ny[p]) / 2);
    }
    pl.tile = large >= LARGE_TILES && sums >= LARGE_SUM * large ? 32 : 16;
    long long off = 0;
    pl.bstart.assign(nprob + 1, 0);
    for (int p = 0; p < nprob; ++p) {
        ProbDev q{};
        q.nx = nx[p]; q.ny = ny[p]; q.off = off;
        for (int s = 0; s < 4; ++s) q.bc[s] = bc[4 * p + s];
        std::vector<double> lx, ly;
        std::array<int, 5> ref{};
        basis(0, q.nx, q.bc[0], q.bc[1], ref[0], ref[1], lx);
        basis(1, q.ny, q.bc[2], q.bc[3], ref[2], ref[3], ly);
        std::vector<double> dinv((size_t)q.nx * q.ny);
        for (int a = 0; a < q.nx; ++a)
            for (int c = 0; c < q.ny; ++c) {
                const double d = lx[a] + ly[c];
                dinv[(size_t)a * q.ny + c] = d > 1e-300 ? 1.0 / d : 0.0;
            }
        ref[4] = (int)pl.mats.size();
        pl.mats.push_back(std::move(dinv));
        for (int r0 = 0; r0 < q.nx; r0 += pl.tile)
            for (int c0 = 0; c0 < q.ny; c0 += pl.tile) pl.tasks.push_back(GemmTask{p, r0, c0, 0});
        pl.bstart[p] = (int)pl.blocks.size();
        for (int i0 = 0; i0 < q.nx * q.ny; i0 += RB) pl.blocks.push_back(make_int2(p, i0));
        pl.probs.push_back(q);
        pl.refs.push_back(ref);
        off += (long long)q.nx * q.ny;
    }
    pl.bstart[nprob] = (int)pl.blocks.size();
    pl.N = off;
    return 0;
}

// Work space of pic_pbatch_solve_noalloc: one array per device, reached
// from host code only through the address hipGetSymbolAddress returns for
// the current device (the symbol's name is not a device address on the
// host).  Every call on a device shares it.
constexpr size_t PB_SCRATCH_BYTES = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[PB_SCRATCH_BYTES];
constexpr int PB_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[PB_MAX_DEVICES];

// address of this device's scratch array (looked up once per device)
static int pb_scratch(int device, unsigned char **out) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            g_pb_err = std::string("cannot locate the solver work space: ") + hipGetErrorString(e);
            return -1;
        }
        g_scratch_ptr[device] = ptr;
    }
    *out = (unsigned char *)g_scratch_ptr[device];
    return 0;
}

// The launch sequence of one batched solve from x = 0: residual and
// convergence test per cycle, then the four GEMMs of the fast inverse on the
// problems not yet converged.  B supplies the problem tables and work
// vectors; b and x are the right-hand sides and the solution.
static void pb_enqueue(const pic_pbatch &B, const double *b, double *x, double tol, int max_cycles, hipStream_t st) {
    const ProbDev *P = B.P;
    const dim3 blk(BT);
    auto product = [&](auto kern, const double *R, int grid) {
        hipLaunchKernelGGL(kern, dim3(grid), blk, 0, st, P, (const GemmTask *)B.tasks, B.ntask, R, B.T1, B.T2, x,
                           (const int *)B.done, (const int *)B.left);
    };
    for (int k = 0; k <= max_cycles; ++k) {
        const double *R = k == 0 ? b : B.r;
        if (k == 0)
            hipLaunchKernelGGL(k_pb_residual<true>, dim3(B.nblk), blk, 0, st, P, (const int2 *)B.blocks, B.nblk, b, x,
                               B.r, B.part, (const int *)B.done, B.left, B.nprob);
        else
            hipLaunchKernelGGL(k_pb_residual<false>, dim3(std::min(B.nblk, 2 * LATER_BLOCKS)), blk, 0, st, P,
                               (const int2 *)B.blocks, B.nblk, b, x, B.r, B.part, (const int *)B.done, B.left, B.nprob);
        hipLaunchKernelGGL(k_pb_finalize, dim3(B.nprob), dim3(64), 0, st, (const int *)B.bstart,
                           (const double *)B.part, tol, k == 0 ? 1 : 0, k == max_cycles ? 1 : 0, B.done, B.left, B.rel);
        if (k == max_cycles) break;
        const int grid = k == 0 ? B.ntask : std::min(B.ntask, LATER_BLOCKS);
        if (B.tile == 32) {
            product(k_pb_gemm<0, 2>, R, grid);
            product(k_pb_gemm<1, 2>, R, grid);
            product(k_pb_gemm<2, 2>, R, grid);
            product(k_pb_gemm<3, 2>, R, grid);
        } else {
            product(k_pb_gemm<0, 1>, R, grid);
            product(k_pb_gemm<1, 1>, R, grid);
            product(k_pb_gemm<2, 1>, R, grid);
            product(k_pb_gemm<3, 1>, R, grid);
        }
    }
}

extern "C" {

const char *pic_pbatch_last_error(void) { return g_pb_err.c_str(); }

int pic_pbatch_create(int nprob, const int *nx, const int *ny, const int *bc, int device, pic_pbatch **out) {
    if (!out) { g_pb_err = "invalid arguments"; return -2; }
    *out = nullptr;
    PbPlan pl;
    if (const int rc = pb_plan(nprob, nx, ny, bc, pl)) return rc;
    pic_pbatch *B = new pic_pbatch();
    B->nprob = nprob;
    B->dev = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&B->st, hipStreamNonBlocking) != hipSuccess) {
        g_pb_err = "cannot open the device";
        pb_destroy(B);
        return -1;
    }
    std::vector<const double *> mdev(pl.mats.size());
    for (size_t m = 0; m < pl.mats.size(); ++m) {
        double *d;
        if (pb_upload(B, &d, pl.mats[m]) != hipSuccess) { g_pb_err = "device allocation failed"; pb_destroy(B); return -1; }
        mdev[m] = d;
    }
    pl.bind(mdev);
    B->host = pl.probs;
    B->N = pl.N;
    B->ntask = (int)pl.tasks.size();
    B->tile = pl.tile;
    B->nblk = (int)pl.blocks.size();
    if (pb_upload(B, &B->P, pl.probs) != hipSuccess || pb_upload(B, &B->tasks, pl.tasks) != hipSuccess ||
        pb_upload(B, &B->blocks, pl.blocks) != hipSuccess || pb_upload(B, &B->bstart, pl.bstart) != hipSuccess ||
        pb_alloc(B, &B->b, pl.N) != hipSuccess || pb_alloc(B, &B->x, pl.N) != hipSuccess ||
        pb_alloc(B, &B->r, pl.N) != hipSuccess || pb_alloc(B, &B->T1, pl.N) != hipSuccess ||
        pb_alloc(B, &B->T2, pl.N) != hipSuccess || pb_alloc(B, &B->part, 2 * (size_t)B->nblk) != hipSuccess ||
        pb_alloc(B, &B->rel, nprob) != hipSuccess || pb_alloc(B, &B->done, nprob) != hipSuccess ||
        pb_alloc(B, &B->left, 1) != hipSuccess) {
        g_pb_err = "device allocation failed";
        pb_destroy(B);
        return -1;
    }
    *out = B;
    return 0;
}

int pic_pbatch_destroy(pic_pbatch *B) { return pb_destroy(B); }

long long pic_pbatch_unknowns(pic_pbatch *B) { return B ? B->N : -1; }

int pic_pbatch_set_rhs(pic_pbatch *B, const double *b) {
    if (!B || !b) { g_pb_err = "invalid arguments"; return -2; }
    PBCHK(hipMemcpyAsync(B->b, b, (size_t)B->N * sizeof(double), hipMemcpyHostToDevice, B->st));
    PBCHK(hipStreamSynchronize(B->st));
    return 0;
}

// Solve all problems from x = 0 with at most max_cycles refinement cycles;
// enqueued on the batch's stream (no host synchronisation).
int pic_pbatch_solve(pic_pbatch *B, double tol, int max_cycles) {
    if (!B || tol <= 0 || max_cycles < 1) { g_pb_err = "invalid arguments"; return -2; }
    pb_enqueue(*B, B->b, B->x, tol, max_cycles, B->st);
    PBCHK(hipGetLastError());
    return 0;
}

// waits for the solve; copies x (may be null), per-problem relative residuals
// (may be null) and returns the number of problems that did not converge
int pic_pbatch_result(pic_pbatch *B, double *x, double *rel_res) {
    if (!B) { g_pb_err = "invalid arguments"; return -2; }
    PBCHK(hipStreamSynchronize(B->st));
    if (x) PBCHK(hipMemcpyAsync(x, B->x, (size_t)B->N * sizeof(double), hipMemcpyDeviceToHost, B->st));
    if (rel_res) PBCHK(hipMemcpyAsync(rel_res, B->rel, (size_t)B->nprob * sizeof(double), hipMemcpyDeviceToHost, B->st));
    std::vector<int> stt(B->nprob);
    PBCHK(hipMemcpyAsync(stt.data(), B->done, (size_t)B->nprob * sizeof(int), hipMemcpyDeviceToHost, B->st));
    PBCHK(hipStreamSynchronize(B->st));
    int bad = 0;
    for (int v : stt) bad += v != 1;
    return bad;
}

int pic_pbatch_sync(pic_pbatch *B) {
    if (!B) { g_pb_err = "invalid arguments"; return -2; }
    PBCHK(hipStreamSynchronize(B->st));
    return 0;
}

// The batch of pic_pbatch_create + pic_pbatch_solve + pic_pbatch_result in
// one call that allocates no device memory: tables, eigenbases and work
// vectors are laid out in the device's scratch array (PB_SCRATCH_BYTES),
// right-hand sides and solution are the caller's device arrays.  The work
// is ordered on `stream` and the call waits for it.  Calls that overlap on
// one device race on the shared array.
int pic_pbatch_solve_noalloc(int nprob, const int *nx, const int *ny, const int *bc, int device, const double *b_dev,
                             double *x_dev, double tol, int max_cycles, double *rel_res, void *stream) {
    if (!b_dev || !x_dev || tol <= 0 || max_cycles < 1) { g_pb_err = "invalid arguments"; return -2; }
    if (device < 0 || device >= PB_MAX_DEVICES) { g_pb_err = "device ordinal out of range"; return -2; }
    PbPlan pl;
    if (const int rc = pb_plan(nprob, nx, ny, bc, pl)) return rc;
    // layout: tables first, then matrices, then the work vectors; every
    // region starts on a 256-byte boundary
    size_t at = 0;
    auto region = [&](size_t bytes) { const size_t o = at; at += (bytes + 255) & ~(size_t)255; return o; };
    const size_t oP = region(pl.probs.size() * sizeof(ProbDev));
    const size_t oT = region(pl.tasks.size() * sizeof(GemmTask));
    const size_t oB = region(pl.blocks.size() * sizeof(int2));
    const size_t oS = region(pl.bstart.size() * sizeof(int));
    std::vector<size_t> oM(pl.mats.size());
    for (size_t m = 0; m < pl.mats.size(); ++m) oM[m] = region(pl.mats[m].size() * sizeof(double));
    const size_t host_bytes = at;   // everything above is copied from the host
    const size_t oR = region((size_t)pl.N * sizeof(double));
    const size_t o1 = region((size_t)pl.N * sizeof(double));
    const size_t o2 = region((size_t)pl.N * sizeof(double));
    const size_t oPart = region(2 * pl.blocks.size() * sizeof(double));
    const size_t oRel = region((size_t)nprob * sizeof(double));
    const size_t oDone = region((size_t)nprob * sizeof(int));
    const size_t oLeft = region(sizeof(int));
    if (at > PB_SCRATCH_BYTES) {
        g_pb_err = "batch needs " + std::to_string(at) + " bytes of work space, more than the " +
                   std::to_string(PB_SCRATCH_BYTES) + " of the no-allocation solve";
        return -3;
    }
    PBCHK(hipSetDevice(device));
    unsigned char *base = nullptr;
    if (pb_scratch(device, &base)) return -1;
    std::vector<const double *> mdev(pl.mats.size());
    for (size_t m = 0; m < pl.mats.size(); ++m) mdev[m] = (const double *)(base + oM[m]);
    pl.bind(mdev);
    std::vector<unsigned char> host(host_bytes, 0);
    auto put = [&](size_t o, const void *src, size_t n) { if (n) memcpy(host.data() + o, src, n); };
    put(oP, pl.probs.data(), pl.probs.size() * sizeof(ProbDev));
    put(oT, pl.tasks.data(), pl.tasks.size() * sizeof(GemmTask));
    put(oB, pl.blocks.data(), pl.blocks.size() * sizeof(int2));
    put(oS, pl.bstart.data(), pl.bstart.size() * sizeof(int));
    for (size_t m = 0; m < pl.mats.size(); ++m) put(oM[m], pl.mats[m].data(), pl.mats[m].size() * sizeof(double));
    const hipStream_t st = (hipStream_t)stream;
    PBCHK(hipMemcpyAsync(base, host.data(), host_bytes, hipMemcpyHostToDevice, st));
    pic_pbatch B;   // a view of the scratch layout (owns nothing)
    B.nprob = nprob;
    B.N = pl.N;
    B.dev = device;
    B.P = (ProbDev *)(base + oP);
    B.tasks = (GemmTask *)(base + oT);
    B.ntask = (int)pl.tasks.size();
    B.tile = pl.tile;
    B.blocks = (int2 *)(base + oB);
    B.nblk = (int)pl.blocks.size();
    B.bstart = (int *)(base + oS);
    B.r = (double *)(base + oR);
    B.T1 = (double *)(base + o1);
    B.T2 = (double *)(base + o2);
    B.part = (double *)(base + oPart);
    B.rel = (double *)(base + oRel);
    B.done = (int *)(base + oDone);
    B.left = (int *)(base + oLeft);
    pb_enqueue(B, b_dev, x_dev, tol, max_cycles, st);
    PBCHK(hipGetLastError());
    std::vector<int> stt(nprob);
    if (rel_res) PBCHK(hipMemcpyAsync(rel_res, B.rel, (size_t)nprob * sizeof(double), hipMemcpyDeviceToHost, st));
    PBCHK(hipMemcpyAsync(stt.data(), B.done, (size_t)nprob * sizeof(int), hipMemcpyDeviceToHost, st));
    PBCHK(hipStreamSynchronize(st));
    int bad = 0;
    for (int v : stt) bad += v != 1;
    return bad;
}

}  // extern "C"
