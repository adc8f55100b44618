// Whole steps of the oxygen chemistries (O2, Ar/O2) in two passes over the
// particles, instead of push, sort, collide and rebuild one after the other
// (which read and wrote every record three times).  Same particles, order and
// ids as the stages: a particle's collision depends on its id, the step and the
// node it lands on, not on where its record lies, so it can happen before the
// sort.
//
//   count     push, walls, null test, queued collisions (the cell's wave); per
//             (cell, slot) the survivors, and where products appeared their
//             number per species
//   victims   per destination with electron detachments: removes that many O-
//             of those that land there, smallest Philox keys first
//   totals    per destination: survivors and products of every species
//   bases     scans, new cell_start, the place of every (cell, slot) entry
//   scatter   survivors to their places (particles that did not collide are
//             pushed again: the same bits), products behind the survivors by
//             (source species, parent, slot)
//
// Bound by memory: 24 bytes read by the count pass and 24 read and written by
// the scatter, per particle, where the stages moved 180.
#include <hip/hip_runtime.h>

#include "mcc_o2_device.h"

namespace pic {

namespace {

constexpr int OW = 4;        // waves per block
constexpr int OQ = 128;      // queued colliders per wave (< 64 wait while 64 particles are tested)
constexpr int OTILE = 256;   // destinations per block of the totals and bases kernels

// per-particle tag of the first pass: move code, collided (record holds its
// final state), removed by its own collision, removed by a detachment, made
// products
enum { O2T_CODE = 15, O2T_DONE = 16, O2T_DEAD = 32, O2T_VICT = 64, O2T_PROD = 128 };

constexpr unsigned long long PMASK = (1ull << 21) - 1;
__device__ inline int made_of(const O2Products &m, int t) {
    return (int)((t < 3 ? m.lo >> (21 * t) : m.hi >> (21 * (t - 3))) & PMASK);
}

// the cells of one wave (-1 past the last) and their contiguous particle range
template <typename R, int CPW>
struct WaveCells {
    int cell[CPW], lo[CPW + 1];
    __device__ void load(const DevConst<R> &k, const PView<R> &p, int w0) {
#pragma unroll
        for (int q = 0; q < CPW; ++q) {
            const int wq = w0 + q;
            cell[q] = wq < k.Csize ? (wq / k.ncy) * k.ngy + (wq % k.ncy) : -1;
        }
        int a0 = 0, a1 = 0;
        if (cell[0] >= 0) cell_range(p, cell[0], a0, a1);
        lo[0] = a0;
        lo[1] = a1;
#pragma unroll
        for (int q = 1; q < CPW; ++q) {
            int b0 = lo[q], b1 = lo[q];
            if (cell[q] >= 0) cell_range(p, cell[q], b0, b1);
            lo[q + 1] = max(b1, lo[q]);
        }
    }
    __device__ int of(int i) const {
        int q = 0;
#pragma unroll
        for (int r = 1; r < CPW; ++r) q += i >= lo[r] ? 1 : 0;
        return q;
    }
    __device__ int node(int q) const {
        int c = cell[0];
#pragma unroll
        for (int r = 1; r < CPW; ++r) c = q == r ? cell[r] : c;
        return c;
    }
};

// routes and E corners of a wave's cells, in LDS
template <typename R, int CPW>
struct WaveTables {
    R e[CPW][8];
    int dest[CPW * ROUTE_SLOTS], info[CPW * ROUTE_SLOTS];
    __device__ void load(const DevConst<R> &k, const WaveCells<R, CPW> &C, int lane) {
        for (int t = lane; t < CPW * ROUTE_SLOTS; t += 64) {
            const int c = C.node(t / ROUTE_SLOTS);
            Route r{-1, 0};
            if (c >= 0) r = k.route[c * ROUTE_SLOTS + (t % ROUTE_SLOTS)];
            dest[t] = r.dest;
            info[t] = r.info;
        }
        if (lane < CPW * 8) {
            const int q = lane >> 3, j = lane & 7, c = C.node(q);
            R v = 0;
            if (c >= 0) {
                const int at = c + ((j & 3) == 1 ? 1 : (j & 3) == 2 ? k.ngy : (j & 3) == 3 ? k.ngy + 1 : 0);
                v = j < 4 ? k.Ex[at] : k.Ey[at];
            }
            e[q][j] = v;
        }
    }
    __device__ int push(int kq, R As, const DevConst<R> &k, R &x, R &y, R &vx, R &vy) const {
        return push_particle<R>(e[kq][0], e[kq][1], e[kq][2], e[kq][3], e[kq][4], e[kq][5], e[kq][6], e[kq][7], As,
                                k.dt_dx, k.dt_dy, x, y, vx, vy);
    }
};

// ---------------------------------------------------------------- count
template <typename R, int CPW>
struct CountLds {
    R qx[OQ], qy[OQ], qvx[OQ], qvy[OQ], qvz[OQ];   // collider queue: post-push state,
    uint32_t qid[OQ];                              // id, particle index and (draw << 8 | cell << 4 | code)
    int qkk[OQ], qmeta[OQ];
    WaveTables<R, CPW> T;
    R pb[CPW * ROUTE_SLOTS];                       // total collision probability where the entry leads
    int cnt[CPW * ROUTE_SLOTS];
    int made[CPW * ROUTE_SLOTS][CHEM_MAXSP];
    int ev[CPW][CHEM_MAXROWS];                     // events of particles that stay in their cell
};

template <typename R, int CPW>
__global__ __launch_bounds__(64 * OW) void k_o2_count(DevConst<R> k, O2Const<R> oc, O2Step<R> S) {
    __shared__ CountLds<R, CPW> lds[OW];
    __shared__ SearchRow<R> tab[CHEM_MAXROWS];
    load_search(oc, tab);
    __syncthreads();
    CountLds<R, CPW> &W = lds[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int isp = blockIdx.y;
    const int w0 = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6)) * CPW;
    if (w0 >= k.Csize) return;
    const PView<R> p = device_view(S.p[isp]);
    uint8_t *tag = device_ptr(S.tag[isp]), *fate = device_ptr(S.fate[isp]);
    R *stash = device_ptr(S.stash[isp]);
    const size_t cap = (size_t)p.cap;
    const uint32_t step = S.clk->step;
    const unsigned long long lt = lanes_below(lane);
    WaveCells<R, CPW> C;
    C.load(k, p, w0);
    const int hi = C.lo[CPW];
    // the first particles, in flight while the tables are made; lanes past
    // the end reload the last particle (never used)
    R x = 0, y = 0, vx = 0, vy = 0, vz = 0;
    uint32_t id = 0;
    if (C.lo[0] < hi) {
        const int i = min(C.lo[0] + lane, hi - 1);
        x = p.x[i]; y = p.y[i]; vx = p.vx[i]; vy = p.vy[i]; vz = p.vz[i]; id = p.id[i];
    }
    const bool collides = isp == 0 || oc.ions;
    const int g0 = kGroup0[oc.chem][isp], ng = kNGroup[oc.chem][isp];
    W.T.load(k, C, lane);
    for (int t = lane; t < CPW * ROUTE_SLOTS; t += 64) {
        const int d = W.T.dest[t];
        W.pb[t] = collides && d >= 0 ? oc.prob[(size_t)d * oc.ntgt + g0 + ng - 1] : (R)0;
        W.cnt[t] = 0;
#pragma unroll
        for (int s = 0; s < CHEM_MAXSP; ++s) W.made[t][s] = 0;
    }
    for (int t = lane; t < CPW * CHEM_MAXROWS; t += 64) (&W.ev[0][0])[t] = 0;
    wave_lds_fence();
    const R As = k.Ascale[isp];
    const int draws = ((oc.sub_mask >> isp) & 1) ? oc.MCCn : 1;
    const uint32_t mtag = mcc_tag(isp);
    int qn = 0;   // wave-uniform queue length

    // collide queue entries [q0, q0 + n), one per lane
    auto collide = [&](int q0, int n) {
        if (lane >= n) return;
        const int e = q0 + lane;
        const int meta = W.qmeta[e], code = meta & 15, kq = (meta >> 4) & 15, jc = meta >> 8;
        const int ent = kq * ROUTE_SLOTS + code, dest = W.T.dest[ent], slot = W.T.info[ent] & 15;
        const int at = kq * ROUTE_SLOTS + slot;
        const R *P = oc.prob + (size_t)dest * oc.ntgt + g0;   // target entries and handler groups share their order
        Stream st;
        st.init(oc.seed, W.qid[e], step, mtag);
        st.seek(jc);
        const R R1 = st.u<R>();
        const int flag = o2_target(P, ng, R1);
        const int kk = W.qkk[e];
        R cvx = W.qvx[e], cvy = W.qvy[e], cvz = W.qvz[e];
        int dead = 0, np = 0, detach = 0, ps[2] = {-1, -1};
        R pv[2][3];
        const int r = o2_handle<R>(oc, tab, isp, g0 + flag, dest, st, cvx, cvy, cvz, dead, ps, pv, np, detach);
        int f = code | O2T_DONE;
        if (r >= 0) {
            if (slot == 0) atomicAdd(&W.ev[kq][r], 1);
            else atomicAdd(&S.mccr[(size_t)dest * oc.TnRct + r], 1ull);
            if (dead) {
                f |= O2T_DEAD;
                atomicSub(&W.cnt[at], 1);
            }
            if (np > 0) {
                f |= O2T_PROD;
                int made = 0;
                for (int q = 0; q < np; ++q) {
                    made |= (ps[q] + 1) << (1 + 3 * q);
                    stash[(3 * q) * cap + kk] = pv[q][0];
                    stash[(3 * q + 1) * cap + kk] = pv[q][1];
                    stash[(3 * q + 2) * cap + kk] = pv[q][2];
                    atomicAdd(&W.made[at][ps[q]], 1);
                }
                fate[kk] = (uint8_t)made;
            }
            if (detach) atomicAdd(&S.delreq[dest], 1);
        }
        p.x[kk] = W.qx[e]; p.y[kk] = W.qy[e];
        if (!dead) { p.vx[kk] = cvx; p.vy[kk] = cvy; p.vz[kk] = cvz; }
        tag[kk] = (uint8_t)f;
    };

    for (int b = C.lo[0]; b < hi; b += 64) {
        R nx = 0, ny = 0, nvx = 0, nvy = 0, nvz = 0;
        uint32_t nid = 0;
        if (b + 64 < hi) {
            const int i = min(b + 64 + lane, hi - 1);
            nx = p.x[i]; ny = p.y[i]; nvx = p.vx[i]; nvy = p.vy[i]; nvz = p.vz[i]; nid = p.id[i];
        }
        const int i = b + lane;
        const bool act = i < hi;
        const int kq = C.of(i);
        const int code = W.T.push(kq, As, k, x, y, vx, vy);
        const int ent = kq * ROUTE_SLOTS + code, dest = W.T.dest[ent], info = W.T.info[ent];
        int key = -1, jc = -1;
        if (act) {
            if (dest >= 0) {
                apply_reflect<R>(info, x, y, vx, vy);
                key = kq * ROUTE_SLOTS + (info & 15);
                if (collides) {
                    const R pb = W.pb[ent];
                    Stream st;
                    st.init(oc.seed, id, step, mtag);
                    for (int j = 0; j < draws; ++j)
                        if (st.u<R>() < pb) { jc = j; break; }
                }
            } else {
                wall_effects<R>(k, Route{dest, info}, isp, C.node(kq), code, x, y, vx, vy, S.condcharge);
            }
        }
        // survivors per (cell, slot): the keys present in these 64, one by one
        unsigned long long pend = __ballot(key >= 0);
        while (pend) {
            const int kf = __builtin_amdgcn_readlane(key, __builtin_ctzll(pend));
            const unsigned long long m = __ballot(key == kf);
            if (lane == 0) W.cnt[kf] += __popcll(m);
            pend &= ~m;
        }
        const unsigned long long cm = __ballot(jc >= 0);
        if (jc >= 0) {
            const int pos = qn + __popcll(cm & lt);
            W.qx[pos] = x; W.qy[pos] = y; W.qvx[pos] = vx; W.qvy[pos] = vy; W.qvz[pos] = vz;
            W.qid[pos] = id;
            W.qkk[pos] = i;
            W.qmeta[pos] = (jc << 8) | (kq << 4) | code;
        } else if (act) {
            tag[i] = (uint8_t)code;
        }
        qn += __popcll(cm);
        wave_lds_fence();
        if (qn >= 64) {
            qn -= 64;
            collide(qn, 64);   // the newest 64; older entries stay in place
            wave_lds_fence();
        }
        x = nx; y = ny; vx = nvx; vy = nvy; vz = nvz; id = nid;
    }
    if (qn > 0) collide(0, qn);
    wave_lds_fence();
    // this wave's counts; products only for the cells that made any
    bool some = false, over = false;
    O2Products made{0, 0};
    if (lane < CPW * ROUTE_SLOTS) {
        const int c = C.node(lane / ROUTE_SLOTS);
        if (c >= 0) S.cnt[isp][c * ROUTE_SLOTS + lane % ROUTE_SLOTS] = W.cnt[lane];
#pragma unroll
        for (int s = 0; s < CHEM_MAXSP; ++s) {
            const unsigned long long m = (unsigned)W.made[lane][s];
            some |= m != 0;
            over |= m > PMASK;
            if (s < 3) made.lo |= m << (21 * s);
            else made.hi |= m << (21 * (s - 3));
        }
    }
    // more products of one species than a 21-bit field counts, from one
    // (cell, slot) in one step: reported as a bucket overflow
    if (over) atomicOr(S.err, 1);
    const unsigned long long sm = __ballot(some);
    if (lane < CPW * ROUTE_SLOTS) {
        const int q = lane / ROUTE_SLOTS, c = C.node(q);
        const bool any = (sm >> (q * ROUTE_SLOTS)) & ((1ull << ROUTE_SLOTS) - 1);
        if (c >= 0) {
            if (lane % ROUTE_SLOTS == 0) S.any[isp][c] = any ? 1 : 0;
            if (any) S.made[isp][(size_t)c * ROUTE_SLOTS + lane % ROUTE_SLOTS] = made;
        }
    }
    for (int t = lane; t < CPW * CHEM_MAXROWS; t += 64) {
        const int n = (&W.ev[0][0])[t];
        if (n) atomicAdd(&S.mccr[(size_t)C.node(t / CHEM_MAXROWS) * oc.TnRct + t % CHEM_MAXROWS], (unsigned long long)n);
    }
}

// ---------------------------------------------------------------- victims
// The O- that land on node d, in the order of its new bucket: the particles of
// d's incoming entries in canonical order.  Position j runs over all particles
// of the entries' cells; those that land elsewhere or were removed by their
// own collision are no candidates.
constexpr int OV_KEYS = 512;   // positions whose keys are kept in LDS

template <typename R>
__global__ __launch_bounds__(64 * OW) void k_o2_step_victims(DevConst<R> k, O2Const<R> oc, O2Step<R> S) {
    __shared__ uint32_t s_key[OW][OV_KEYS];
    __shared__ unsigned char s_ok[OW][OV_KEYS];
    int lane;
    const int d = wave_cell(k.ncy, k.ngy, k.Csize, lane);
    if (d < 0) return;
    const int req = S.delreq[d];
    if (req == 0) return;
    const int wv = threadIdx.x >> 6;
    const PView<R> p = S.p[oc.neg];
    uint8_t *tag = S.tag[oc.neg];
    const uint32_t step = S.clk->step;
    const uint32_t s0 = (uint32_t)oc.seed, s1 = (uint32_t)(oc.seed >> 32);
    const int e0 = S.inv_start[d], ne = S.inv_start[d + 1] - e0;   // <= 9
    int ent[ROUTE_SLOTS], first[ROUTE_SLOTS], at[ROUTE_SLOTS + 1];
    at[0] = 0;
#pragma unroll
    for (int q = 0; q < ROUTE_SLOTS; ++q) {
        ent[q] = q < ne ? S.inv_ent[e0 + q] : -1;
        int k0 = 0, k1 = 0;
        if (ent[q] >= 0) cell_range(p, ent[q] / ROUTE_SLOTS, k0, k1);
        first[q] = k0;
        at[q + 1] = at[q] + (k1 - k0);
    }
    const int n = at[ROUTE_SLOTS];
    // particle and entry of position j; whether it is a candidate
    auto find = [&](int j, int &kk, int &en) {
        kk = 0;
        en = -1;
#pragma unroll
        for (int q = 0; q < ROUTE_SLOTS; ++q)
            if (j >= at[q] && j < at[q + 1]) { kk = first[q] + (j - at[q]); en = ent[q]; }
        if (en < 0) return false;
        const int t = tag[kk];
        const Route r = k.route[(en / ROUTE_SLOTS) * ROUTE_SLOTS + (t & O2T_CODE)];
        return r.dest >= 0 && (r.info & 15) == en % ROUTE_SLOTS && !(t & O2T_DEAD);
    };
    auto key_of = [&](int j, bool &ok, int &kk, int &en) -> uint32_t {
        ok = find(j, kk, en);
        if (!ok) return 0u;
        uint32_t o[4];
        philox4x32_10(p.id[kk], step, oc.victim_tag, 0u, s0, s1, o);
        return o[0];
    };
    const bool cached = n <= OV_KEYS;
    int ncand = 0;
    for (int b = 0; b < n; b += 64) {
        const int j = b + lane;
        bool ok;
        int kk, en;
        uint32_t key = 0;
        if (cached) key = key_of(j, ok, kk, en);
        else ok = find(j, kk, en);
        ncand += __popcll(__ballot(ok));
        if (cached && j < n) {
            s_key[wv][j] = key;
            s_ok[wv][j] = ok ? 1 : 0;
        }
    }
    wave_lds_fence();
    const int kdel = min(req, ncand);
    if (kdel == 0) return;
    if (lane == 0) atomicAdd(&S.delcnt[d], (unsigned long long)kdel);
    for (int a0 = 0; a0 < n; a0 += 64) {
        const int j = a0 + lane;
        bool ok;
        int kk, en;
        const uint32_t key = key_of(j, ok, kk, en);
        int rank = 0;
        if (cached) {
            if (ok)
                for (int m = 0; m < n; ++m)
                    if (s_ok[wv][m]) {
                        const uint32_t km = s_key[wv][m];
                        if (km < key || (km == key && m < j)) ++rank;
                    }
        } else {
            for (int b0 = 0; b0 < n; b0 += 64) {
                bool om;
                int mk, me;
                const uint32_t km = key_of(b0 + lane, om, mk, me);
                for (int q = 0; q < 64; ++q) {
                    const uint32_t kv = (uint32_t)__shfl((int)km, q, 64);
                    const int av = __shfl((int)om, q, 64);
                    if (av && (kv < key || (kv == key && b0 + q < j))) ++rank;
                }
            }
        }
        // only O2T_DEAD decides candidacy, so marking here leaves the other
        // lanes' candidates unchanged
        if (ok && rank < kdel) {
            tag[kk] = (uint8_t)(tag[kk] | O2T_VICT);
            atomicSub(&S.cnt[oc.neg][en], 1);
        }
    }
}

// ---------------------------------------------------------------- totals, bases
// One thread per destination, all species: its incoming entries' survivors
// and products.  All loads of a kind are issued together, those of cells
// without products from entry 0 (their value is not used): as 45 branches that
// each waited for their own load, the bases of a 73x66 grid took 27 us.
template <int NSP>
struct DestCounts {
    int n, ent[ROUTE_SLOTS];
    int cnt[NSP][ROUTE_SLOTS];
    unsigned some[NSP];   // bit q: entry q's cell has products of species s
    int alive[NSP], prod[NSP];
    template <typename R>
    __device__ O2Products made(const O2Step<R> &S, int s, int q) const {
        const bool m = (some[s] >> q) & 1;
        const O2Products v = device_ptr(S.made[s])[m ? ent[q] : 0];
        return O2Products{m ? v.lo : 0, m ? v.hi : 0};
    }
    template <typename R>
    __device__ void load(const O2Step<R> &S, int d) {
        const int e0 = S.inv_start[d];
        n = S.inv_start[d + 1] - e0;
#pragma unroll
        for (int q = 0; q < ROUTE_SLOTS; ++q) ent[q] = q < n ? S.inv_ent[e0 + q] : -1;
#pragma unroll
        for (int s = 0; s < NSP; ++s) {
            unsigned char any[ROUTE_SLOTS];
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) {
                const int e = max(ent[q], 0);
                cnt[s][q] = S.cnt[s][e];
                any[q] = S.any[s][e / ROUTE_SLOTS];
            }
            alive[s] = 0;
            some[s] = 0;
            prod[s] = 0;
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) {
                if (ent[q] < 0) cnt[s][q] = 0;
                alive[s] += cnt[s][q];
                some[s] |= ent[q] >= 0 && any[q] ? 1u << q : 0u;
            }
        }
#pragma unroll
        for (int s = 0; s < NSP; ++s) {
            if (!__any(some[s] != 0)) continue;
            O2Products m[ROUTE_SLOTS];
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) m[q] = made(S, s, q);
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q)
#pragma unroll
                for (int t = 0; t < NSP; ++t) prod[t] += made_of(m[q], t);
        }
    }
};

template <typename R, int NSP>
__global__ __launch_bounds__(OTILE) void k_o2_step_totals(O2Step<R> S, int G) {
    __shared__ int sh[OTILE / 64][2 * NSP];
    const int d = blockIdx.x * OTILE + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int v[2 * NSP];
#pragma unroll
    for (int a = 0; a < 2 * NSP; ++a) v[a] = 0;
    if (d < G) {
        DestCounts<NSP> E;
        E.load(S, d);
#pragma unroll
        for (int t = 0; t < NSP; ++t) {
            v[t] = E.alive[t] + E.prod[t];
            v[NSP + t] = E.prod[t];
        }
    }
#pragma unroll
    for (int a = 0; a < 2 * NSP; ++a) {
        int x = v[a];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane == 0) sh[w][a] = x;
    }
    __syncthreads();
    if (threadIdx.x < 2 * NSP) {
        int x = 0;
        for (int q = 0; q < OTILE / 64; ++q) x += sh[q][threadIdx.x];
        S.sums[threadIdx.x * gridDim.x + blockIdx.x] = x;
    }
}

template <typename R, int NSP>
__global__ __launch_bounds__(OTILE) void k_o2_step_bases(O2Step<R> S, int G) {
    constexpr int NA = 2 * NSP, NW = OTILE / 64;
    __shared__ int off[NA], all[NA], wtot[NA][NW];
    const int d = blockIdx.x * OTILE + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nt = gridDim.x;
    const bool in = d < G;
    DestCounts<NSP> E;
    if (in) E.load(S, d);
    // the tiles before this one, and all tiles, per array
    for (int a = w; a < NA; a += NW) {
        int before = 0, sum = 0;
        for (int t = lane; t < nt; t += 64) {
            const int v = S.sums[a * nt + t];
            sum += v;
            if (t < (int)blockIdx.x) before += v;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            before += __shfl_xor(before, o, 64);
            sum += __shfl_xor(sum, o, 64);
        }
        if (lane == 0) { off[a] = before; all[a] = sum; }
    }
    int v[NA], incl[NA];
#pragma unroll
    for (int t = 0; t < NSP; ++t) {
        v[t] = in ? E.alive[t] + E.prod[t] : 0;
        v[NSP + t] = in ? E.prod[t] : 0;
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        incl[a] = v[a];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(incl[a], o, 64);
            if (lane >= o) incl[a] += u;
        }
        if (lane == 63) wtot[a][w] = incl[a];
    }
    __syncthreads();
    int run[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        int before = 0;
        for (int q = 0; q < w; ++q) before += wtot[a][q];
        run[a] = off[a] + before + incl[a] - v[a];
    }
    if (in) {
        int placed[NSP];
#pragma unroll
        for (int t = 0; t < NSP; ++t) {
            S.q[t].cell_start[d] = run[t];
            S.alive[(size_t)t * G + d] = run[t] + E.alive[t];   // where the products start
            S.pstart[(size_t)t * (G + 1) + d] = run[NSP + t];
            placed[t] = 0;
        }
#pragma unroll
        for (int s = 0; s < NSP; ++s) {
            int at = run[s];
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) {
                if (q < E.n) S.base[s][E.ent[q]] = at;
                at += E.cnt[s][q];
            }
            if (!E.some[s]) continue;
            O2Products m[ROUTE_SLOTS];
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) m[q] = E.made(S, s, q);
#pragma unroll
            for (int q = 0; q < ROUTE_SLOTS; ++q) {
                O2Products b{0, 0};
#pragma unroll
                for (int t = 0; t < NSP; ++t) {
                    if (t < 3) b.lo |= (unsigned long long)placed[t] << (21 * t);
                    else b.hi |= (unsigned long long)placed[t] << (21 * (t - 3));
                    placed[t] += made_of(m[q], t);
                }
                // this entry's own thread, after its count was read
                if ((E.some[s] >> q) & 1) S.made[s][E.ent[q]] = b;
            }
        }
        // the products of one destination are counted in 21 bits too
#pragma unroll
        for (int t = 0; t < NSP; ++t)
            if ((unsigned)placed[t] > (unsigned)PMASK) atomicOr(S.err, 1);
    }
    if (blockIdx.x == nt - 1 && threadIdx.x < NA) {
        const int a = threadIdx.x;
        if (a < NSP) S.q[a].cell_start[G] = all[a];
        else S.pstart[(size_t)(a - NSP) * (G + 1) + G] = all[a];
    }
}

// ---------------------------------------------------------------- scatter
template <typename R, int CPW>
struct ScatterTables {
    WaveTables<R, CPW> T;
    int made[CPW * ROUTE_SLOTS][CHEM_MAXSP];   // products placed so far
};

// A wave walks its cells' range 256 particles at a time, all loads of the 256
// in flight together; lane key holds the next place of (cell, slot) key.
template <typename R, int CPW>
__global__ __launch_bounds__(64 * OW) void k_o2_step_scatter(DevConst<R> k, O2Const<R> oc, O2Step<R> S) {
    constexpr int U = 4;
    static_assert(CPW * ROUTE_SLOTS <= 64, "one lane per (cell, slot)");
    __shared__ ScatterTables<R, CPW> lds[OW];
    ScatterTables<R, CPW> &W = lds[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int isp = blockIdx.y;
    const int w0 = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6)) * CPW;
    if (w0 >= k.Csize) return;
    const PView<R> p = device_view(S.p[isp]), q = device_view(S.q[isp]);
    const uint8_t *tag = device_ptr(S.tag[isp]);
    const unsigned long long lt = lanes_below(lane);
    WaveCells<R, CPW> C;
    C.load(k, p, w0);
    const int hi = C.lo[CPW];
    if (C.lo[0] >= hi) return;
    int next = 0;
    if (lane < CPW * ROUTE_SLOTS) {
        const int c = C.node(lane / ROUTE_SLOTS);
        if (c >= 0) next = S.base[isp][c * ROUTE_SLOTS + lane % ROUTE_SLOTS];
#pragma unroll
        for (int s = 0; s < CHEM_MAXSP; ++s) W.made[lane][s] = 0;
    }
    W.T.load(k, C, lane);
    wave_lds_fence();
    const R As = k.Ascale[isp];
    for (int b0 = C.lo[0]; b0 < hi; b0 += 64 * U) {
        R x[U], y[U], vx[U], vy[U], vz[U];
        uint32_t id[U];
        int tg[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int i = min(b0 + j * 64 + lane, hi - 1);
            tg[j] = tag[i];
            x[j] = p.x[i]; y[j] = p.y[i]; vx[j] = p.vx[i]; vy[j] = p.vy[i]; vz[j] = p.vz[i]; id[j] = p.id[i];
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int i = b0 + j * 64 + lane;
            if (b0 + j * 64 >= hi) break;
            const int t = tg[j];
            const int kq = C.of(i), ent = kq * ROUTE_SLOTS + (t & O2T_CODE);
            const int dest = W.T.dest[ent], info = W.T.info[ent];
            if (!(t & O2T_DONE)) {
                W.T.push(kq, As, k, x[j], y[j], vx[j], vy[j]);
                if (dest >= 0) apply_reflect<R>(info, x[j], y[j], vx[j], vy[j]);
            }
            const bool lands = i < hi && dest >= 0;
            const int key = kq * ROUTE_SLOTS + (info & 15);
            const int keep = lands && !(t & (O2T_DEAD | O2T_VICT)) ? key : -1;
            int pos = -1;
            unsigned long long pend = __ballot(keep >= 0);
            while (pend) {
                const int kf = __builtin_amdgcn_readlane(keep, __builtin_ctzll(pend));
                const unsigned long long m = __ballot(keep == kf);
                const int at = __builtin_amdgcn_readlane(next, kf);
                if (keep == kf) pos = at + __popcll(m & lt);
                if (lane == kf) next += __popcll(m);
                pend &= ~m;
            }
            if (keep >= 0) {
                if (pos < q.cap) {
                    q.x[pos] = x[j]; q.y[pos] = y[j]; q.vx[pos] = vx[j]; q.vy[pos] = vy[j]; q.vz[pos] = vz[j];
                    q.id[pos] = id[j];
                } else {
                    atomicOr(S.err, 1);
                }
            }
            // products, parent by parent: most groups of 64 have none
            unsigned long long pm = __ballot(lands && (t & O2T_PROD));
            if (!pm) continue;
            const int made = lands && (t & O2T_PROD) ? S.fate[isp][i] : 0;
            while (pm) {
                const int L = __builtin_ctzll(pm);
                pm &= pm - 1;
                const int kL = __builtin_amdgcn_readlane(key, L);
                const int mL = __builtin_amdgcn_readlane(made, L);
                for (int s2 = 0; s2 < 2; ++s2) {
                    const int ts = o2_fate_prod((uint8_t)mL, s2);
                    if (ts < 0) continue;
                    const int r = W.made[kL][ts];
                    wave_lds_fence();
                    if (lane == L) {
                        W.made[kL][ts] = r + 1;
                        const O2Products b = S.made[isp][(size_t)C.node(kq) * ROUTE_SLOTS + kL % ROUTE_SLOTS];
                        const int rank = made_of(b, ts) + r;
                        const int at = S.alive[(size_t)ts * oc.G + dest] + rank;
                        const PView<R> &d = S.q[ts];
                        if (at < d.cap) {
                            const R *sv = S.stash[isp] + (size_t)(3 * s2) * p.cap + i;
                            d.x[at] = x[j]; d.y[at] = y[j];
                            d.vx[at] = sv[0]; d.vy[at] = sv[(size_t)p.cap]; d.vz[at] = sv[2 * (size_t)p.cap];
                            d.id[at] = S.next_id[ts] + (uint32_t)(S.pstart[(size_t)ts * (oc.G + 1) + dest] + rank);
                        } else {
                            atomicOr(S.err, 1);
                        }
                    }
                    wave_lds_fence();
                }
            }
        }
    }
}

template <typename R, int CPW>
void launch_cpw(const DevConst<R> &k, const O2Const<R> &oc, const O2Step<R> &S, hipStream_t s) {
    const int nb = (k.Csize + CPW * OW - 1) / (CPW * OW), nt = (oc.G + OTILE - 1) / OTILE;
    const int cells = (k.Csize + OW - 1) / OW;
    hipLaunchKernelGGL((k_o2_count<R, CPW>), dim3(nb, oc.nsp), dim3(64 * OW), 0, s, k, oc, S);
    hipLaunchKernelGGL(k_o2_step_victims<R>, dim3(cells), dim3(64 * OW), 0, s, k, oc, S);
    if (oc.nsp == 5) {
        hipLaunchKernelGGL((k_o2_step_totals<R, 5>), dim3(nt), dim3(OTILE), 0, s, S, oc.G);
        hipLaunchKernelGGL((k_o2_step_bases<R, 5>), dim3(nt), dim3(OTILE), 0, s, S, oc.G);
    } else {
        hipLaunchKernelGGL((k_o2_step_totals<R, 4>), dim3(nt), dim3(OTILE), 0, s, S, oc.G);
        hipLaunchKernelGGL((k_o2_step_bases<R, 4>), dim3(nt), dim3(OTILE), 0, s, S, oc.G);
    }
    hipLaunchKernelGGL((k_o2_step_scatter<R, CPW>), dim3(nb, oc.nsp), dim3(64 * OW), 0, s, k, oc, S);
}

}  // namespace

int o2_step_sums(int G, int nsp) { return 2 * nsp * ((G + OTILE - 1) / OTILE); }

// cells per wave: as in the argon count pass, four where that leaves enough
// waves to fill the chip (72x65 cells, 24 particles per cell: the scatter takes
// 18 us with one cell per wave and 37 with four)
template <typename R>
void launch_o2_step(const DevConst<R> &k, const O2Const<R> &oc, const O2Step<R> &S, hipStream_t s) {
    launch_o2_probs<R>(oc, S.delreq, s);
    if (k.Csize >= 16384) launch_cpw<R, 4>(k, oc, S, s);
    else launch_cpw<R, 1>(k, oc, S, s);
}
template void launch_o2_step<float>(const DevConst<float> &, const O2Const<float> &, const O2Step<float> &, hipStream_t);
template void launch_o2_step<double>(const DevConst<double> &, const O2Const<double> &, const O2Step<double> &,
                                     hipStream_t);

}  // namespace pic
