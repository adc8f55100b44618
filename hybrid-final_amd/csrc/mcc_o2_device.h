// Device code shared by the kernels of the oxygen chemistries: the collision
// tables and the handling of one collision.
#pragma once
#include <hip/hip_runtime.h>

#include "mcc_o2.h"

namespace pic {
namespace {

struct ChemRow {
    int r, sum, type, emode;
    double gain;
    int p0, p1, th;
};
struct ChemGroup {
    int sp, flag, sig, first, n, vsrc;
};
struct ChemTarget {
    int sp, flag, sig, kind, idx;
};

// both chemistries in one form: O2 rows subtract their own threshold, and
// its O2+ and O+ collide in the frame of a neutral at BackVel1
#define PIC_O2_ROW(r, sm, ty, em, g, a, b) {r, sm, ty, em, g, a, b, r},
#define PIC_ARO2_ROW(r, sm, ty, em, g, a, b, th) {r, sm, ty, em, g, a, b, th},
#define PIC_O2_GRP(s, f, sg, fi, n) {s, f, sg, fi, n, (s) == 1 || (s) == 2 ? 1 : 0},
#define PIC_ARO2_GRP(s, f, sg, fi, n, v) {s, f, sg, fi, n, v},
#define PIC_TGT(s, f, sg, kd, ix) {s, f, sg, kd, ix},
__constant__ ChemRow kRow[2][CHEM_MAXROWS] = {{O2_REACTIONS(PIC_O2_ROW)}, {ARO2_REACTIONS(PIC_ARO2_ROW)}};
__constant__ ChemGroup kGrp[2][CHEM_MAXGROUPS] = {{O2_GROUPS(PIC_O2_GRP)}, {ARO2_GROUPS(PIC_ARO2_GRP)}};
__constant__ ChemTarget kTgt[2][CHEM_MAXTARGETS] = {{O2_TARGETS(PIC_TGT)}, {ARO2_TARGETS(PIC_TGT)}};
__constant__ int kGroup0[2][CHEM_MAXSP] = {O2_GROUP0, ARO2_GROUP0};
__constant__ int kNGroup[2][CHEM_MAXSP] = {O2_NGROUP, ARO2_NGROUP};
#undef PIC_O2_ROW
#undef PIC_ARO2_ROW
#undef PIC_O2_GRP
#undef PIC_ARO2_GRP
#undef PIC_TGT

template <typename R>
__device__ inline void o2_maxwell(const O2Const<R> &k, R vti, Stream &st, R &vx, R &vy, R &vz) {
    const int n = (int)((R)(k.nvel - 1) * st.u<R>());
    const R rphi = st.u<R>(), rthe = st.u<R>();
    maxwell_draw<R>(vx, vy, vz, k.vsave[n], vti, rphi, rthe);
}

// What the reaction search reads of a row, in LDS: a lane's rows differ from
// its neighbours', and each read of the constant tables, then of the
// threshold, was a round trip to L2 on the search's serial chain.
template <typename R>
struct SearchRow {
    R th;
    int r, sum;
};
template <typename R>
__device__ inline void load_search(const O2Const<R> &k, SearchRow<R> *tab) {
    for (int q = threadIdx.x; q < CHEM_MAXROWS; q += blockDim.x) {
        const int r = kRow[k.chem][q].r;
        tab[q] = SearchRow<R>{k.Th_e[r], r, kRow[k.chem][q].sum};
    }
}

// The handler group of a collision draw: the first of the species' ng
// cumulative target probabilities that reaches R1, all of them loaded together
constexpr int CHEM_MAXNG = 9;
template <typename R>
__device__ inline int o2_target(const R *P, int ng, R R1) {
    R v[CHEM_MAXNG];
#pragma unroll
    for (int j = 0; j < CHEM_MAXNG; ++j) v[j] = P[min(j, ng - 1)];
    int flag = ng - 1;
#pragma unroll
    for (int j = CHEM_MAXNG - 1; j >= 0; --j)
        if (j < ng - 1 && !(R1 > v[j])) flag = j;
    return flag;
}

// One collision of a particle of species isp with the target of group grp.
// Returns the reaction (or -1 for a null collision); vx..vz are updated for
// a survivor, and dead / products / detach describe the rest.
template <typename R>
__device__ inline int o2_handle(const O2Const<R> &k, const SearchRow<R> *tab, int isp, int grp, int c, Stream &st,
                                R &vx, R &vy, R &vz,
                                int &dead, int ps[2], R pv[2][3], int &np, int &detach) {
    const ChemGroup g = kGrp[k.chem][grp];
    R vnx = 0, vny = 0, vnz = 0;
    const bool heavy = g.vsrc != 0;   // positive ions collide in the neutral's frame
    if (heavy) o2_maxwell<R>(k, g.vsrc == 2 ? k.BackVel2[c] : k.BackVel1[c], st, vnx, vny, vnz);
    R VX = vx - vnx, VY = vy - vny, VZ = vz - vnz;
    const R dum = VX * VX + VY * VY + VZ * VZ;
    R vel = rsqrt_ieee<R>(dum);
    if (!heavy) { VX /= vel; VY /= vel; VZ /= vel; }
    R engy = k.Escale[isp] * dum;
    const R R1 = st.u<R>() * k.sigv[g.sig] / vel;
    ArXs<R> xs;
    xs.init(k, engy);
    R sum = 0;
    int hit = -1;
    // four reactions' lookups in flight, then their comparisons in order
    const int end = g.first + g.n;
    for (int q0 = g.first; q0 < end && hit < 0; q0 += 4) {
        R th[4], sg[4];
        int add[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const SearchRow<R> row = tab[min(q0 + j, end - 1)];
            th[j] = row.th;
            add[j] = row.sum;
            sg[j] = xs.sigma(k, row.r);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (hit < 0 && q0 + j < end && engy > th[j]) {
                sum = add[j] ? sum + sg[j] : sg[j];
                if (R1 <= sum) hit = q0 + j;
            }
    }
    if (hit < 0) return -1;
    const ChemRow row = kRow[k.chem][hit];
    const R Es = k.Escale[isp];
    switch (row.type) {
    case O2T_LOSS:
    case O2T_ION:
    case O2T_DETACH: {
        if (row.emode == O2E_LOSS) {
            engy -= k.Th_e[row.th];
            vel = rsqrt_ieee<R>(rabs<R>(engy) / Es);
        } else if (row.emode == O2E_GAIN) {
            engy += (R)row.gain;
            vel = rsqrt_ieee<R>(rabs<R>(engy) / Es);
        }
        if (row.type == O2T_ION) {
            for (int slot = 0; slot < 2; ++slot) {
                const int sp = slot ? row.p1 : row.p0;
                ps[np] = sp;
                if (sp == 0) { pv[np][0] = VX; pv[np][1] = VY; pv[np][2] = VZ; }
                else o2_maxwell<R>(k, k.BackVel1[c], st, pv[np][0], pv[np][1], pv[np][2]);
                ++np;
            }
        } else if (row.type == O2T_DETACH) {
            ps[np] = 0; pv[np][0] = VX; pv[np][1] = VY; pv[np][2] = VZ; ++np;
            detach = 1;
        }
        const R a = st.u<R>(), b = st.u<R>();
        anewvel<R>(engy, vel, VX, VY, VZ, a, b);
        vx = VX; vy = VY; vz = VZ;
        break;
    }
    case O2T_IONSHARE: {
        engy -= k.Th_e[row.th];
        const R u = st.u<R>();
        const R rengy = (R)10 * PMath<R>::tan(u * PMath<R>::atan(engy / (R)20));
        engy -= rengy;
        const R velr = rsqrt_ieee<R>(rabs<R>(rengy) / Es);
        const R vel2 = rsqrt_ieee<R>(rabs<R>(engy) / Es);
        for (int slot = 0; slot < 2; ++slot) {
            const int sp = slot ? row.p1 : row.p0;
            ps[np] = sp;
            if (sp == 0) {
                R ex = VX, ey = VY, ez = VZ;
                const R a = st.u<R>(), b = st.u<R>();
                anewvel<R>(rengy, velr, ex, ey, ez, a, b);
                pv[np][0] = ex; pv[np][1] = ey; pv[np][2] = ez;
            } else {
                o2_maxwell<R>(k, k.BackVel1[c], st, pv[np][0], pv[np][1], pv[np][2]);
            }
            ++np;
        }
        const R a = st.u<R>(), b = st.u<R>();
        anewvel<R>(engy, vel2, VX, VY, VZ, a, b);
        vx = VX; vy = VY; vz = VZ;
        break;
    }
    case O2T_ATTACH:
        dead = 1;
        ps[np] = row.p0;
        o2_maxwell<R>(k, k.BackVel1[c], st, pv[np][0], pv[np][1], pv[np][2]);
        ++np;
        break;
    case O2T_DEL:
        dead = 1;
        break;
    case O2T_SCAT: {
        const R a = st.u<R>(), b = st.u<R>();
        newvel_ionsc<R>(VX, VY, VZ, vel, a, b);
        if (heavy) { vx = VX + vnx; vy = VY + vny; vz = VZ + vnz; }
        else { vx = VX; vy = VY; vz = VZ; }
        break;
    }
    case O2T_CXKEEP:
        vx = vnx; vy = vny; vz = vnz;
        break;
    case O2T_CXTO:
        dead = 1;
        ps[np] = row.p0; pv[np][0] = vnx; pv[np][1] = vny; pv[np][2] = vnz; ++np;
        break;
    default:   // O2T_NEGDET
        dead = 1;
        ps[np] = 0; pv[np][0] = VX; pv[np][1] = VY; pv[np][2] = VZ; ++np;
        break;
    }
    return row.r;
}

}  // namespace
}  // namespace pic
