// Register-resident PCG (pcg_resident.hip): plan and entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pic_kernels.h"

namespace pic {

struct ResidentState {
    unsigned int solve;   // number of the solve, the upper bits of its exchange tags
    unsigned int abort;   // a wait ran out of time; every block then leaves
};

// Launch shape, column map and exchange words of one operator
struct PcgResident {
    int N = 0, bs = 0, rpt = 0, nblk = 0, rows = 0;
    size_t lds = 0;
    uint16_t *lcol = nullptr;
    double *off = nullptr, *diag = nullptr;
    float *weight = nullptr;
    uint8_t *pub = nullptr;
    int *ghost_start = nullptr, *ghost = nullptr;
    unsigned long long *halo = nullptr, *part = nullptr;
    ResidentState *st = nullptr;
};

// col, val: the operator's 5N columns and values (host).  Returns null with
// *err == 0 for an operator outside the range (more unknowns than half the
// CUs hold, rows coupled to more of them than a block's LDS takes, or no row
// weights that make it symmetric).
PcgResident *pcg_resident_create(int N, const int *col, const double *val, int ncu, int want_blocks, bool split, hipStream_t s, int *err);
void pcg_resident_destroy(PcgResident *w);
hipError_t pcg_resident_reset(PcgResident *w, hipStream_t s);
hipError_t pcg_resident_plain(PcgResident *w, const PcgOperator &A, const double *b, double *x, double tol, int maxit,
                              unsigned long long spin_limit, PcgResult *res, hipStream_t s);
hipError_t pcg_resident_refined(PcgResident *w, const PcgOperator &A, const float *b, double *x, double tol,
                                double inner_tol, int maxit, unsigned long long spin_limit, PcgResult *res,
                                hipStream_t s);

}  // namespace pic
