// npt_box.h -- the box of the NPT step's inner loop (k_npt.hip,
// k_integrate.hip).
#pragma once
#include "engine.h"
#include "../../include/mspms_gpu.h"

// The replica's box after n inner steps (src/nptnh.c:179-199), and the
// tables that the force kernels read.  The barostat's velocity stays as it
// is over the inner loop, and nothing there reads the box, so only the edges
// take every step.
__device__ inline void npt_box(RepDev& R, NptDev& S, double delts, int n) {
#pragma clang fp contract(off)
    constexpr double PI = 3.141592653589793;  // src/defs.h:98
    const double expfactor = exp(delts * S.vbs);
    const int nc[3] = {R.ncx, R.ncy, R.ncz};
    for (int d = 0; d < 3; d++) {
        double L = R.L[d];
        for (int k = 0; k < n; k++) L = L * expfactor;
        R.L[d] = L;
        R.invL[d] = 1.0 / L;
        R.h[d] = L / nc[d];
        R.inv_h[d] = 1.0 / R.h[d];
    }
    const double boxv = R.L[0] * R.L[1] * R.L[2];
    S.boxv = boxv;
    double p = 0.0;
    for (int k = 0; k < S.nlrc; k++) p += S.lrc[k] / boxv / boxv;
    S.pljlrc = p;
    if (R.charge_type == MSPMS_ELEC_EWALD) {
        R.vfactor = 2.0 * PI / boxv;
        for (int d = 0; d < 3; d++) R.twopi_l[d] = 2.0 * PI / R.L[d];
        R.twopi_over_3v = 2.0 * PI / 3.0 / boxv;
    }
}
