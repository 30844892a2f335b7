// inner_terms.h -- the bonded terms of the device integrators' inner loops
// (k_integrate.hip, k_nvt.hip): bonded_term with shorter dependency chains
// for the harmonic bond and angle.
#pragma once
#include "terms.h"

// bonded_term for the inner loop's latency chain: the harmonic bond and the
// harmonic angle with reciprocal square roots (the hardware estimate and two
// Newton steps, a shorter dependency chain) in place of sqrt and division, no
// further from the exact force than bonded_term is: RMS against quad precision,
// in fractions of the force 3% off a bond's length and 0.08 rad off an angle,
// bond 5.5e-17 (bonded_term 9.6e-16; 1.5e-15 without the low part of r, since
// r - r0 cancels), angle 7.5e-16 (7.7e-16).  Every other term but the cosine
// dihedral is bonded_term's.  The caller's force copy holds this one term only and starts
// from zero, so the two fast terms store their forces (0 + f is f) instead of
// reading the copy back.
__device__ inline int bonded_term_inner(const TermDev& T, int base, const double* xx,
                                        const double* yy, const double* zz, double* fxs,
                                        double* fys, double* fzs, double* u, double* vir,
                                        int* singular, int stride, bool energy = true) {
#pragma clang fp contract(off)
    const double* pr = T.para;
    if (T.kind == TERM_BOND && T.type == MSPMS_BOND_HARMONIC) {
        const int i1 = base + T.idx[0] * stride, i2 = base + T.idx[1] * stride;
        const double rx = xx[i1] - xx[i2], ry = yy[i1] - yy[i2], rz = zz[i1] - zz[i2];
        const double rsq = rx * rx + ry * ry + rz * rz, ri = rsqrt_fma(rsq), r = rsq * ri;
        // sqrt(rsq) is r + fma(-r, r, rsq) / (2 r) to the last bit and beyond
        const double dr = fma(fma(-r, r, rsq), 0.5 * ri, r - pr[1]);
        *u = 0.5 * pr[0] * dr * dr;
        const double fij = -pr[0] * dr * ri;
        *vir = fij * rsq;
        fxs[i1] = fij * rx;
        fys[i1] = fij * ry;
        fzs[i1] = fij * rz;
        fxs[i2] = -(fij * rx);
        fys[i2] = -(fij * ry);
        fzs[i2] = -(fij * rz);
        return 0;
    }
    if (T.kind == TERM_ANGLE && T.type == MSPMS_ANGLE_HARMONIC) {
        const int ia = base + T.idx[0] * stride, ib = base + T.idx[1] * stride,
                  ic = base + T.idx[2] * stride;
        double xab = xx[ia] - xx[ib], yab = yy[ia] - yy[ib], zab = zz[ia] - zz[ib];
        double xbc = xx[ic] - xx[ib], ybc = yy[ic] - yy[ib], zbc = zz[ic] - zz[ib];
        const double rrab = rsqrt_fma(xab * xab + yab * yab + zab * zab);
        const double rrbc = rsqrt_fma(xbc * xbc + ybc * ybc + zbc * zbc);
        xab = xab * rrab;
        yab = yab * rrab;
        zab = zab * rrab;
        xbc = xbc * rrbc;
        ybc = ybc * rrbc;
        zbc = zbc * rrbc;
        double cost = xab * xbc + yab * ybc + zab * zbc;
        // (a straight molecule's cosine can come out an ulp beyond 1, of which
        // acos has no value; NaN stays NaN)
        if (fabs(cost) > 1.0) cost = copysign(1.0, cost);
        const double theta = acos(cost);
        // 1 / max(1e-8, sin theta)
        const double s2 = 1.0 - cost * cost;
        const double rsint = s2 > 1.0e-16 ? rsqrt_fma(s2) : 1.0e8;
        const double dth = theta - pr[1];
        *u = 0.5 * pr[0] * dth * dth;
        const double gam = pr[0] * dth * rsint;
        const double fxa = gam * (xbc - xab * cost) * rrab, fya = gam * (ybc - yab * cost) * rrab,
                     fza = gam * (zbc - zab * cost) * rrab;
        const double fxc = gam * (xab - xbc * cost) * rrbc, fyc = gam * (yab - ybc * cost) * rrbc,
                     fzc = gam * (zab - zbc * cost) * rrbc;
        *vir = 0.0;
        fxs[ia] = fxa;
        fys[ia] = fya;
        fzs[ia] = fza;
        fxs[ib] = -fxa - fxc;
        fys[ib] = -fya - fyc;
        fzs[ib] = -fza - fzc;
        fxs[ic] = fxc;
        fys[ic] = fyc;
        fzs[ic] = fzc;
        return 1;
    }
    if (T.kind == TERM_DIH && T.type == MSPMS_DIH_OPLS_COSIN) {
        // the angle's cosine and sine follow from the cross products, the sines
        // of its multiples from the addition theorems: no atan2 and no
        // trigonometric functions on the way to the force (17,627 dihedrals, 5
        // steps: 65 us with them, 33 without; the force's error against
        // extended precision, over random and nearly planar forms, is 1.3e-10 in
        // the mean and 4.6e-14 in the median against 1.7e-10 and 6.1e-14).  The
        // energy, whose error would grow by a quarter, is the reference's
        // expression, taken where it is asked for
        const int ia = base + T.idx[0] * stride, ib = base + T.idx[1] * stride,
                  ic = base + T.idx[2] * stride, id = base + T.idx[3] * stride;
        const double xab = xx[ia] - xx[ib], yab = yy[ia] - yy[ib], zab = zz[ia] - zz[ib];
        const double xbc = xx[ib] - xx[ic], ybc = yy[ib] - yy[ic], zbc = zz[ib] - zz[ic];
        const double xcd = xx[ic] - xx[id], ycd = yy[ic] - yy[id], zcd = zz[ic] - zz[id];
        const double rrbc = rsqrt_fma(xbc * xbc + ybc * ybc + zbc * zbc);
        const double pbx = yab * zbc - zab * ybc, pby = zab * xbc - xab * zbc,
                     pbz = xab * ybc - yab * xbc;
        const double rpb1 = rsqrt_fma(pbx * pbx + pby * pby + pbz * pbz), rpb2 = rpb1 * rpb1;
        const double pcx = ybc * zcd - zbc * ycd, pcy = zbc * xcd - xbc * zcd,
                     pcz = xbc * ycd - ybc * xcd;
        const double rpc1 = rsqrt_fma(pcx * pcx + pcy * pcy + pcz * pcz), rpc2 = rpc1 * rpc1;
        const double pbpc = pbx * pcx + pby * pcy + pbz * pcz, rr = rpb1 * rpc1;
        const double cost = pbpc * rr;
        const double sint = (xbc * (pcy * pbz - pcz * pby) + ybc * (pbx * pcz - pbz * pcx) +
                             zbc * (pcx * pby - pcy * pbx)) * (rr * rrbc);
        // on the unit circle to the rounding error squared
        const double nrm = 1.5 - 0.5 * (cost * cost + sint * sint);
        const double c1 = cost * nrm, s1 = sint * nrm;
        const double c2 = c1 * c1 - s1 * s1, s2 = 2.0 * s1 * c1;
        const double s3 = s1 * c2 + c1 * s2;
        *u = 0.0;
        if (energy) {
            const double theta = atan2(sint, cost);
            *u = pr[0] + 0.5 * (pr[1] * (1.0 + cos(theta)) + pr[2] * (1.0 - cos(2.0 * theta)) +
                                pr[3] * (1.0 + cos(3.0 * theta)));
        }
        *vir = 0.0;
        const double dopls = -0.5 * (pr[1] * s1 - 2.0 * pr[2] * s2 + 3.0 * pr[3] * s3);
        const double gam = dopls * rr / copysign(fmax(1.0e-8, fabs(sint)), sint);
        const double qb = pbpc * rpb2, qc = pbpc * rpc2;
        // d cos / d pb and d cos / d pc, up to gam
        const double ubx = pcx - qb * pbx, uby = pcy - qb * pby, ubz = pcz - qb * pbz;
        const double ucx = pbx - qc * pcx, ucy = pby - qc * pcy, ucz = pbz - qc * pcz;
        const double fax = gam * (ubz * ybc - uby * zbc), fay = gam * (ubx * zbc - ubz * xbc),
                     faz = gam * (uby * xbc - ubx * ybc);
        const double fcx = gam * (ubz * yab - uby * zab), fcy = gam * (ubx * zab - ubz * xab),
                     fcz = gam * (uby * xab - ubx * yab);
        const double fbx = gam * (ucz * ycd - ucy * zcd), fby = gam * (ucx * zcd - ucz * xcd),
                     fbz = gam * (ucy * xcd - ucx * ycd);
        const double fdx = gam * (ucz * ybc - ucy * zbc), fdy = gam * (ucx * zbc - ucz * xbc),
                     fdz = gam * (ucy * xbc - ucx * ybc);
        fxs[ia] += fax;
        fys[ia] += fay;
        fzs[ia] += faz;
        fxs[ib] += (-fax - fcx + fbx);
        fys[ib] += (-fay - fcy + fby);
        fzs[ib] += (-faz - fcz + fbz);
        fxs[ic] += fcx - fbx - fdx;
        fys[ic] += fcy - fby - fdy;
        fzs[ic] += fcz - fbz - fdz;
        fxs[id] += fdx;
        fys[id] += fdy;
        fzs[id] += fdz;
        return 2;
    }
    return bonded_term(T, base, xx, yy, zz, fxs, fys, fzs, u, vir, singular, stride);
}
