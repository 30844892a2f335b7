// physics.h -- pair terms shared by the gfx950 kernels.
//
// FP64 versions keep the reference's expression order with contraction
// disabled, so that they round like the reference's x86-64 build; the libm
// calls become ROCm device-library calls (erfc, exp: ~1 ulp).  The exact pair
// kernel takes Ewald and Wolf terms in another form (erfc_exp64, rsqrt_fma),
// whose rounding error is smaller.
// FP32 versions are the mixed-precision pair arithmetic.
#pragma once
#include <hip/hip_runtime.h>

#define MSPMS_PI 3.141592653589793  // src/defs.h:100

// ---- FP64 ---------------------------------------------------------------
// ljfrc (src/ljfrc.c:21-71)
__host__ __device__ inline void lj64(double rijsq, double sigmaij, double epsilonij, int switch_on,
                            double rcutoffsq, double rcutonsq, double roff2_ron2_cube,
                            double shift1, double* uij, double* fij, double* ushift) {
#pragma clang fp contract(off)
    double sw = 0.0;
    if (switch_on) {
        if (rijsq < rcutonsq)
            sw = 1.0;
        else
            sw = (rcutoffsq - rijsq) * (rcutoffsq - rijsq) * (rcutoffsq + 2.0 * rijsq - 3.0 * rcutonsq) /
                 roff2_ron2_cube;
    }
    double r_rijsq = 1.0 / rijsq;
    double s2 = sigmaij * sigmaij;
    double r6 = s2 * r_rijsq;
    r6 = r6 * r6 * r6;
    double r12 = r6 * r6;
    double u = 4.0 * epsilonij * (r12 - r6);
    if (switch_on) {
        if (rijsq < rcutonsq) {
            *fij = 24.0 * epsilonij * (2 * r12 - r6) * r_rijsq;
        } else {
            *fij = 24.0 * epsilonij * (2 * r12 - r6) * r_rijsq * sw -
                   u * 12.0 * (rcutoffsq - rijsq) * (rcutonsq - rijsq) / roff2_ron2_cube;
            u *= sw;
        }
        *ushift = 0.0;
    } else {
        *fij = 24.0 * epsilonij * (2 * r12 - r6) * r_rijsq;
        double s6 = s2 * s2 * s2;
        *ushift = epsilonij * s6 * (s6 * shift1 - 1.0);
    }
    *uij = u;
}

// Parameter derivatives of the ljfrc energy: du/dsigma_ij and du/deps_ij of
// u = 4 eps (s^12 - s^6) [* sw(r)], s = sigma / r; the switch factor does
// not depend on the parameters.
__host__ __device__ inline void lj64_dparam(double rijsq, double sigmaij, double epsilonij, int switch_on,
                                   double rcutoffsq, double rcutonsq, double roff2_ron2_cube,
                                   double* du_dsigma, double* du_deps) {
    double sw = 1.0;
    if (switch_on && !(rijsq < rcutonsq))
        sw = (rcutoffsq - rijsq) * (rcutoffsq - rijsq) * (rcutoffsq + 2.0 * rijsq - 3.0 * rcutonsq) /
             roff2_ron2_cube;
    double r6 = sigmaij * sigmaij / rijsq;
    r6 = r6 * r6 * r6;
    const double r12 = r6 * r6;
    *du_deps = 4.0 * (r12 - r6) * sw;
    *du_dsigma = 24.0 * epsilonij * (2.0 * r12 - r6) / sigmaij * sw;
}

// d eps_ij / d eps_i of the mixing rule eps_ij = sqrt(eps_i eps_j): infinite
// at eps_i = 0 < eps_j, where the square root has no derivative
__host__ __device__ inline double deps_mix(double eij, double eps_j) {
    if (eij > 0.0) return 0.5 * eps_j / eij;
    return eps_j == 0.0 ? 0.0 : __builtin_huge_val();
}

// ewald_real_frc (src/elecfrc.c:17-33)
__host__ __device__ inline void ewald_real64(double rijsq, double qq, double C, double kappa, double* uij,
                                    double* fij) {
#pragma clang fp contract(off)
    double rij = sqrt(rijsq);
    double ut = C * qq / rij;
    *uij = ut * erfc(kappa * rij);
    double t1 = kappa * rij;
    double t2 = ut * erfc(t1);
    *fij = (t2 + ut * 2.0 * t1 * exp(-t1 * t1) / sqrt(MSPMS_PI)) / rijsq;
}

// ewald_excl_frc (src/elecfrc.c:35-46)
__host__ __device__ inline void ewald_excl64(double rijsq, double qq, double C, double* uij, double* fij) {
#pragma clang fp contract(off)
    double rij = sqrt(rijsq);
    *uij = C * qq / rij;
    *fij = -*uij / rijsq;
}

// xatom_coulomb_frc (src/elecfrc.c:159-170): bare Coulomb, u = C qq / r,
// F_i = (u / r^2) r_ij
__host__ __device__ inline void coulomb64(double rijsq, double qq, double C, double* uij,
                                          double* fij) {
#pragma clang fp contract(off)
    double rij = sqrt(rijsq);
    *uij = C * qq / rij;
    *fij = *uij / rijsq;
}

// wolf_real_frc (src/elecfrc.c:48-60)
__host__ __device__ inline void wolf_real64(double rijsq, double qq, double C, double kappa, double rc,
                                   double v1, double v2, double f1, double f2, double* uij,
                                   double* fij) {
#pragma clang fp contract(off)
    double rij = sqrt(rijsq);
    *uij = C * qq * (erfc(kappa * rij) / rij + v1 + v2 * (rij - rc));
    *fij = C * (qq / rij) * (erfc(kappa * rij) / rijsq + f1 * exp(-(kappa * rij) * (kappa * rij)) / rij +
                             f2);
}

// ---- FP64, shared transcendentals ------------------------------------------
// 1 / x within an ulp: the hardware estimate and two Newton steps
__device__ inline double rcp_nr(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}

// 1 / sqrt(x) within an ulp, x > 0 (NaN at 0)
__device__ inline double rsqrt_fma(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double h = 0.5 * x * y;
    y = fma(y, fma(-h, y, 0.5), y);
    h = 0.5 * x * y;
    return fma(y, fma(-h, y, 0.5), y);
}

// erfc(x) and exp(-x^2) for x >= 0 without a branch: erfc(x) = exp(-x^2)
// P(t) / (1 + 2 x) with t = (x - K) / (x + K), the mapping of Shepherd and
// Laframboise (Math. Comp. 36, 1981) with K = 3.75; P is the degree-22
// truncation of the Chebyshev series of (1 + 2 x) exp(x^2) erfc(x) in t,
// computed with 70 digits and summed into powers of t (all coefficients
// below 1.24, so Horner's rule loses nothing); the truncation is 1.4e-16
// relative on [0, 12], the result within 6.4e-16 (1.3e-16 in the mean).  The
// exponential is 2^n exp(r), |r| <= ln 2 / 2, by its Taylor polynomial of
// degree 13 (remainder 4e-18), with the rounding of x^2 taken back out.  xl is
// the part of the argument below x's last bit: exp(-x^2) changes by the
// fraction 2 x xl, 2 x^2 times the argument's own relative error, the rest
// of erfc by no more than that error itself.  The math library's erfc branches
// by range, so that a wave with mixed arguments runs every range, and
// evaluates its own exponential.
//
// The coefficients (highest power first, then 1 / 13! .. 1 / 2!) are read
// through the scalar cache where they are used: as literals they would be
// kept in 70 vector registers across the caller's loop, half of what a wave
// has at four waves per SIMD.
constexpr int ERFC_NP = 23, ERFC_NE = 12;
__device__ __constant__ const double erfc_coef[ERFC_NP + ERFC_NE] = {
    -2.623107347133476e-09, -1.9551358868985616e-09, 3.197926671666804e-08,
    1.879082322370048e-08, -2.4857126248016745e-07, -5.084465378687302e-08,
    1.7419821586224816e-06, -9.792625707303523e-07, -1.1438048033346894e-05,
    2.2387565714911816e-05, 5.164652974177416e-05, -0.00029015535246077655,
    0.000293714378044958, 0.0017556261651970652, -0.009746579683265262,
    0.02836227737211114, -0.05869339857664934, 0.09230432116428125,
    -0.10880393014244462, 0.08227673848999506, 0.0035854154854790257,
    -0.14024059858554525, 1.2375126308378275,
    1.6059043836821613e-10, 2.08767569878681e-09, 2.505210838544172e-08,
    2.755731922398589e-07, 2.7557319223985893e-06, 2.48015873015873e-05,
    0.0001984126984126984, 0.001388888888888889, 0.008333333333333333,
    0.041666666666666664, 0.16666666666666666, 0.5};
typedef const double __attribute__((address_space(4))) scalar_double;

// a b + c with c in scalar registers (the compiler's own choice, the
// two-operand form, first copies c into vector registers: as many cycles as
// the multiply-add)
__device__ inline double fma_sc(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
}

__device__ inline double erfc_exp64(double x, double xl, double* ex) {
    scalar_double* c = (scalar_double*)erfc_coef;
    asm volatile("" : "+s"(c));  // loaded here, not ahead of the caller's loop
    const double s = x * x;
    // exp(-s)
    const double n = rint(s * -1.4426950408889634);
    double r = fma(n, -0x1.62e42fefa39efp-1, -s);
    r = fma(n, -0x1.abc9e3b39803fp-56, r);
    double e = c[ERFC_NP];
#pragma unroll
    for (int k = 1; k < ERFC_NE; k++) e = fma_sc(e, r, c[ERFC_NP + k]);
    e = ldexp(fma(e * r, r, r) + 1.0, (int)n);
    e = fma(-fma(2.0 * x, xl, fma(x, x, -s)), e, e);
    const double a = x + 3.75, b = fma(2.0, x, 1.0);
    const double q = rcp_nr(a * b);
    const double t = (x - 3.75) * (q * b);
    double p = c[0];
#pragma unroll
    for (int k = 1; k < ERFC_NP; k++) p = fma_sc(p, t, c[k]);
    *ex = e;
    return e * (p * (q * a));
}

// ---- FP32 ---------------------------------------------------------------
// erfc(x) = exp(-x^2) * P(t), t = 1/(1 + x/2), x >= 0.  P is a degree-9
// weighted least-squares fit of the scaled complementary error function
// exp(x^2) erfc(x) on [0, 12] (max relative error 4e-8 in exact
// arithmetic, 3.3e-7 evaluated in FP32).  exp(-x^2) is shared with the
// Ewald / Wolf force term.
__device__ inline float erfc_scaled_poly(float x) {
    // hardware reciprocal (v_rcp_f32, ~1 ulp): the fit's error stays ~4e-7
    float t = __builtin_amdgcn_rcpf(1.0f + 0.5f * x);
    float p = -5.734027581e-02f;
    p = fmaf(p, t, 2.758059454e-01f);
    p = fmaf(p, t, -4.681025672e-01f);
    p = fmaf(p, t, 2.547098534e-01f);
    p = fmaf(p, t, -9.007769349e-03f);
    p = fmaf(p, t, 1.942188194e-01f);
    p = fmaf(p, t, 2.456883800e-01f);
    p = fmaf(p, t, 2.818937015e-01f);
    p = fmaf(p, t, 2.821360283e-01f);
    p = fmaf(p, t, -2.151000532e-06f);
    return p;
}

#define MSPMS_TWO_OVER_SQRTPI_F 1.1283791670955126f
