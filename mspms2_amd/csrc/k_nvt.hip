// k_nvt.hip -- Nose-Hoover NVT RESPA step on gfx950: vver_nh_3
// (src/nvtnh.c:11-221), two thermostats (outer: ss, ps, qq; inner: sss,
// pss, qqs) as in Frenkel and Smit.
//
// The end-of-(sub)step half kick is implicit: v' = v + h (u - p' v') with
// u = f / m and p' following from sum m v'^2, which the reference solves by
// a Newton iteration over all atoms (src/nvtnh.c:61-157, :167-252).  Its
// iterates are v_k = a_k v + b_k u with the same a_k, b_k for every atom
// (v_0 = v, and each pass maps v_k to (v + h u - h dp v_k) / (1 + p h)), so
// the sums that a pass needs follow from
//     A = sum m v.v,   B = sum v.f,   C = sum f.f / m
// and the iteration runs on (a, b, p) alone: one sum over the atoms and one
// pass that applies a v + b u, where the reference sweeps the atoms twice
// per pass.  With the sweeps in one workgroup per replica the 12,288-site
// water step took 1500 us (8 inner solves of 126 us); this way it takes
// 160 us, and the LJ-864 step 47 us where it took 75.
//
// The atoms of a replica are spread over workgroups; a kernel's sums are
// stored per workgroup and every workgroup of the next kernel adds them up
// again in workgroup order, so that all hold the same bits and the run is
// deterministic.  Kernels of a step, nstep_inner times the first:
//   k_nvt_sub    [the previous inner solve; on the first substep the outer
//                half kick instead], the inner half kick and drift, frcshort
//                of the workgroup's molecules, A, B, C of the new state
//                (and on the first substep sum m v^2 before the inner kick)
//   frclong
//   k_nvt_close  the last inner solve; A, B, C with the long forces
//   k_nvt_outer  the outer solve; ukin, tinst, thermostat energies (:254-263)
// Molecules of more than four sites or terms run a substep as k_nvt_kick,
// k_bonded, k_nvt_sums.  The thermostat variables move from kernel to
// kernel in two alternating records per replica; the caller's state is read
// by the first kernel and written by the last.
//
// Arithmetic is FP64 in the reference's expression order where it has one
// (no contraction).  The Newton loop ends as the reference's does: after 100
// passes or when |(p_new - p_old) / p_new| <= 1e-10 -- the reference's
// per-atom test reads the unused element natom (loop index left at natom,
// zero), so 0/0 is never greater than the tolerance and only the thermostat
// test decides.
#include "engine.h"
#include "inner_terms.h"
#include "wave.h"
#include "../../include/mspms_gpu.h"

namespace {

constexpr int NVT_AT = 256;           // atoms (and threads) per workgroup of the atom passes
constexpr double NVT_ERR = 1.0e-10;   // src/nvtnh.c:19

// the scalars of one solve: v' = a v + b u, the momentum p and sum m v'^2
struct Solve {
    double p, a, b, s2;
};

// the reference's Newton iteration on the sums A, B, C of (v, u)
__device__ Solve nvt_newton(double A, double B, double C, double p0, double q, double g,
                            double treq, double dt, double h) {
#pragma clang fp contract(off)
    Solve s = {p0, 1.0, 0.0, A};
    bool ready = false;
    for (int iter = 0; !ready && iter < 100; iter++) {
        const double po = s.p;
        // b_i of the reference: -h (u - po v_k) - (v - v_k) = bv v + bu u
        const double bv = h * po * s.a + (s.a - 1.0);
        const double bu = h * po * s.b + (s.b - h);
        double delp = dt / q * (s.a * bv * A + (s.a * bu + s.b * bv) * B + s.b * bu * C);
        const double di = -(po * h + 1.0);
        delp = delp - di * ((-s.s2 + g * treq) * h / q - (p0 - po));
        delp = delp / (-dt * h * s.s2 / q + di);
        s.a = s.a + (bv + h * s.a * delp) / di;
        s.b = s.b + (bu + h * s.b * delp) / di;
        s.s2 = s.a * s.a * A + 2.0 * s.a * s.b * B + s.b * s.b * C;
        s.p = po + delp;
        ready = !(fabs((s.p - po) / s.p) > NVT_ERR);
    }
    return s;
}

// the workgroup's sum of v, in every thread; sh: NT / 64 entries
template <int NT>
__device__ inline double4 wg_sum4(double4 v, double4* sh) {
    v.x = wave_sum64(v.x);
    v.y = wave_sum64(v.y);
    v.z = wave_sum64(v.z);
    v.w = wave_sum64(v.w);
    if (NT == 64) return v;
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double4 t = sh[0];
#pragma unroll
    for (int k = 1; k < NT / 64; k++) {
        t.x += sh[k].x;
        t.y += sh[k].y;
        t.z += sh[k].z;
        t.w += sh[k].w;
    }
    __syncthreads();
    return t;
}

// the sums that the replica's workgroups stored, in workgroup order (every
// thread of every workgroup gets the same bits)
template <int NT>
__device__ inline double4 part_sum(const double4* __restrict__ part, int2 blk, double4* sh) {
    double4 s = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int i = threadIdx.x; i < blk.y; i += NT) {
        const double4 p = part[blk.x + i];
        s.x += p.x;
        s.y += p.y;
        s.z += p.z;
        s.w += p.w;
    }
    return wg_sum4<NT>(s, sh);
}

// the inner solve of the substep whose sums are t (first: that substep was
// the step's first, whose sum m v^2 before its kick is t.w)
__device__ Solve inner_solve(const mspms_nvt_state& S, const NvtScal& in, double4 t, bool first,
                             const NvtTimes& T, NvtScal& out) {
#pragma clang fp contract(off)
    const double s2 = first ? t.w : in.s2;
    out = in;
    out.sss = in.sss + in.pss * T.delts + (s2 - S.ggs * S.treq) * T.delts_sqby2 / S.qqs;
    const double p = in.pss + (s2 - S.ggs * S.treq) * T.deltsby2 / S.qqs;
    const Solve r = nvt_newton(t.x, t.y, t.z, p, S.qqs, S.ggs, S.treq, T.delts, T.deltsby2);
    out.pss = r.p;
    out.s2 = r.s2;
    return r;
}

// what every kernel of a substep does first: the previous substep's solve
// or, on the step's first substep (ll 0), the caller's state
template <int NT>
__device__ Solve enter(const NvtArgs& P, int r, int ll, bool lead, double4* sh, NvtScal& sc) {
    const mspms_nvt_state& S = P.st[r];
    Solve sv = {0.0, 1.0, 0.0, 0.0};
    if (ll == 0) {
        sc.ss = S.ss;
        sc.ps = S.ps;
        sc.sss = S.sss;
        sc.pss = S.pss;
        sc.s2 = 0.0;
    } else {
        const double4 t = part_sum<NT>(P.part_in, P.blk_in[r], sh);
        sv = inner_solve(S, P.scal_in[r], t, ll == 1, P.t, sc);
    }
    if (lead && threadIdx.x == 0) P.scal_out[r] = sc;
    return sv;
}

// One atom's part of a substep: the previous solve or the outer half kick
// (FIRST), then the inner half kick and drift.  m2: the atom's m v^2 before
// the inner kick.
template <bool FIRST>
__device__ inline void kick_drift(const NvtArgs& P, int i, const Solve& sv, const NvtScal& sc,
                                  double r_mass, double3& X, double3& V, const double3& F,
                                  double& m2) {
#pragma clang fp contract(off)
    if (FIRST) {
        V.x = V.x + P.t.deltby2 * (P.fl[i] * r_mass - sc.ps * V.x);
        V.y = V.y + P.t.deltby2 * (P.fl[P.n + i] * r_mass - sc.ps * V.y);
        V.z = V.z + P.t.deltby2 * (P.fl[2 * P.n + i] * r_mass - sc.ps * V.z);
        m2 = (V.x * V.x + V.y * V.y + V.z * V.z) / r_mass;
    } else {
        V.x = sv.a * V.x + sv.b * (F.x * r_mass);
        V.y = sv.a * V.y + sv.b * (F.y * r_mass);
        V.z = sv.a * V.z + sv.b * (F.z * r_mass);
        m2 = 0.0;
    }
    V.x = V.x + P.t.deltsby2 * (F.x * r_mass - sc.pss * V.x);
    V.y = V.y + P.t.deltsby2 * (F.y * r_mass - sc.pss * V.y);
    V.z = V.z + P.t.deltsby2 * (F.z * r_mass - sc.pss * V.z);
    X.x = X.x + P.t.delts * V.x;
    X.y = X.y + P.t.delts * V.y;
    X.z = X.z + P.t.delts * V.z;
}

__device__ inline double3 load3(const double* p, size_t n, int i) {
    return make_double3(p[i], p[n + i], p[2 * n + i]);
}
__device__ inline void store3(double* p, size_t n, int i, const double3& v) {
    p[i] = v.x;
    p[n + i] = v.y;
    p[2 * n + i] = v.z;
}

// One substep of the workgroup's 64 G molecules of at most NW sites and NW
// bonded terms: wave w of a group owns site w of its 64 molecules (lane =
// molecule) and computes their term w into its own LDS copy of their forces,
// as k_respa_inner_tw does; a site's force is the sum of the copies in term
// order.
template <int NW, int G, bool FIRST>
__global__ void __launch_bounds__(64 * NW * G) k_nvt_sub(NvtArgs P, int ll, int last) {
    constexpr int NT = 64 * NW * G;
    __shared__ double4 sh[NT / 64];
    __shared__ double lx[G][NW * 64], ly[G][NW * 64], lz[G][NW * 64];
    __shared__ double cfx[G][NW][NW * 64], cfy[G][NW][NW * 64], cfz[G][NW][NW * 64];
    const int4 wk = P.work[blockIdx.x];
    const int r = wk.x;
    if (P.active && !P.active[r]) return;  // a frozen replica (whole workgroup)
    NvtScal sc;
    const Solve sv = enter<NT>(P, r, ll, wk.w != 0, sh, sc);
    const int wave = threadIdx.x >> 6, mi = threadIdx.x & 63, g = wave / NW, w = wave % NW;
    const int k = g * 64 + mi;
    const bool live = k < wk.z;
    const int m = wk.y + k;
    int na = 0, a0 = 0, nbt = 0;
    TermDev T{};
    if (live) {
        const MolDev M = P.mols[m];
        na = M.natom;
        a0 = M.atom0;
        nbt = M.nbterm;
        if (w < nbt) T = P.terms[M.bterm0 + w];
    }
    const bool own = live && w < na, term = live && w < nbt;
    const int i = a0 + w, sl = w * 64 + mi;
    double r_mass = 0.0, m2 = 0.0;
    double3 X{}, V{}, F{};
    if (own) {
        r_mass = P.rmass[i];
        X = load3(P.x, P.n, i);
        V = load3(P.v, P.n, i);
        F = load3(P.fs, P.n, i);
        kick_drift<FIRST>(P, i, sv, sc, r_mass, X, V, F, m2);
        lx[g][sl] = X.x;
        ly[g][sl] = X.y;
        lz[g][sl] = X.z;
    }
#pragma unroll
    for (int c = 0; c < NW; c++) {
        cfx[g][w][c * 64 + mi] = 0.0;
        cfy[g][w][c * 64 + mi] = 0.0;
        cfz[g][w][c * 64 + mi] = 0.0;
    }
    __syncthreads();
    double e[4] = {0.0, 0.0, 0.0, 0.0}, vir = 0.0;
    if (term) {
        double u = 0.0;
        int sing = 0;
        const int cls = bonded_term_inner(T, mi, lx[g], ly[g], lz[g], cfx[g][w], cfy[g][w],
                                          cfz[g][w], &u, &vir, &sing, 64);
        if (sing) atomicOr(&P.status->flags, ST_SINGULAR);
        e[cls] = u;
    }
    __syncthreads();
    double4 t = make_double4(0.0, 0.0, 0.0, m2);
    if (own) {
#pragma clang fp contract(off)
        F = make_double3(0.0, 0.0, 0.0);
#pragma unroll
        for (int c = 0; c < NW; c++) {
            F.x += cfx[g][c][sl];
            F.y += cfy[g][c][sl];
            F.z += cfz[g][c][sl];
        }
        store3(P.x, P.n, i, X);
        store3(P.v, P.n, i, V);
        store3(P.fs, P.n, i, F);
        t.x = (V.x * V.x + V.y * V.y + V.z * V.z) / r_mass;
        t.y = V.x * F.x + V.y * F.y + V.z * F.z;
        t.z = (F.x * F.x + F.y * F.y + F.z * F.z) * r_mass;
    }
    t = wg_sum4<NT>(t, sh);
    if (threadIdx.x == 0) P.part_out[blockIdx.x] = t;
    if (!last) return;  // uniform
    // the last substep's bonded energies, in term order (wg_sum4's barriers
    // have freed the force copies)
    if constexpr (NW == 1) {
        if (live) {
            double* ep = P.epart + (size_t)m * 5;
            for (int c = 0; c < 4; c++) ep[c] = e[c];
            ep[4] = vir;
        }
    } else {
        static_assert(NW >= 3, "the energies' copies fit the force copies");
        double* le = &cfx[g][0][0];  // [3][NW][64]
        double* lf = &cfy[g][0][0];  // [2][NW][64]
#pragma unroll
        for (int c = 0; c < 3; c++) le[(c * NW + w) * 64 + mi] = e[c];
        lf[w * 64 + mi] = e[3];
        lf[(NW + w) * 64 + mi] = vir;
        __syncthreads();
        if (live && w == 0) {
            double* ep = P.epart + (size_t)m * 5;
#pragma unroll
            for (int c = 0; c < 5; c++) {
                const double* q = c < 3 ? le + c * NW * 64 : lf + (c - 3) * NW * 64;
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < NW; d++) s += q[d * 64 + mi];
                ep[c] = s;
            }
        }
    }
}

// The substep of larger molecules, around k_bonded: kick and drift ...
template <bool FIRST>
__global__ void __launch_bounds__(NVT_AT) k_nvt_kick(NvtArgs P, int ll) {
    __shared__ double4 sh[NVT_AT / 64];
    const int4 wk = P.work[blockIdx.x];
    const int r = wk.x;
    if (P.active && !P.active[r]) return;
    NvtScal sc;
    const Solve sv = enter<NVT_AT>(P, r, ll, wk.w != 0, sh, sc);
    double m2 = 0.0;
    if ((int)threadIdx.x < wk.z) {
        const int i = wk.y + threadIdx.x;
        double3 X = load3(P.x, P.n, i), V = load3(P.v, P.n, i);
        const double3 F = load3(P.fs, P.n, i);
        kick_drift<FIRST>(P, i, sv, sc, P.rmass[i], X, V, F, m2);
        store3(P.x, P.n, i, X);
        store3(P.v, P.n, i, V);
    }
    const double4 t = wg_sum4<NVT_AT>(make_double4(0.0, 0.0, 0.0, m2), sh);
    if (threadIdx.x == 0) P.part_out[blockIdx.x].w = t.w;
}

// ... and the sums with the new forces
__global__ void __launch_bounds__(NVT_AT) k_nvt_sums(NvtArgs P) {
#pragma clang fp contract(off)
    __shared__ double4 sh[NVT_AT / 64];
    const int4 wk = P.work[blockIdx.x];
    if (P.active && !P.active[wk.x]) return;
    double4 t = make_double4(0.0, 0.0, 0.0, 0.0);
    if ((int)threadIdx.x < wk.z) {
        const int i = wk.y + threadIdx.x;
        const double r_mass = P.rmass[i];
        const double3 V = load3(P.v, P.n, i), F = load3(P.fs, P.n, i);
        t.x = (V.x * V.x + V.y * V.y + V.z * V.z) / r_mass;
        t.y = V.x * F.x + V.y * F.y + V.z * F.z;
        t.z = (F.x * F.x + F.y * F.y + F.z * F.z) * r_mass;
    }
    t = wg_sum4<NVT_AT>(t, sh);
    if (threadIdx.x == 0) {
        double4* o = P.part_out + blockIdx.x;
        o->x = t.x;
        o->y = t.y;
        o->z = t.z;
    }
}

// The last inner solve, and the sums of the outer one
__global__ void __launch_bounds__(NVT_AT) k_nvt_close(NvtArgs P, int ll) {
#pragma clang fp contract(off)
    __shared__ double4 sh[NVT_AT / 64];
    const int4 wk = P.work[blockIdx.x];
    const int r = wk.x;
    if (P.active && !P.active[r]) return;
    NvtScal sc;
    const Solve sv = enter<NVT_AT>(P, r, ll, wk.w != 0, sh, sc);
    double4 t = make_double4(0.0, 0.0, 0.0, 0.0);
    if ((int)threadIdx.x < wk.z) {
        const int i = wk.y + threadIdx.x;
        const double r_mass = P.rmass[i];
        double3 V = load3(P.v, P.n, i);
        const double3 F = load3(P.fs, P.n, i), L = load3(P.fl, P.n, i);
        V.x = sv.a * V.x + sv.b * (F.x * r_mass);
        V.y = sv.a * V.y + sv.b * (F.y * r_mass);
        V.z = sv.a * V.z + sv.b * (F.z * r_mass);
        store3(P.v, P.n, i, V);
        t.x = (V.x * V.x + V.y * V.y + V.z * V.z) / r_mass;
        t.y = V.x * L.x + V.y * L.y + V.z * L.z;
        t.z = (L.x * L.x + L.y * L.y + L.z * L.z) * r_mass;
    }
    t = wg_sum4<NVT_AT>(t, sh);
    if (threadIdx.x == 0) P.part_out[blockIdx.x] = t;
}

// The outer solve and the step's thermostat outputs
__global__ void __launch_bounds__(NVT_AT) k_nvt_outer(NvtArgs P, double* __restrict__ ukin) {
#pragma clang fp contract(off)
    __shared__ double4 sh[NVT_AT / 64];
    const int4 wk = P.work[blockIdx.x];
    const int r = wk.x;
    if (P.active && !P.active[r]) return;
    const double4 t = part_sum<NVT_AT>(P.part_in, P.blk_in[r], sh);
    // the fields that the lead workgroup writes below are read from sc only
    const NvtScal sc = P.scal_in[r];
    mspms_nvt_state* S = P.st + r;
    const double treq = S->treq, qq = S->qq, gg = S->gg;
    // src/nvtnh.c:161-162, with the sum m v^2 the last inner solve left
    const double ss = sc.ss + sc.ps * P.t.delt + (sc.s2 - gg * treq) * P.t.delt_sqby2 / qq;
    const double p = sc.ps + (sc.s2 - gg * treq) * P.t.deltby2 / qq;
    const Solve sv = nvt_newton(t.x, t.y, t.z, p, qq, gg, treq, P.t.delt, P.t.deltby2);
    if ((int)threadIdx.x < wk.z) {
        const int i = wk.y + threadIdx.x;
        const double r_mass = P.rmass[i];
        double3 V = load3(P.v, P.n, i);
        const double3 L = load3(P.fl, P.n, i);
        V.x = sv.a * V.x + sv.b * (L.x * r_mass);
        V.y = sv.a * V.y + sv.b * (L.y * r_mass);
        V.z = sv.a * V.z + sv.b * (L.z * r_mass);
        store3(P.v, P.n, i, V);
    }
    if (!wk.w || threadIdx.x != 0) return;
    S->sss = sc.sss;
    S->pss = sc.pss;
    S->unhtss = (sc.pss * sc.pss * S->qqs) / 2.0 + S->ggs * treq * sc.sss;
    S->ss = ss;
    S->ps = sv.p;
    const double uk = sv.s2 / 2.0;
    S->ukin = uk;
    S->unhts = (sv.p * sv.p * qq) / 2.0 + gg * treq * ss;
    S->tinst = 2.0 * uk / S->nfree;
    if (ukin) ukin[r] = uk;
}

}  // namespace

// Molecules per workgroup of the substep kernel, and whether the molecules
// fit it (one site and term per wave); larger ones go by atoms.
int nvt_mols_per_block(int max_mol_atoms, int max_mol_terms) {
    if (max_mol_atoms <= 1 && max_mol_terms <= 1) return 256;
    if (max_mol_atoms <= 4 && max_mol_terms <= 4) return 64;
    return 0;
}
int nvt_atoms_per_block() { return NVT_AT; }

void launch_nvt_substep(const LaunchCtx& c, const NvtPlan& N, const SpeciesDev* species, NvtArgs P,
                        int ll, int last) {
    P.scal_in = N.scal + (size_t)((ll + 1) & 1) * c.nrep;
    P.scal_out = N.scal + (size_t)(ll & 1) * c.nrep;
    P.part_in = N.part + (size_t)((ll + 1) & 1) * N.npart;
    P.part_out = N.part + (size_t)(ll & 1) * N.npart;
    const bool by_mol = N.nwork_m > 0;
    P.work = by_mol ? N.work_m : N.work_a;
    P.blk_in = by_mol ? N.blk_m : N.blk_a;
#define NVT_SUB(NW, G)                                                                       \
    do {                                                                                     \
        if (ll == 0)                                                                         \
            hipLaunchKernelGGL((k_nvt_sub<NW, G, true>), dim3(N.nwork_m), dim3(64 * NW * G), 0,  \
                               c.stream, P, ll, last);                                       \
        else                                                                                 \
            hipLaunchKernelGGL((k_nvt_sub<NW, G, false>), dim3(N.nwork_m), dim3(64 * NW * G), 0, \
                               c.stream, P, ll, last);                                       \
    } while (0)
    if (by_mol) {
        if (c.max_mol_atoms <= 1)
            NVT_SUB(1, 4);
        else if (c.max_mol_atoms <= 3 && c.max_mol_terms <= 3)
            NVT_SUB(3, 1);
        else
            NVT_SUB(4, 1);
        return;
    }
#undef NVT_SUB
    if (ll == 0)
        hipLaunchKernelGGL(k_nvt_kick<true>, dim3(N.nwork_a), dim3(NVT_AT), 0, c.stream, P, ll);
    else
        hipLaunchKernelGGL(k_nvt_kick<false>, dim3(N.nwork_a), dim3(NVT_AT), 0, c.stream, P, ll);
    launch_bonded(c, species, P.terms, P.x, P.x + P.n, P.x + 2 * P.n, P.fs, P.fs + P.n,
                  P.fs + 2 * P.n, P.epart);
    hipLaunchKernelGGL(k_nvt_sums, dim3(N.nwork_a), dim3(NVT_AT), 0, c.stream, P);
}

void launch_nvt_outer(const LaunchCtx& c, const NvtPlan& N, NvtArgs P, int nstep_inner,
                      double* ukin) {
    const int ll = nstep_inner;
    P.work = N.work_a;
    P.blk_in = N.nwork_m > 0 ? N.blk_m : N.blk_a;
    P.scal_in = N.scal + (size_t)((ll + 1) & 1) * c.nrep;
    P.scal_out = N.scal + (size_t)(ll & 1) * c.nrep;
    P.part_in = N.part + (size_t)((ll + 1) & 1) * N.npart;
    P.part_out = N.part + (size_t)(ll & 1) * N.npart;
    hipLaunchKernelGGL(k_nvt_close, dim3(N.nwork_a), dim3(NVT_AT), 0, c.stream, P, ll);
    P.blk_in = N.blk_a;
    P.scal_in = P.scal_out;
    P.part_in = P.part_out;
    hipLaunchKernelGGL(k_nvt_outer, dim3(N.nwork_a), dim3(NVT_AT), 0, c.stream, P, ukin);
}
