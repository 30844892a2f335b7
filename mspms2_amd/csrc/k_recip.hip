// k_recip.hip -- Ewald reciprocal space (FP64) on gfx950, as matrix products.
// Reference: src/frclong.c:988-1048.  For every k = 2*pi*(kx/Lx, ky/Ly,
// kz/Lz) with 0 < kx^2+ky^2+kz^2 <= KSQMAX:
//   S(k) = sum_i q_i exp(i k.r_i),  U_k = kvec |S(k)|^2,
//   F_i += 2 q_i (S_r sin(k.r_i) - S_i cos(k.r_i)) Vf kvec C k.
// With E_r(i) = exp(i (kx tx + ky ty)) of a row r = (kx, ky), t = 2 pi x / L,
// and c_n, s_n = cos, sin of n tz, the z components +n and -n share their
// products:
//   P_rn = sum_i q_i E_r c_n,  Q_rn = sum_i q_i E_r s_n,
//   S(r, +n) = P + i Q,  S(r, -n) = P - i Q,
// a product of the (2 rows) x (atoms) matrix (Re, Im of q E_r) with the
// (atoms) x (2 kmaxz) matrix (c_n, s_n).  The forces are the transpose: per
// row the four sums over n
//   U = sum a_n c_n + b_n s_n, V, and U', V' with the weight n,
// with E_r = C + i D, give D U + C V for the x and y components (times kx,
// ky) and D U' + C V' for z: a (4 rows) x (2 kmaxz) by (2 kmaxz) x (atoms)
// product.  Both run on the FP64 matrix instruction (v_mfma_f64_16x16x4).  Per
// row and n the first takes 4 multiply-adds an atom and the second 8, for the
// two k's +n and -n: 6 multiply-adds, 12 FLOP, per (k, atom) of the half space,
// and per (row, atom) 25 FLOP outside the products (E_r twice, the row's share
// of the forces).  There is no recurrence along kz, where a lane per
// (row, kz segment) and a lane per atom were bound by their chains and by LDS and
// scalar loads per product.
//
//   k_sk     one workgroup per (replica, chunk of atoms): power tables of 64
//            atoms at a time in LDS; a wave owns TW row tiles (8 rows = 16
//            matrix rows) and keeps their sums in registers over the chunk.
//            The sums go out in the registers' layout, per chunk (no atomics).
//   k_sred   per (row tile, quarter of it, kz tile): the chunks' sums in a
//            fixed order, U_k, and the force product's left matrix in the
//            layout in which k_kforce loads it.
//   k_kforce one workgroup per 16 G atoms; its waves share the row tiles (4
//            rows x {U, V, U', V'}); each atom's force is written once.
// Rows are sorted by their kz extent, so that short rows share tiles and the
// tiles past their extent are left out.
//
// Kernel times (us; before: a lane per (row, kz segment), per k and per atom):
//                                 k_sk        k_sred      k_kforce
//   98,304 sites, 8434 k       571 -> 130    57 -> 13    578 -> 169
//   12,288 sites, 1054 k      16.5 -> 10.5    5 -> 7    12.9 -> 9.1
//   648 sites, 61 k           17.3 -> 5.4   4.9 -> 4.9   4.1 -> 4.4
// At 98,304 sites the matrix instructions alone take about 60 and 130 us;
// k_sk is held by its LDS reads, k_kforce by the operations per (row, atom)
// between the products.  The small ones are launch and load latency.
#include "engine.h"
#include "../../include/mspms_gpu.h"

namespace {

struct cplx {
    double re, im;
};
__device__ inline cplx cmul(cplx a, cplx b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

typedef double d4 __attribute__((ext_vector_type(4)));

// D = A B + C on 16x16x4: lane l holds A[l & 15][l >> 4], B[l >> 4][l & 15]
// and, in register v, D[(l >> 4) + 4 v][l & 15].
__device__ inline d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One axis of the power tables of `na` atoms (of nt slots): row[n] = s e^n,
// n = n0 .. n0 + cnt - 1, in tab[atom * stride + off + n - n0]; entries past
// km are zero.
__device__ inline void fill_powers(double2* row, cplx e, double s, int n0, int cnt, int km) {
    cplx v = {s, 0.0};
    if (n0 == 1) v = cmul(v, e);
    for (int n = n0; n < n0 + cnt; n++) {
        row[n - n0] = n <= km ? make_double2(v.re, v.im) : make_double2(0.0, 0.0);
        v = cmul(v, e);
    }
}

// The table of an atom: x powers 0..KX, y powers 0..KY, z powers 1..8 NT
// (zero past the replica's kmaxz); KX, KY are the largest of all replicas.
// The stride is odd in 16-byte units, so that the four atoms of an
// operand's lanes fall on different banks.
struct TabShape {
    int yoff, zoff, stride;
};

template <int NT, int TW>
__global__ void __launch_bounds__(512) k_sk(const int4* __restrict__ work,
                                           const RepDev* __restrict__ reps,
                                           const KTileRow* __restrict__ trows, TabShape ts,
                                           const double* __restrict__ x,
                                           const double* __restrict__ y,
                                           const double* __restrict__ z,
                                           const int* __restrict__ atom_site,
                                           const SiteDev* __restrict__ sites,
                                           double* __restrict__ s_part, size_t s_stride,
                                           int ntile_max, double2* __restrict__ eatom,
                                           int natom) {
    extern __shared__ double2 tab[];
    const int4 wk = work[blockIdx.x];
    const RepDev& R = reps[wk.x];
    const int nw = blockDim.x >> 6, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m = lane & 15, kq = lane >> 4, comp = m & 1;
    // the rows of this lane's matrix row in the wave's tiles
    int xo[TW], yo[TW];
    bool neg[TW], two[TW];
    d4 acc[TW][NT];
    double s0[TW];
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const int t = w + i * nw;
        const KTileRow K = trows[(size_t)(R.ktile0 + (t < R.nktile ? t : 0)) * 8 + (m >> 1)];
        xo[i] = K.kx;
        yo[i] = ts.yoff + (K.ky < 0 ? -K.ky : K.ky);
        neg[i] = K.ky < 0;
        // rows come sorted by extent: the tile's first row has its largest
        two[i] = NT > 1 && __builtin_amdgcn_readfirstlane(K.nz) > 8;
        s0[i] = 0.0;
#pragma unroll
        for (int k = 0; k < NT; k++) acc[i][k] = d4{0.0, 0.0, 0.0, 0.0};
    }
    for (int b0 = 0; b0 < wk.w; b0 += 64) {
        const int a0 = wk.z + b0, na = min(64, wk.w - b0);
        if (b0 > 0) __syncthreads();  // the tables have been read
        // thread t -> (atom t & 63, axis t >> 6)
        for (int t = threadIdx.x; t < 3 * 64; t += blockDim.x) {
            const int a = t & 63, d = t >> 6;
            double s = 0.0, c = 1.0, q = 0.0;
            if (a < na) {
                const double* p = d == 0 ? x : (d == 1 ? y : z);
                sincos(R.twopi_l[d] * p[a0 + a], &s, &c);
                eatom[(size_t)d * natom + a0 + a] = make_double2(c, s);  // for k_kforce
                q = d == 0 ? sites[atom_site[a0 + a]].charge : 1.0;
            }
            double2* row = tab + a * ts.stride;
            if (d == 0)  // (the charge rides on the x powers)
                fill_powers(row, cplx{c, s}, q, 0, R.kmax[0] + 1, R.kmax[0]);
            else if (d == 1)
                fill_powers(row + ts.yoff, cplx{c, s}, 1.0, 0, R.kmax[1] + 1, R.kmax[1]);
            else
                fill_powers(row + ts.zoff, cplx{c, s}, 1.0, 1, 8 * NT, R.kmax[2]);
        }
        __syncthreads();
        const int nk = (na + 3) >> 2;
        for (int k = 0; k < nk; k++) {
            const double2* base = tab + (4 * k + kq) * ts.stride;
            double bz[NT];
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const double2 v = base[ts.zoff + 8 * j + (m >> 1)];
                bz[j] = comp ? v.y : v.x;
            }
#pragma unroll
            for (int i = 0; i < TW; i++) {
                if (w + i * nw >= R.nktile) continue;  // uniform
                const double2 X = base[xo[i]], Y = base[yo[i]];
                const double yi = neg[i] ? -Y.y : Y.y;
                // Re or Im of q exp(i (kx tx + ky ty))
                const double a = X.x * (comp ? yi : Y.x) + X.y * (comp ? Y.x : -yi);
                s0[i] += a;
                acc[i][0] = mfma(a, bz[0], acc[i][0]);
                if (NT > 1 && two[i]) acc[i][NT - 1] = mfma(a, bz[NT - 1], acc[i][NT - 1]);
            }
        }
    }
    double* out = s_part + (size_t)wk.y * s_stride;
#pragma unroll
    for (int i = 0; i < TW; i++) {
        const int t = w + i * nw;
        if (t >= R.nktile) continue;
#pragma unroll
        for (int k = 0; k < NT; k++) {
            if (k > 0 && !two[i]) continue;
#pragma unroll
            for (int v = 0; v < 4; v++)
                out[((size_t)(t * NT + k) * 4 + v) * 64 + lane] = acc[i][k][v];
        }
        double s = s0[i];
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (lane < 16) out[(size_t)ntile_max * NT * 256 + t * 16 + m] = s;
    }
}

// Workgroup (row tile, kz tile and quarter v): 64 sums of the accumulator
// register v by 16 groups of chunks, the groups added in order; then one
// thread per (row, n): S, U_k and the force matrix's entries.
constexpr int SRED_G = 16;

// the sum of p[c * stride], c = c0, c0 + SRED_G, ... < c1: up to 12 loads in
// flight (all that 192 chunks need), since each is a trip to memory (another
// XCD wrote it)
__device__ inline double sum_chunks(const double* __restrict__ p, size_t stride, int c0, int c1) {
    double s = 0.0;
    for (int c = c0; c < c1; c += 12 * SRED_G) {
        double v[12];
#pragma unroll
        for (int k = 0; k < 12; k++)
            v[k] = c + k * SRED_G < c1 ? p[(size_t)(c + k * SRED_G) * stride] : 0.0;
#pragma unroll
        for (int k = 0; k < 12; k++) s += v[k];
    }
    return s;
}

template <int NT>
__global__ void __launch_bounds__(64 * SRED_G) k_sred(
    const int* __restrict__ tile_rep, const RepDev* __restrict__ reps,
    const KTileRow* __restrict__ trows, const int* __restrict__ rep_chunk0,
    const double* __restrict__ s_part, size_t s_stride, int ntile_max,
    const double* __restrict__ kvec, double* __restrict__ uk, double* __restrict__ wmat,
    double2* __restrict__ w0) {
    __shared__ double sh[SRED_G][68], val[68];
    const int gt = blockIdx.x, v = blockIdx.y & 3, nt = blockIdx.y >> 2;
    const int r = tile_rep[gt];
    const RepDev& R = reps[r];
    const int t = gt - R.ktile0;
    if (nt > 0 && trows[(size_t)gt * 8].nz <= 8 * nt) return;  // uniform
    const int e = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int c0 = rep_chunk0[r], c1 = rep_chunk0[r + 1];
    const double* p = s_part + ((size_t)(t * NT + nt) * 4 + v) * 64 + e;
    sh[g][e] = sum_chunks(p, s_stride, c0 + g, c1);
    if (nt == 0 && e < 4) {
        // the n = 0 sums of the four matrix rows
        const double* p0 = s_part + (size_t)ntile_max * NT * 256 + t * 16 + 4 * v + e;
        sh[g][64 + e] = sum_chunks(p0, s_stride, c0 + g, c1);
    }
    __syncthreads();
    if (threadIdx.x < 64 + (nt == 0 ? 4 : 0)) {
        double q = sh[0][threadIdx.x];
#pragma unroll
        for (int k = 1; k < SRED_G; k++) q += sh[k][threadIdx.x];
        val[threadIdx.x] = q;
    }
    __syncthreads();
    // threads 0..15: (row 2 v + b, n); 16, 17: its n = 0
    if (threadIdx.x >= 18 || (threadIdx.x >= 16 && nt > 0)) return;
    const int b = threadIdx.x < 16 ? threadIdx.x >> 3 : threadIdx.x - 16;
    const int row8 = 2 * v + b;
    const KTileRow K = trows[(size_t)gt * 8 + row8];
    const double sc = 2.0 * R.vfactor * R.C;
    const int ft = 2 * gt + (row8 >> 2), rr = row8 & 3;
    if (threadIdx.x >= 16) {
        double2 o = make_double2(0.0, 0.0);
        if (K.k0 >= 0 && K.kz_lo <= 0) {
            const int k = K.k0 - K.kz_lo;
            const double sr = val[64 + 2 * b], si = val[64 + 2 * b + 1], kv = kvec[k];
            uk[k] = kv * (sr * sr + si * si);
            o = make_double2(sc * kv * sr, -(sc * kv * si));
        }
        w0[ft * 4 + rr] = o;
        return;
    }
    const int j = threadIdx.x & 7, n = 8 * nt + j + 1;
    if (K.k0 < 0 || n > K.nz) return;
    const double rp = val[2 * b * 16 + 2 * j], rq = val[2 * b * 16 + 2 * j + 1];
    const double ip = val[(2 * b + 1) * 16 + 2 * j], iq = val[(2 * b + 1) * 16 + 2 * j + 1];
    double ap, bp, am = 0.0, bm = 0.0;  // force coefficients of +n and -n
    {
        const int k = K.k0 + (n - K.kz_lo);
        const double sr = rp - iq, si = ip + rq, kv = kvec[k];
        uk[k] = kv * (sr * sr + si * si);
        ap = sc * kv * sr;
        bp = sc * kv * si;
    }
    if (-n >= K.kz_lo) {
        const int k = K.k0 + (-n - K.kz_lo);
        const double sr = rp + iq, si = ip - rq, kv = kvec[k];
        uk[k] = kv * (sr * sr + si * si);
        am = sc * kv * sr;
        bm = sc * kv * si;
    }
    // columns 2 (n - 1) (cos) and 2 (n - 1) + 1 (sin) of the four rows
    double* o = wmat + ((size_t)ft * (4 * NT) + (n - 1) / 2) * 64 + rr + 32 * ((n - 1) & 1);
    o[0] = ap + am;
    o[16] = bp - bm;
    o[4] = -(bp + bm);
    o[16 + 4] = ap - am;
    o[8] = n * (ap - am);
    o[16 + 8] = n * (bp + bm);
    o[12] = -(n * (bp - bm));
    o[16 + 12] = n * (ap + am);
}

// work: (rep, first atom, atoms <= 16 G).  Wave w takes the tiles w, w +
// KF_W, ... of four rows; lane l has atom l & 15 of each group of 16 and row l >> 4,
// and the matrix product leaves that row's U, V, U', V' in its four result
// registers.
// GRAD: also dU_fourier/dq_i = sum_k (A_k cos + B_k sin) = C U - D V, added
// into gq.
// The next tile's left matrix is loaded while this one's products run.
template <bool GRAD, int NT, int G, int KF_W>
__global__ void __launch_bounds__(64 * KF_W) k_kforce(
    const int4* __restrict__ work, const RepDev* __restrict__ reps,
    const KTileRow* __restrict__ trows, TabShape ts, const double* __restrict__ wmat,
    const double2* __restrict__ w0, const int* __restrict__ atom_site,
    const SiteDev* __restrict__ sites, double* fx, double* fy, double* fz, double* gq,
    const double2* __restrict__ eatom, int natom) {
    constexpr int NA = 16 * G, NF = GRAD ? 4 : 3, KK = 4 * NT;
    extern __shared__ double2 tab[];
    __shared__ double sh[KF_W][NF][NA];
    const int4 wk = work[blockIdx.x];
    const RepDev& R = reps[wk.x];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int t = threadIdx.x; t < 3 * NA; t += 64 * KF_W) {
        const int a = t % NA, d = t / NA;
        // atoms past the last one: e = 1, their sums are dropped
        const double2 v = a < wk.z ? eatom[(size_t)d * natom + wk.y + a] : make_double2(1.0, 0.0);
        const cplx e = {v.x, v.y};
        double2* row = tab + a * ts.stride;
        if (d == 0)
            fill_powers(row, e, 1.0, 0, R.kmax[0] + 1, R.kmax[0]);
        else if (d == 1)
            fill_powers(row + ts.yoff, e, 1.0, 0, R.kmax[1] + 1, R.kmax[1]);
        else
            fill_powers(row + ts.zoff, e, 1.0, 1, 8 * NT, R.kmax[2]);
    }
    __syncthreads();
    const int m = lane & 15, rq = lane >> 4;
    // the right matrix of every group: element (column 4 k + rq, atom m)
    double bz[G][KK];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int k = 0; k < KK; k++) {
            const double2 v = tab[(16 * g + m) * ts.stride + ts.zoff + 2 * k + (rq >> 1)];
            bz[g][k] = (rq & 1) ? v.y : v.x;
        }
    double f[G][NF];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int d = 0; d < NF; d++) f[g][d] = 0.0;
    const int nft = 2 * R.nktile, ft0 = 2 * R.ktile0;
    KTileRow Kn{};
    double2 cn = make_double2(0.0, 0.0);
    double wn[KK];
    auto fetch = [&](int t) {
        Kn = trows[(size_t)(ft0 + t) * 4 + rq];
        cn = w0[(ft0 + t) * 4 + rq];
        const double* wp = wmat + (size_t)(ft0 + t) * KK * 64 + lane;
#pragma unroll
        for (int k = 0; k < KK; k++) wn[k] = wp[k * 64];
    };
    if (w < nft) fetch(w);
    for (int t = w; t < nft; t += KF_W) {
        const KTileRow K = Kn;
        // the tile's first row has its largest extent
        const int kk = (__builtin_amdgcn_readfirstlane(K.nz) + 1) >> 1;
        d4 acc[G];
#pragma unroll
        for (int g = 0; g < G; g++) acc[g] = d4{cn.x, cn.y, 0.0, 0.0};
        double wc[KK];
#pragma unroll
        for (int k = 0; k < KK; k++) wc[k] = wn[k];
        if (t + KF_W < nft) fetch(t + KF_W);
#pragma unroll
        for (int k = 0; k < KK; k++) {
            if (k >= kk) break;  // uniform
#pragma unroll
            for (int g = 0; g < G; g++) acc[g] = mfma(wc[k], bz[g][k], acc[g]);
        }
        const int ay = ts.yoff + (K.ky < 0 ? -K.ky : K.ky);
        const double dkx = K.kx, dky = K.ky;
#pragma unroll
        for (int g = 0; g < G; g++) {
            const double2* base = tab + (16 * g + m) * ts.stride;
            const double2 X = base[K.kx], Y = base[ay];
            const double yi = K.ky < 0 ? -Y.y : Y.y;
            const double C = X.x * Y.x - X.y * yi, D = X.x * yi + X.y * Y.x;
            const double s = D * acc[g][0] + C * acc[g][1];
            f[g][0] += dkx * s;
            f[g][1] += dky * s;
            f[g][2] += D * acc[g][2] + C * acc[g][3];
            if (GRAD) f[g][NF - 1] += C * acc[g][0] - D * acc[g][1];
        }
    }
    // the four rows of a tile sit in lanes 16 apart; then the waves in order
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int d = 0; d < NF; d++) {
            double s = f[g][d];
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            if (rq == 0) sh[w][d][16 * g + m] = s;
        }
    __syncthreads();
    const int a = threadIdx.x;
    if (a >= wk.z || a >= NA) return;
    double s[NF];
#pragma unroll
    for (int d = 0; d < NF; d++) {
        s[d] = sh[0][d][a];
#pragma unroll
        for (int k = 1; k < KF_W; k++) s[d] += sh[k][d][a];
    }
    const int i = wk.y + a;
    const double q = sites[atom_site[i]].charge;
    fx[i] += q * s[0] * R.twopi_l[0];
    fy[i] += q * s[1] * R.twopi_l[1];
    fz[i] += q * s[2] * R.twopi_l[2];
    if (GRAD) gq[i] += s[NF - 1];
}

TabShape tab_shape(const RecipBufs& rb) {
    TabShape t;
    t.yoff = rb.kx_max + 1;
    t.zoff = t.yoff + rb.ky_max + 1;
    t.stride = (t.zoff + 8 * rb.nt) | 1;
    return t;
}

}  // namespace

// Tiles of 8 kz (16 columns) that the largest kmaxz needs.
int recip_kz_tiles(int kmaxz) { return kmaxz <= 8 ? 1 : 2; }

// Atoms per workgroup of k_sk: 64 (one table) up to 512 tables in all, beyond
// that as many tables as leave 256 workgroups, plus at most one partial chunk
// for each replica (a chunk holds atoms of one replica, so there are never
// fewer workgroups than replicas).  More atoms per workgroup mean fewer partial
// sums to write and read back (98,304 sites at kmax 16: 213 KB each), fewer
// than one workgroup per CU leaves CUs idle.  Many small replicas, whose
// workgroups then run over a whole replica, fare alike: NVE steps of 300 boxes
// of 180 sites 232 us and 238 with one table a workgroup, 200 of 330 sites 232
// and 228, 1000 of 180 sites 721 and 745.
int recip_s_chunk(long blocks64) {
    return 64 * (int)(blocks64 <= 512 ? 1 : (blocks64 + 255) / 256);
}

// Atoms per workgroup of k_kforce: 64 where that still fills the chip with
// four workgroups per CU, else 32 (12,288 sites: 384 workgroups).
int recip_f_group(long natom) { return natom >= 65536 ? 64 : 32; }

void launch_recip_s(const LaunchCtx& c, const RecipBufs& rb, const double* x, const double* y,
                    const double* z) {
    const TabShape ts = tab_shape(rb);
    const size_t lds = (size_t)64 * ts.stride * sizeof(double2);
    // tiles per wave: the fewest of the built counts that need at most 8 waves
    // (69 tiles at most: KMAX 16 without the KSQMAX sphere)
    const int need = (rb.ntile_max + 7) / 8;
#define SK(NT, TW)                                                                             \
    hipLaunchKernelGGL((k_sk<NT, TW>), dim3(rb.nwork_s),                                          \
                       dim3(64 * std::max(3, (rb.ntile_max + TW - 1) / TW)), lds, c.stream,       \
                       rb.work_s, c.reps, rb.trows, ts, x, y, z, c.atom_site, c.sites, rb.s_part, \
                       rb.s_stride, rb.ntile_max, rb.eatom, c.natom)
#define SK_NT(NT)                                                                              \
    do {                                                                                       \
        if (need <= 1)                                                                         \
            SK(NT, 1);                                                                         \
        else if (need <= 2)                                                                    \
            SK(NT, 2);                                                                         \
        else if (need <= 4)                                                                    \
            SK(NT, 4);                                                                         \
        else if (need <= 7)                                                                    \
            SK(NT, 7);                                                                         \
        else                                                                                   \
            SK(NT, 9);                                                                         \
    } while (0)
    if (rb.nt == 1) {
        SK_NT(1);
        hipLaunchKernelGGL(k_sred<1>, dim3(rb.ntile, 4), dim3(64 * SRED_G), 0, c.stream,
                           rb.tile_rep, c.reps, rb.trows, rb.rep_chunk0, rb.s_part, rb.s_stride,
                           rb.ntile_max, rb.kvec, rb.uk, rb.wmat, rb.w0);
    } else {
        SK_NT(2);
        hipLaunchKernelGGL(k_sred<2>, dim3(rb.ntile, 8), dim3(64 * SRED_G), 0, c.stream,
                           rb.tile_rep, c.reps, rb.trows, rb.rep_chunk0, rb.s_part, rb.s_stride,
                           rb.ntile_max, rb.kvec, rb.uk, rb.wmat, rb.w0);
    }
#undef SK_NT
#undef SK
}

void launch_recip_f(const LaunchCtx& c, const RecipBufs& rb, double* fx, double* fy, double* fz,
                    double* gq) {
    const TabShape ts = tab_shape(rb);
    const size_t lds = (size_t)rb.f_group * ts.stride * sizeof(double2);
#define KFORCE(GR, NT, G, W)                                                                   \
    hipLaunchKernelGGL((k_kforce<GR, NT, G, W>), dim3(rb.nwork_f), dim3(64 * W), lds, c.stream,   \
                       rb.work_f, c.reps, rb.trows, ts, rb.wmat, rb.w0, c.atom_site, c.sites, fx, \
                       fy, fz, gq, rb.eatom, c.natom)
#define KFORCE_G(GR, NT)                                                                       \
    do {                                                                                       \
        if (rb.f_group == 64)                                                                  \
            KFORCE(GR, NT, 4, 4);                                                                 \
        else                                                                                   \
            KFORCE(GR, NT, 2, 8);                                                                 \
    } while (0)
    if (gq) {
        if (rb.nt == 1)
            KFORCE_G(true, 1);
        else
            KFORCE_G(true, 2);
    } else {
        if (rb.nt == 1)
            KFORCE_G(false, 1);
        else
            KFORCE_G(false, 2);
    }
#undef KFORCE_G
#undef KFORCE
}
