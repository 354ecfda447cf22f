// Training outputs of the gtinv model on the device: the design matrices a
// fit needs (MLIPModel::prepare_features, src/USER-MLIP/mlipkk.cpp:461-470,
// getters :1322-1381).  For every atom the structural features
// X[i][f] = d_f^(i) (all n_des, f = n * n_gtinv + itc) and the polynomial
// features P[i][p] = prod_{f in p} X[i][f]; the force features
// FF[k][p] = -dX_p/dr_k with X_p = sum_i P[i][p]; per structure the stress
// features SF[p] = sum over pairs del (x) (force term) in the order
// xx, yy, zz, yz, zx, xy (mlipkk.cpp:1260-1271).  With the regression
// weights w: sum_p w_p X_p = E, sum_p w_p FF[k][p] = F_k and sum_p w_p SF[p]
// is the virial.
//
// Kernels (a_nlm from k_anlm in FP64 first):
//   k_tr_dirj    workgroup per (centre, group of features): the features, and
//                dirj = d d_f^(i)/d del_q for every pair q of the centre
//                (mlipkk.cpp:992-1157 restated for a full list: each
//                directed pair carries its own centre's derivative)
//   k_tr_poly    thread per (atom, coefficient)
//   k_tr_force   thread per (atom, coefficient): the atom's gather list in
//                pair order, g_qp = sum_nu prod_{nu' != nu} X[cen][f_nu'] dirj[q][f_nu],
//                -g on the centre, +g on the neighbor (fixed order)
//   k_tr_stress  workgroup per (structure, 64 coefficients, part of its pairs):
//                del (x) (-g), lanes over coefficients, fixed-order sums
// All FP64.  Work and memory scale with pairs x n_des (dirj) and atoms x
// n_coeff (force features): a training-sized structure or batch, not the
// 256k-atom evaluation workload.
#include <algorithm>
#include <climits>
#include <cstring>

#include "device_common.h"
#include "engine_internal.h"

namespace mlip {

struct TrItc {
    int32_t tbeg, tend;   // term range of the itc's irrep
    int32_t order;
    int32_t spec[2][4];   // [centre type][factor] -> neighbor species, -1: absent
};

struct TrTerm {
    double c;
    // per factor: lmh index of (l, -|m|); bit 16: m > 0 (conjugate);
    // bit 17: m > 0 and odd (negate)
    int32_t code[4];
};

struct TrainWork {
    bool built = false;
    DBuf<TrItc> itc;
    DBuf<TrTerm> term;
    DBuf<int32_t> rows;   // n_coeff x 3 feature ids (-1 padded)
    DBuf<double> X, P, FF, SF, SFpart, dirj;
    DBuf<int32_t> pcen, range;
    void release() {
        itc.release();
        term.release();
        rows.release();
        X.release();
        P.release();
        FF.release();
        SF.release();
        SFpart.release();
        dirj.release();
        pcen.release();
        range.release();
    }
};

namespace {

using namespace dev;

constexpr int kTrThreads = 256;
constexpr int kTrPairs = 16;    // pairs per chunk of k_tr_dirj (at most)
constexpr int kTrMaxF = 128;    // features per workgroup of k_tr_dirj (at most)
constexpr int kTrMaxFn = 16;    // radial functions of the training path
constexpr int kTrMaxL = 12;     // angular momenta of the training path (2 n_lmh / 4 <= 64 depth steps)
constexpr int kTrL1 = kTrMaxL + 1;

struct TrArgs {
    const TrItc* itc;
    const TrTerm* term;
    const int32_t* rows;
    int n_des, n_coeff, n_gtinv;
    double* X;
    double* P;
    double* FF;
    double* SF;
    double* dirj;
    int32_t* pcen;
};

// a_{l,m} of factor `code` from the m <= 0 row value v
__device__ __forceinline__ void fac(int code, double& re, double& im) {
    if (code & (1 << 16)) {
        im = -im;
        if (code & (1 << 17)) {
            re = -re;
            im = -im;
        }
    }
}

__global__ __launch_bounds__(kTrThreads) void k_tr_poly(int natoms, TrArgs T) {
    const int64_t w = (int64_t)blockIdx.x * kTrThreads + threadIdx.x;
    if (w >= (int64_t)natoms * T.n_coeff) return;
    const int atom = (int)(w / T.n_coeff), p = (int)(w % T.n_coeff);
    double v = 1.0;
    for (int k = 0; k < 3; ++k) {
        const int f = T.rows[3 * p + k];
        if (f >= 0) v *= T.X[(size_t)atom * T.n_des + f];
    }
    T.P[w] = v;
}

__global__ __launch_bounds__(kTrThreads) void k_tr_pcen(DevSystem S, int32_t* pcen) {
    const int a = blockIdx.x * kTrThreads + threadIdx.x;
    if (a >= S.nown) return;
    for (int q = S.poff[a]; q < S.pend[a]; ++q) pcen[q] = a;
}

// Shape of a k_tr_dirj launch: F features and `pairs` pairs at a time per
// workgroup, kp = 2 n_lmh rounded up to the matrix instruction's depth of 4,
// and the rows of radial indices F consecutive features can span.
struct TrShape {
    int F, pairs, kp, nrow;
    __host__ __device__ int ypitch() const { return kp + 2; }
};

struct TrLds {
    double yt_diag[kTrL1 + 1];
    double yt_alm[kTrL1][kTrL1];
    double yt_ainv[kTrL1][kTrL1];
    double yt_grad[kTrL1][kTrL1];
    double ux[kTrPairs], uy[kTrPairs], uz[kTrPairs], rr[kTrPairs], fc[kTrPairs], fcd[kTrPairs];
    int spec[kTrPairs];
    double gn[kTrPairs][kTrMaxFn], gd[kTrPairs][kTrMaxFn];
    unsigned long long steps[kTrMaxF / 16][2];
};

// Structural features and their derivatives along every pair of the centre.
// Workgroup = (centre, F consecutive features).
//  1. Thread per feature: d_f and, since d d_f / d a_{s,n,lm} does not depend
//     on the pair, its partials B_f[s][(lm, re/im)] over all terms and factors
//     into the thread's own LDS column (m > 0 folded onto m <= 0).
//  2. Per tile of pairs: Y_lm and grad Y_lm of each pair into LDS, then
//     [(pair, Y / x / y / z)][(lm, c)] x B[(lm, c)][f] on the matrix cores
//     (v_mfma_f64_16x16x4f64, lanes as in k_anlm_mfma): 4 pairs x 16 features
//     per instruction tile; rows of pairs of the other species are masked, and
//     the depth steps no feature of the tile uses are skipped.  Row i = pair
//     i % 4, quantity i / 4, so a lane ends with the four sums of one pair and
//     feature.
// Bound: the products of step 1 and the matrix steps.  Forming each pair's
// derivative from all terms took one product chain per (pair, term, factor):
// 12 random cells of 8-32 atoms (gtinv-820, ~1,900 features, ~70 pairs per
// atom) 51.0 ms, now 2.3 ms.
__global__ __launch_bounds__(kTrThreads) void k_tr_dirj(DevModel M, DevSystem S, TrArgs T, TrShape H, int grad) {
    extern __shared__ double tr_dyn[];
    __shared__ TrLds C;
    typedef double dbl4 __attribute__((ext_vector_type(4)));
    const int atom = blockIdx.x;
    const int tid = threadIdx.x;
    const int nfn = M.n_fn, ns = M.n_type, nlmh = M.n_lmh, maxl = M.maxl;
    const int slot = S.slot_of_atom[atom];
    const int blk = slot / kBlock, slane = slot % kBlock;
    const int tcen = S.elem[atom];
    const int f0 = blockIdx.y * H.F, f1 = min(f0 + H.F, T.n_des);
    const int nlo = f0 / T.n_gtinv, nhi = (f1 - 1) / T.n_gtinv;
    double* aL = tr_dyn;                                          // [n - nlo][s][lm] (re, im)
    double* bL = aL + static_cast<size_t>(2) * H.nrow * ns * nlmh;  // [s][kp][F]
    double* yL = bL + static_cast<size_t>(ns) * H.kp * H.F;       // [pair][quantity][ypitch]
    const int yp = H.ypitch();
    for (int k = tid; k < (nhi - nlo + 1) * ns * nlmh; k += kTrThreads) {
        const int lm = k % nlmh, s = (k / nlmh) % ns, n = nlo + k / (nlmh * ns);
        aL[2 * k] = S.A[a_index(M, blk, n, s, lm, 0, slane)];
        aL[2 * k + 1] = S.A[a_index(M, blk, n, s, lm, 1, slane)];
    }
    if (grad) {
        for (int k = tid; k < ns * H.kp * H.F; k += kTrThreads) bL[k] = 0.0;
        for (int k = tid; k < H.pairs * 4 * yp; k += kTrThreads) yL[k] = 0.0;
        if (tid < 2 * (kTrMaxF / 16)) C.steps[tid / 2][tid % 2] = 0;
        const YTab<double>* yt = M.yt64;
        for (int k = tid; k < kTrL1 * kTrL1; k += kTrThreads) {
            const int l = k / kTrL1, mm = k % kTrL1;
            C.yt_alm[l][mm] = yt->alm[l][mm];
            C.yt_ainv[l][mm] = yt->ainv[l][mm];
            C.yt_grad[l][mm] = yt->grad[l][mm];
        }
        if (tid <= kTrL1) C.yt_diag[tid] = yt->diag[tid];
    }
    __syncthreads();
    if (f0 + tid < f1) {
        const int f = f0 + tid, itc = f % T.n_gtinv, n = f / T.n_gtinv;
        const TrItc& I = T.itc[itc];
        bool seen = true;
        for (int mu = 0; mu < I.order; ++mu) seen = seen && I.spec[tcen][mu] >= 0;
        double d = 0.0;
        if (seen) {
            const double* ar = aL + static_cast<size_t>(2) * (n - nlo) * ns * nlmh;
            unsigned long long used[2] = {0, 0};
            for (int k = I.tbeg; k < I.tend; ++k) {
                const TrTerm& tm = T.term[k];
                double vr[4], vi[4];
                double pr = tm.c, pi = 0.0;
#pragma unroll
                for (int mu = 0; mu < 4; ++mu) {
                    if (mu >= I.order) break;
                    const double* av = ar + 2 * (I.spec[tcen][mu] * nlmh + (tm.code[mu] & 0xffff));
                    vr[mu] = av[0];
                    vi[mu] = av[1];
                    fac(tm.code[mu], vr[mu], vi[mu]);
                    const double nr = pr * vr[mu] - pi * vi[mu];
                    pi = pr * vi[mu] + pi * vr[mu];
                    pr = nr;
                }
                d += pr;
                if (!grad) continue;
#pragma unroll
                for (int mu = 0; mu < 4; ++mu) {
                    if (mu >= I.order) break;
                    double qr = tm.c, qi = 0.0;
#pragma unroll
                    for (int m2 = 0; m2 < 4; ++m2) {
                        if (m2 >= I.order || m2 == mu) continue;
                        const double nr = qr * vr[m2] - qi * vi[m2];
                        qi = qr * vi[m2] + qi * vr[m2];
                        qr = nr;
                    }
                    // Re(q Y_m) with Y_m = (-1)^m conj(Y_{-m}) for m > 0 is
                    // Re((-1)^m conj(q) Y_{-m})
                    const int code = tm.code[mu], kk = 2 * (code & 0xffff), s = I.spec[tcen][mu];
                    fac(code, qr, qi);
                    double* col = bL + (static_cast<size_t>(s) * H.kp + kk) * H.F + tid;
                    col[0] += qr;
                    col[H.F] += qi;
                    used[s] |= 1ull << (kk >> 2);
                }
            }
            if (grad)
                for (int s = 0; s < ns; ++s) atomicOr(&C.steps[tid / 16][s], used[s]);
        }
        T.X[static_cast<size_t>(atom) * T.n_des + f] = d;
    }
    if (!grad) return;
    const int p0 = S.poff[atom], p1 = S.pend[atom];
    const double pir = 3.141592653589793 / M.cutoff;
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int ftiles = (f1 - f0 + 15) / 16;
    for (int pc = p0; pc < p1; pc += H.pairs) {
        const int np = min(H.pairs, p1 - pc);
        __syncthreads();
        if (tid < H.pairs) {
            const int q = pc + tid;
            int spec = -1;
            if (tid < np) {
                const int nb = S.pnbr[q];
                double dx = S.x[3 * atom] - S.x[3 * nb], dy = S.x[3 * atom + 1] - S.x[3 * nb + 1],
                       dz = S.x[3 * atom + 2] - S.x[3 * nb + 2];
                if (S.pshift) {
                    dx += S.pshift[3 * q];
                    dy += S.pshift[3 * q + 1];
                    dz += S.pshift[3 * q + 2];
                }
                const double r = sqrt(dx * dx + dy * dy + dz * dz);
                if ((r < M.cutoff) && (r > 0.0)) {
                    spec = S.elem[nb];
                    C.ux[tid] = dx / r;
                    C.uy[tid] = dy / r;
                    C.uz[tid] = dz / r;
                    C.rr[tid] = r;
                    double sa, ca;
                    sincos(pir * r, &sa, &ca);
                    C.fc[tid] = 0.5 * (ca + 1.0);
                    C.fcd[tid] = -0.5 * pir * sa;
                }
            }
            C.spec[tid] = spec;
        }
        __syncthreads();
        for (int it = tid; it < np * (maxl + 1); it += kTrThreads) {
            // column m of pair j: Y_{l,-m} and grad Y_{l,-m} for l = m..maxl,
            // imaginary parts negated (Re(B Y) = Br Yr + Bi (-Yi))
            const int j = it % np, m = it / np;
            if (C.spec[j] < 0) continue;
            const double x = C.ux[j], y = C.uy[j], z = C.uz[j], ir = 1.0 / C.rr[j];
            double cr = 1.0, ci = 0.0;  // conj(u)^m
            double mr = 0.0, mi = 0.0;  // conj(u)^(m-1)
            for (int k = 0; k < m; ++k) {
                mr = cr;
                mi = ci;
                const double nr = cr * x + ci * y;
                ci = ci * x - cr * y;
                cr = nr;
            }
            const double pr = cr * x + ci * y, pi = ci * x - cr * y;  // conj(u)^(m+1)
            const double sg = (m & 1) ? -1.0 : 1.0, zz = 1.0 - z * z, fm = (double)m;
            double a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
            for (int l = m; l <= maxl; ++l) {
                const double q = (l == m) ? C.yt_diag[m] : C.yt_alm[l][m] * (z * a1 - C.yt_ainv[l][m] * a2);
                a2 = a1;
                a1 = q;
                double qp = 0.0;
                if (l == m + 1)
                    qp = C.yt_diag[m + 1];
                else if (l > m + 1)
                    qp = C.yt_alm[l][m + 1] * (z * b1 - C.yt_ainv[l][m + 1] * b2);
                b2 = b1;
                b1 = qp;
                double gxr, gxi, gyr, gyi, gzr, gzi;
                if (m == 0) {
                    const double c = C.yt_grad[l][0] * qp;
                    gxr = c * z * x;
                    gxi = 0.0;
                    gyr = c * z * y;
                    gyi = 0.0;
                    gzr = -c * zz;
                    gzi = 0.0;
                } else {
                    const double c = C.yt_grad[l][m];
                    const double A = fm * z * q + zz * c * qp;
                    const double B = fm * q - z * c * qp;
                    const double E = fm * (1.0 + z * z) * q + z * zz * c * qp;
                    gxr = 0.5 * (-B * pr + E * mr);
                    gxi = 0.5 * (-B * pi + E * mi);
                    const double zr = B * pr + E * mr, zi = B * pi + E * mi;
                    gyr = 0.5 * zi;
                    gyi = -0.5 * zr;
                    gzr = -A * cr;
                    gzi = -A * ci;
                }
                double* o = yL + static_cast<size_t>(4 * j) * yp + 2 * (l * (l + 1) / 2 + l - m);
                o[0] = sg * q * cr;
                o[1] = -sg * q * ci;
                o[yp] = sg * gxr * ir;
                o[yp + 1] = -sg * gxi * ir;
                o[2 * yp] = sg * gyr * ir;
                o[2 * yp + 1] = -sg * gyi * ir;
                o[3 * yp] = sg * gzr * ir;
                o[3 * yp + 1] = -sg * gzi * ir;
            }
        }
        for (int it = tid; it < np * nfn; it += kTrThreads) {
            const int j = it / nfn, n = it % nfn;
            if (C.spec[j] < 0) continue;
            const double dd = C.rr[j] - M.mu[n], be = M.beta[n];
            const double b = exp(-be * (dd * dd));
            C.gn[j][n] = b * C.fc[j];
            C.gd[j][n] = b * (C.fcd[j] - 2.0 * be * dd * C.fc[j]);
        }
        __syncthreads();
        const int ptiles = (np + 3) / 4;
        for (int task = wave; task < ptiles * ftiles; task += kTrThreads / 64) {
            const int ft = task % ftiles, pt = task / ftiles;
            // A[i][k] from lane 16 k + i, B[k][j] from lane 16 k + j
            const int ja = 4 * pt + (lane & 3), quant = (lane >> 2) & 3, kl = lane >> 4;
            const int sa = ja < np ? C.spec[ja] : -1;
            const double* ya = yL + static_cast<size_t>(4 * ja + quant) * yp + kl;
            const double* bb = bL + static_cast<size_t>(kl) * H.F + 16 * ft + (lane & 15);
            dbl4 acc = {0.0, 0.0, 0.0, 0.0};
            for (int s = 0; s < ns; ++s) {
                if (__ballot(sa == s) == 0) continue;
                unsigned long long left = C.steps[ft][s];
                while (left) {
                    const int k = 4 * __builtin_ctzll(left);
                    left &= left - 1;
                    const double a = sa == s ? ya[k] : 0.0;
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        a, bb[(static_cast<size_t>(s) * H.kp + k) * H.F], acc, 0, 0, 0);
                }
            }
            // lane: D[i = lane / 16 + 4 r][lane % 16] = quantity r of pair lane / 16
            const int j = 4 * pt + (lane >> 4), f = f0 + 16 * ft + (lane & 15);
            if (j < np && f < f1) {
                double* out = T.dirj + (static_cast<size_t>(pc + j) * T.n_des + f) * 3;
                double gd = 0.0, gn = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
                if (C.spec[j] >= 0) {
                    const int n = f / T.n_gtinv;
                    gd = C.gd[j][n];
                    gn = C.gn[j][n];
                    ux = C.ux[j];
                    uy = C.uy[j];
                    uz = C.uz[j];
                }
                out[0] = gd * ux * acc[0] + gn * acc[1];
                out[1] = gd * uy * acc[0] + gn * acc[2];
                out[2] = gd * uz * acc[0] + gn * acc[3];
            }
        }
    }
}

// LDS bytes of a launch shape, and the shape for a model: 128 features and 16
// pairs per workgroup where the tables leave two workgroups per CU, fewer as
// l_max grows (B takes n_type kp 8 bytes per feature, a pair 32 kp), down to 16
// and 4, which is taken even where only one workgroup then fits (two species at
// l_max 12).
size_t tr_lds(const DevModel& m, const TrShape& h) {
    return sizeof(double) * (static_cast<size_t>(2) * h.nrow * m.n_type * m.n_lmh +
                             static_cast<size_t>(m.n_type) * h.kp * h.F + static_cast<size_t>(h.pairs) * 4 * h.ypitch());
}

TrShape tr_shape(const DevModel& m, int n_gtinv) {
    TrShape h{kTrMaxF, kTrPairs, (2 * m.n_lmh + 3) / 4 * 4, 0};
    for (;;) {
        h.nrow = std::min(m.n_fn, (h.F - 1) / n_gtinv + 2);
        if (tr_lds(m, h) + sizeof(TrLds) <= 80 * 1024 || (h.F == 16 && h.pairs == 4)) return h;
        // the larger of the two tables first
        if (h.F > 16 && (h.pairs == 4 || m.n_type * h.F >= 4 * h.pairs))
            h.F /= 2;
        else
            h.pairs /= 2;
    }
}

// g_{q,p} = d P_cen(p) / d del_q
__device__ __forceinline__ void coef_grad(const TrArgs& T, int p, int cen, int64_t q, double g[3]) {
    const int f0 = T.rows[3 * p], f1 = T.rows[3 * p + 1], f2 = T.rows[3 * p + 2];
    const double* xc = T.X + (size_t)cen * T.n_des;
    const double* dq = T.dirj + (size_t)q * T.n_des * 3;
    double c0 = 1.0, c1 = 0.0, c2 = 0.0;
    if (f1 >= 0) {
        c0 = xc[f1];
        c1 = xc[f0];
        if (f2 >= 0) {
            c0 *= xc[f2];
            c1 *= xc[f2];
            c2 = xc[f0] * xc[f1];
        }
    }
    for (int k = 0; k < 3; ++k) {
        double v = c0 * dq[3 * f0 + k];
        if (f1 >= 0) v += c1 * dq[3 * f1 + k];
        if (f2 >= 0) v += c2 * dq[3 * f2 + k];
        g[k] = v;
    }
}

__global__ __launch_bounds__(kTrThreads) void k_tr_force(DevSystem S, TrArgs T, int pchunks) {
    const int atom = blockIdx.x / pchunks;
    const int p = (blockIdx.x % pchunks) * kTrThreads + threadIdx.x;
    if (atom >= S.nown || p >= T.n_coeff) return;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    for (int e = S.goff[atom]; e < S.gend[atom]; ++e) {
        const int en = S.gent[e];
        const int64_t q = (en > 0 ? en : -en) - 1;
        double g[3];
        coef_grad(T, p, T.pcen[q], q, g);
        if (en > 0) {
            fx += g[0];
            fy += g[1];
            fz += g[2];
        } else {
            fx -= g[0];
            fy -= g[1];
            fz -= g[2];
        }
    }
    double* o = T.FF + ((size_t)atom * T.n_coeff + p) * 3;
    o[0] = fx;
    o[1] = fy;
    o[2] = fz;
}

// Stress features: workgroup = (structure, 64 coefficients, part of the
// structure's pairs).  Lane = coefficient, so the pairs' derivative rows are
// read in runs; the workgroup's waves take every fourth pair and are added in
// order, the parts by k_tr_stress_sum.  A workgroup per (structure,
// coefficient) with its threads over the pairs read 24 bytes per line: 12 small
// cells, 6,695 coefficients, 2.11 ms.
constexpr int kTrStressWaves = 4;

__global__ __launch_bounds__(64 * kTrStressWaves) void k_tr_stress(DevSystem S, TrArgs T, const int32_t* sbeg,
                                                                   const int32_t* send, int pchunks, double* out,
                                                                   int64_t part_stride) {
    __shared__ double red[kTrStressWaves][6][64];
    const int s = blockIdx.x / pchunks, lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
    const int p = (blockIdx.x % pchunks) * 64 + lane;
    const int a0 = sbeg[s], a1 = send[s];
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (a1 > a0 && p < T.n_coeff) {
        const int64_t q0 = S.poff[a0], nq = S.pend[a1 - 1] - q0;
        const int64_t b = q0 + nq * blockIdx.y / gridDim.y, e = q0 + nq * (blockIdx.y + 1) / gridDim.y;
        for (int64_t q = b + wave; q < e; q += kTrStressWaves) {
            const int cen = T.pcen[q], nb = S.pnbr[q];
            double dx = S.x[3 * cen] - S.x[3 * nb], dy = S.x[3 * cen + 1] - S.x[3 * nb + 1],
                   dz = S.x[3 * cen + 2] - S.x[3 * nb + 2];
            if (S.pshift) {
                dx += S.pshift[3 * q];
                dy += S.pshift[3 * q + 1];
                dz += S.pshift[3 * q + 2];
            }
            double g[3];
            coef_grad(T, p, cen, q, g);
            // force term on the centre is -g
            v[0] -= dx * g[0];
            v[1] -= dy * g[1];
            v[2] -= dz * g[2];
            v[3] -= dy * g[2];
            v[4] -= dz * g[0];
            v[5] -= dx * g[1];
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) red[wave][k][lane] = v[k];
    __syncthreads();
    const int np = min(64, T.n_coeff - (static_cast<int>(blockIdx.x) % pchunks) * 64);
    double* o = out + blockIdx.y * part_stride +
                (static_cast<size_t>(s) * T.n_coeff + (blockIdx.x % pchunks) * 64) * 6;
    for (int e = threadIdx.x; e < 6 * np; e += 64 * kTrStressWaves) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < kTrStressWaves; ++w) sum += red[w][e % 6][e / 6];
        o[e] = sum;
    }
}

__global__ __launch_bounds__(kTrThreads) void k_tr_stress_sum(const double* part, int parts, int64_t n, double* out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kTrThreads + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int k = 0; k < parts; ++k) s += part[k * n + i];
    out[i] = s;
}

bool build_tables(mlip_ctx* c, TrainWork& w) {
    const Model& m = c->model;
    std::vector<TrItc> itc(m.n_gtinv);
    std::vector<TrTerm> term;
    std::vector<int32_t> tbeg(m.irreps.size()), tend(m.irreps.size());
    for (size_t r = 0; r < m.irreps.size(); ++r) {
        const Irrep& ir = m.irreps[r];
        tbeg[r] = static_cast<int32_t>(term.size());
        for (size_t k = 0; k < ir.m.size(); ++k) {
            TrTerm t{};
            t.c = ir.c[k];
            for (size_t mu = 0; mu < ir.l.size(); ++mu) {
                const int l = ir.l[mu], mm = ir.m[k][mu];
                const int am = mm < 0 ? -mm : mm;
                if (l > m.maxl) {
                    c->err = "invariant with l above the model's max_l";
                    return false;
                }
                int code = lmh_index(l, -am);
                if (mm > 0) code |= 1 << 16;
                if (mm > 0 && (mm & 1)) code |= 1 << 17;
                t.code[mu] = code;
            }
            term.push_back(t);
        }
        tend[r] = static_cast<int32_t>(term.size());
    }
    for (int i = 0; i < m.n_gtinv; ++i) {
        const Itc& it = m.itcs[i];
        TrItc& d = itc[i];
        std::memset(&d, 0, sizeof d);
        d.tbeg = tbeg[it.irrep];
        d.tend = tend[it.irrep];
        d.order = it.order;
        for (int t = 0; t < 2; ++t)
            for (int mu = 0; mu < 4; ++mu)
                d.spec[t][mu] = (t < m.n_type && mu < it.order) ? m.tcp_other[it.tc[mu]][t] : -1;
    }
    std::vector<int32_t> rows(3 * static_cast<size_t>(m.n_coeff), -1);
    for (int f = 0; f < m.n_des; ++f) rows[3 * f] = f;
    int p = m.n_des;
    for (const auto& cb : m.comb2) {
        rows[3 * p] = cb[0];
        rows[3 * p + 1] = cb[1];
        ++p;
    }
    for (const auto& cb : m.comb3) {
        rows[3 * p] = cb[0];
        rows[3 * p + 1] = cb[1];
        rows[3 * p + 2] = cb[2];
        ++p;
    }
    if (!upload(c, w.itc, itc.data(), itc.size(), "training tables") ||
        !upload(c, w.term, term.data(), term.size(), "training tables") ||
        !upload(c, w.rows, rows.data(), rows.size(), "training tables"))
        return false;
    w.built = true;
    return true;
}

}  // namespace

int train_features(mlip_ctx* c, double* X, double* P, double* FF, double* SF) {
    const Model& m = c->model;
    if (m.pair_model) {
        c->err = "training features are defined for the gtinv descriptor";
        return MLIP_ERR_MODEL;
    }
    static_assert((kTrL1 * (kTrL1 + 1) + 3) / 4 <= 64, "depth steps of k_tr_dirj in one mask");
    static_assert(kTrMaxF <= kTrThreads, "a thread per feature in k_tr_dirj");
    if (m.maxl > kTrMaxL) {
        c->err = "training features support max_l up to 12";
        return MLIP_ERR_MODEL;
    }
    if (m.n_type > 2 || m.n_fn > kTrMaxFn) {
        c->err = "training features support up to two species and 16 radial functions";
        return MLIP_ERR_MODEL;
    }
    for (const Itc& it : m.itcs)
        if (it.order > 4) {
            c->err = "training features support invariants up to order 4";
            return MLIP_ERR_MODEL;
        }
    if (!c->resident) {
        c->err = "no resident structure";
        return MLIP_ERR_STATE;
    }
    if (!c->trw) c->trw = new TrainWork();
    TrainWork& w = *c->trw;
    if (!w.built && !build_tables(c, w)) return MLIP_ERR_DEVICE;
    const DevSystem& s = c->ds;
    const int n = s.nown;
    const int64_t np = c->npairs;
    const size_t dbytes = static_cast<size_t>(np) * m.n_des * 3 * sizeof(double);
    const size_t fbytes = static_cast<size_t>(n) * m.n_coeff * 3 * sizeof(double);
    if (dbytes > (size_t(24) << 30) || fbytes > (size_t(24) << 30)) {
        c->err = "training features of this structure need more than 24 GB; use smaller batches";
        return MLIP_ERR_ARG;
    }
    const int nstruct = c->nstruct > 0 ? c->nstruct : 1;
    if (static_cast<int64_t>(nstruct) * m.n_coeff > INT_MAX) {
        c->err = "too many structures x coefficients";
        return MLIP_ERR_ARG;
    }
    if (!w.X.ensure(static_cast<size_t>(n) * m.n_des) || !w.P.ensure(static_cast<size_t>(n) * m.n_coeff) ||
        !w.FF.ensure(static_cast<size_t>(n) * m.n_coeff * 3) ||
        !w.SF.ensure(static_cast<size_t>(nstruct) * m.n_coeff * 6) ||
        !w.dirj.ensure(static_cast<size_t>(np) * m.n_des * 3) || !w.pcen.ensure(static_cast<size_t>(np))) {
        c->err = "device allocation failed for training features";
        return MLIP_ERR_DEVICE;
    }
    // single structure: one range over all atoms
    const int32_t* sb = c->sbeg;
    const int32_t* se = c->send;
    hipStream_t st = c->stream;
    if (c->nstruct == 0) {
        const int32_t r[2] = {0, n};
        if (!upload(c, w.range, r, 2, "structure range")) return MLIP_ERR_DEVICE;
        sb = w.range.p;
        se = w.range.p + 1;
    }
    TrArgs a{w.itc.p, w.term.p, w.rows.p, m.n_des, m.n_coeff, m.n_gtinv, w.X.p, w.P.p, w.FF.p, w.SF.p, w.dirj.p,
             w.pcen.p};
    if (!hip_ok(c, launch_anlm(c->dm, s, kFP64, st), "a_nlm launch")) return MLIP_ERR_DEVICE;
    const bool grad = n > 0 && np > 0 && (FF || SF);
    if (n > 0) {
        const TrShape h = tr_shape(c->dm, m.n_gtinv);
        const size_t lds = tr_lds(c->dm, h);
        if (lds + sizeof(TrLds) > lds_limit()) {
            c->err = "training features: the model's per-centre LDS tile exceeds the device limit";
            return MLIP_ERR_MODEL;
        }
        if (!hip_ok(c, hipFuncSetAttribute(reinterpret_cast<const void*>(k_tr_dirj),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
                    "training LDS"))
            return MLIP_ERR_DEVICE;
        hipLaunchKernelGGL(k_tr_dirj, dim3(n, (m.n_des + h.F - 1) / h.F), dim3(kTrThreads), lds, st, c->dm, s, a, h,
                           grad ? 1 : 0);
        if (!hip_ok(c, launched(), "feature derivative launch")) return MLIP_ERR_DEVICE;
    }
    const int64_t npw = static_cast<int64_t>(n) * m.n_coeff;
    if (npw > 0) {
        hipLaunchKernelGGL(k_tr_poly, dim3(static_cast<unsigned>((npw + kTrThreads - 1) / kTrThreads)),
                           dim3(kTrThreads), 0, st, n, a);
        if (!hip_ok(c, launched(), "polynomial feature launch")) return MLIP_ERR_DEVICE;
    }
    if (grad) {
        hipLaunchKernelGGL(k_tr_pcen, dim3((n + kTrThreads - 1) / kTrThreads), dim3(kTrThreads), 0, st, s, w.pcen.p);
        if (!hip_ok(c, launched(), "pair centre launch")) return MLIP_ERR_DEVICE;
        const int pchunks = (m.n_coeff + kTrThreads - 1) / kTrThreads;
        if (FF) {
            hipLaunchKernelGGL(k_tr_force, dim3(static_cast<unsigned>(static_cast<int64_t>(n) * pchunks)),
                               dim3(kTrThreads), 0, st, s, a, pchunks);
            if (!hip_ok(c, launched(), "force feature launch")) return MLIP_ERR_DEVICE;
        }
        if (SF) {
            // parts of a structure's pairs until some 4,096 workgroups run
            // (12 small cells fill them alone; one structure needs the parts),
            // each part at least 64 pairs
            const int chunks = (m.n_coeff + 63) / 64;
            const int64_t groups = static_cast<int64_t>(nstruct) * chunks, want = (4096 + groups - 1) / groups;
            const int parts = static_cast<int>(std::max<int64_t>(1, std::min(want, np / nstruct / 64)));
            const int64_t nout = static_cast<int64_t>(nstruct) * m.n_coeff * 6;
            if (parts > 1 && !w.SFpart.ensure(static_cast<size_t>(nout) * parts)) {
                c->err = "device allocation failed for training features";
                return MLIP_ERR_DEVICE;
            }
            hipLaunchKernelGGL(k_tr_stress, dim3(static_cast<unsigned>(groups), parts), dim3(64 * kTrStressWaves), 0,
                               st, s, a, sb, se, chunks, parts > 1 ? w.SFpart.p : w.SF.p, nout);
            if (parts > 1)
                hipLaunchKernelGGL(k_tr_stress_sum, dim3(static_cast<unsigned>((nout + kTrThreads - 1) / kTrThreads)),
                                   dim3(kTrThreads), 0, st, w.SFpart.p, parts, nout, w.SF.p);
            if (!hip_ok(c, launched(), "stress feature launch")) return MLIP_ERR_DEVICE;
        }
    } else {
        if (FF && !hip_ok(c, hipMemsetAsync(w.FF.p, 0, fbytes, st), "force features")) return MLIP_ERR_DEVICE;
        if (SF && !hip_ok(c, hipMemsetAsync(w.SF.p, 0, sizeof(double) * nstruct * m.n_coeff * 6, st),
                          "stress features"))
            return MLIP_ERR_DEVICE;
    }
    if (!hip_ok(c, hipGetLastError(), "training kernels")) return MLIP_ERR_DEVICE;
    bool ok = true;
    if (X) ok = ok && hip_ok(c, hipMemcpyAsync(X, w.X.p, sizeof(double) * n * m.n_des, hipMemcpyDeviceToHost, st), "X");
    if (P) ok = ok && hip_ok(c, hipMemcpyAsync(P, w.P.p, sizeof(double) * npw, hipMemcpyDeviceToHost, st), "P");
    if (FF) ok = ok && hip_ok(c, hipMemcpyAsync(FF, w.FF.p, fbytes, hipMemcpyDeviceToHost, st), "FF");
    if (SF)
        ok = ok && hip_ok(c, hipMemcpyAsync(SF, w.SF.p, sizeof(double) * nstruct * m.n_coeff * 6,
                                            hipMemcpyDeviceToHost, st),
                          "SF");
    ok = ok && hip_ok(c, hipStreamSynchronize(st), "training features");
    return ok ? MLIP_OK : MLIP_ERR_DEVICE;
}

void train_free(mlip_ctx* c) {
    if (!c->trw) return;
    c->trw->release();
    delete c->trw;
    c->trw = nullptr;
}

}  // namespace mlip
