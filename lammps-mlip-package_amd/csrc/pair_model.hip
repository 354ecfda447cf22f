// Radial-only style (reference: pair_style mlip_pair,
// src/USER-MLIP/pair_mlip_pair.cpp:56-258).  Per centre i of type t:
//   d_{tc(t,s),n} = sum_{j of type s, r < r_c} g_n(r_ij)
//   E_i = sum_a w_a d_a + sum_terms w prod d,   H_a = dE_i/dd_a
// and per directed pair dE_i/d(del) = sum_n g'_n(r) H_{tc,n} del / r.  The
// pair results go through the same gather and reductions as the gtinv path.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "device_api.h"
#include "device_common.h"

namespace mlip {

namespace {

using namespace dev;

constexpr double kPiRef = 3.141592653589793;  // mlip_basis_function.cpp:26
constexpr int kPairThreads = 64;

__device__ __forceinline__ bool pair_geom(const DevModel& M, const DevSystem& S, int atom, int64_t p, double& dx,
                                          double& dy, double& dz, double& r) {
    const int nb = S.pnbr[p];
    const int c = S.pcen ? S.pcen[p] : atom;
    dx = S.x[3 * c] - S.x[3 * nb];
    dy = S.x[3 * c + 1] - S.x[3 * nb + 1];
    dz = S.x[3 * c + 2] - S.x[3 * nb + 2];
    if (S.pshift) {
        dx += S.pshift[3 * p];
        dy += S.pshift[3 * p + 1];
        dz += S.pshift[3 * p + 2];
    }
    r = sqrt(dx * dx + dy * dy + dz * dz);
    return r < M.cutoff && r > 0.0;
}

// One wave per slot.  Batches of 64 pairs: lane = pair for the geometry (r,
// cutoff function and species into LDS), then lane = (radial index, group)
// sums its g_n over the batch's pairs group, group + G, ... (G = 64 / NF), the
// groups added by a fixed butterfly at the end.  Bound: the exponentials, one
// per (pair, n).  A thread per slot walked its ~440 pairs alone (2,048 atoms,
// r_c 12 A, 20 radial functions: 1,600 us, 32 waves on the device).
template <int NF>
__global__ __launch_bounds__(kPairThreads) void k_pair_feat(DevModel M, DevSystem S) {
    constexpr int G = 64 / NF;
    __shared__ double rr[64], fc[64];
    __shared__ int spec[64];
    const int slot = blockIdx.x, lane = threadIdx.x;
    const int atom = S.atom_of_slot[slot];
    const int nfn = M.n_fn, t = atom < 0 ? 0 : S.elem[atom];
    double* row = S.D + static_cast<size_t>(slot) * M.n_p;
    for (int a = lane; a < M.n_p; a += 64) {
        const int tc = a / nfn;
        bool seen = false;
        for (int s = 0; s < M.n_type; ++s) seen = seen || M.pair_tc[t][s] == tc;
        if (atom < 0 || !seen) row[a] = 0.0;
    }
    if (atom < 0) return;
    const int n = lane % NF, grp = lane / NF;
    const double mu = n < nfn ? M.mu[n] : 0.0, beta = n < nfn ? M.beta[n] : 0.0;
    double acc0 = 0.0, acc1 = 0.0;
    const double pir = kPiRef / M.cutoff;
    const int64_t p0 = S.poff[atom], p1 = S.pend[atom];
    for (int64_t b = p0; b < p1; b += 64) {
        int s = -1;
        if (b + lane < p1) {
            double dx, dy, dz, r;
            if (pair_geom(M, S, atom, b + lane, dx, dy, dz, r)) {
                s = S.elem[S.pnbr[b + lane]];
                rr[lane] = r;
                fc[lane] = 0.5 * (cos(pir * r) + 1.0);
            }
        }
        spec[lane] = s;
        __syncthreads();
        const int nb = static_cast<int>(p1 - b < 64 ? p1 - b : 64);
        for (int j = grp; j < nb; j += G) {
            const int sj = spec[j];
            if (sj < 0) continue;
            const double d = rr[j] - mu;
            const double g = exp(-beta * d * d) * fc[j];
            if (sj == 0)
                acc0 += g;
            else
                acc1 += g;
        }
        __syncthreads();
    }
    for (int off = NF; off < 64; off *= 2) {
        acc0 += __shfl_xor(acc0, off);
        acc1 += __shfl_xor(acc1, off);
    }
    if (lane < nfn) {
        row[M.pair_tc[t][0] * nfn + n] = acc0;
        if (M.n_type > 1) row[M.pair_tc[t][1] * nfn + n] = acc1;
    }
}

// H and the energy as one product per 16 centres of a species on the matrix
// cores (v_mfma_f64_16x16x4f64: A[i][k] from lane 16 k + i, B[k][j] from lane
// 16 k + j, result r of lane l = D[l / 16 + 4 r][l % 16]): A = the centre's
// factors d_b, then its products d_b d_c formed on the fly from LDS, B = the
// model's dense weights (Model::pd_w).  Wave (tile, split): 16 columns of H, a
// quarter of the rows; the splits are added in order through LDS.  The
// quadratic and cubic sums stay apart, since the energy E = sum_a d_a (w_a +
// s2_a / 2 + s3_a / 3) and the per-atom energy split weight them by 1 / degree.
// Bound: the row loop's latency.  One thread per centre over the derivative
// lists (66k entries, dependent loads) took 12.3 ms at 2,048 atoms of the
// 20-function cubic model whatever the atom count up to one wave per CU.
// Rounding: the products reach 1e5 against energies of a few eV, so the order of
// the additions decides what is lost.  rms force error against 80 bits (500 and
// 2,048 atoms of that model, of the rms force): one chain per derivative over the
// lists 2.9e-13 .. 3.2e-13; four plain chains per column, as the split alone gives,
// 6.1e-13 .. 6.5e-13; with the additions of eight rows each compensated (Kahan)
// 2.4e-13 (224 us a step of the 2,048 atoms; the plain four chains 227 us).
constexpr int kPolySplit = 4;

__global__ __launch_bounds__(1024) void k_pair_poly_dense(DevModel M, DevSystem S) {
    extern __shared__ double pd_lds[];
    typedef double dbl4 __attribute__((ext_vector_type(4)));
    const int nf = M.n_type * M.n_fn, nfn = M.n_fn, pitch = (nf + 1) | 1;
    const int slot0 = blockIdx.x * 16;
    const int t = uniform(S.block_type[slot0 / kBlock]);
    double* d = pd_lds;                    // [16][pitch]: factors, then 1
    double* part = pd_lds + 16 * pitch;    // [2][tile][split][4][64]
    const int nth = blockDim.x, lane = threadIdx.x & 63;
    for (int e = threadIdx.x; e < 16 * (nf + 1); e += nth) {
        const int i = e / (nf + 1), b = e % (nf + 1);
        const int s = b / nfn;
        d[i * pitch + b] =
            b == nf ? 1.0 : S.D[static_cast<size_t>(slot0 + i) * M.n_p + M.pair_tc[t][s] * nfn + (b - s * nfn)];
    }
    __syncthreads();
    const int ntile = M.pd_cols / 16;
    const int wave = uniform(threadIdx.x >> 6), tile = wave % ntile, split = wave / ntile;
    const double* w = M.pd_w + static_cast<size_t>(t) * (M.pd_k2 + M.pd_k3) * M.pd_cols + tile * 16 + (lane & 15);
    const double* di = d + (lane & 15) * pitch;
    // two steps' products by the instruction, added with the rounding of each
    // addition carried into the next (see above)
    auto sum = [&](int k0, int k1) {
        const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
        auto step = [&](int k, dbl4 acc) __attribute__((always_inline)) {
            const int kk = k + (lane >> 4);
            const int bc = M.pd_bc[kk];
            const double a = di[bc & 0xffff] * di[bc >> 16];
            return __builtin_amdgcn_mfma_f64_16x16x4f64(a, w[static_cast<size_t>(kk) * M.pd_cols], acc, 0, 0, 0);
        };
        dbl4 acc = zero, over = zero;
        auto add = [&](dbl4 p) __attribute__((always_inline)) {
            const dbl4 y = p - over, t = acc + y;
            over = (t - acc) - y;
            acc = t;
        };
        int k = k0;
#pragma unroll 4
        for (; k + 4 < k1; k += 8) add(step(k + 4, step(k, zero)));
        if (k < k1) add(step(k, zero));
        return acc - over;
    };
    // row ranges of the split, in steps of 4
    const int q2 = M.pd_k2 / 4, q3 = M.pd_k3 / 4;
    const dbl4 s2 = sum(4 * (q2 * split / kPolySplit), 4 * (q2 * (split + 1) / kPolySplit));
    const dbl4 s3 = sum(M.pd_k2 + 4 * (q3 * split / kPolySplit), M.pd_k2 + 4 * (q3 * (split + 1) / kPolySplit));
    double* p2 = part + (tile * kPolySplit + split) * 256;
    double* p3 = p2 + ntile * kPolySplit * 256;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        p2[r * 64 + lane] = s2[r];
        p3[r * 64 + lane] = s3[r];
    }
    __syncthreads();
    // thread (centre i, column a): sums of the splits, H, He and the energy
    double* es = d + 16 * pitch + 2 * ntile * kPolySplit * 256;  // [16][16 ntile]
    for (int e = threadIdx.x; e < 16 * M.pd_cols; e += nth) {
        const int i = e / M.pd_cols, a = e % M.pd_cols;
        double v = 0.0;
        if (a < nf) {
            const int at = (i >> 2) * 64 + (i & 3) * 16 + (a & 15);
            const double* q = part + (a >> 4) * kPolySplit * 256 + at;
            double h2 = 0.0, h3 = 0.0;
#pragma unroll
            for (int k = 0; k < kPolySplit; ++k) {
                h2 += q[k * 256];
                h3 += q[(ntile * kPolySplit + k) * 256];
            }
            const int s = a / nfn, f = M.pair_tc[t][s] * nfn + (a - s * nfn);
            const size_t at_row = static_cast<size_t>(slot0 + i) * M.n_p + f;
            const double lin = M.pair_w[f], he = lin + (0.5 * h2 + h3 / 3.0);
            S.H[at_row] = lin + (h2 + h3);
            // each term weighted by 1 / its degree: the reference's per-pair
            // energy split (pair_mlip_pair.cpp:159-162)
            S.Hq[at_row] = he;
            v = d[i * pitch + a] * he;
        }
        es[i * M.pd_cols + a] = v;
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        double e = 0.0;
        for (int a = 0; a < nf; ++a) e += es[threadIdx.x * M.pd_cols + a];
        S.Ep[slot0 + threadIdx.x] = e;
    }
}

// Models whose derivative lists are sparse (model_type 1: one entry per
// column): thread per slot over the lists.
__global__ __launch_bounds__(kPairThreads) void k_pair_poly(DevModel M, DevSystem S) {
    const int slot = blockIdx.x * kPairThreads + threadIdx.x;
    if (slot >= S.nblocks * kBlock) return;
    const int atom = S.atom_of_slot[slot];
    if (atom < 0) {
        S.Ep[slot] = 0.0;
        return;
    }
    const double* d = S.D + static_cast<size_t>(slot) * M.n_p;
    double* h = S.H + static_cast<size_t>(slot) * M.n_p;
    cptr<int32_t> off = as_const(M.ph_off);
    cptr<PairHEntry> ent = as_const(M.ph_ent);
    cptr<double> w = as_const(M.pair_w);
    double e = 0.0;
    for (int a = 0; a < M.n_p; ++a) {
        double hs = 0.0, he = 0.0;
        for (int k = off[a]; k < off[a + 1]; ++k) {
            const PairHEntry q = ent[k];
            double v = (q.b >= 0 ? d[q.b] : 1.0) * (q.c >= 0 ? d[q.c] : 1.0);
            hs = fma(q.w, v, hs);
            he = fma(q.ew, v, he);
        }
        h[a] = w[a] + hs;
        // the same derivative with each term weighted by 1 / its degree: the
        // reference's per-pair energy split (pair_mlip_pair.cpp:159-162)
        S.Hq[static_cast<size_t>(slot) * M.n_p + a] = w[a] + he;
        e = fma(d[a], w[a] + he, e);
    }
    S.Ep[slot] = e;
}

// One wave per slot, lane = pair; the slot's H of both neighbor species in
// LDS.  The virial goes over the lanes by a fixed butterfly.  (A thread per
// slot: 1,573 us at 2,048 atoms, ~440 pairs each.)
__global__ __launch_bounds__(kPairThreads) void k_pair_force(DevModel M, DevSystem S) {
    __shared__ double h[2][kMaxFnPair];
    const int slot = blockIdx.x, lane = threadIdx.x;
    const int atom = S.atom_of_slot[slot];
    if (atom < 0) return;
    const int t = S.elem[atom], nfn = M.n_fn;
    for (int e = lane; e < M.n_type * nfn; e += 64)
        h[e / nfn][e % nfn] = S.H[static_cast<size_t>(slot) * M.n_p + M.pair_tc[t][e / nfn] * nfn + e % nfn];
    __syncthreads();
    const double pir = kPiRef / M.cutoff;
    double v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
    for (int64_t p = S.poff[atom] + lane; p < S.pend[atom]; p += 64) {
        double dx, dy, dz, r;
        double gx = 0.0, gy = 0.0, gz = 0.0;
        if (pair_geom(M, S, atom, p, dx, dy, dz, r)) {
            const double* hr = h[S.elem[S.pnbr[p]]];
            double sa, ca;
            sincos(pir * r, &sa, &ca);
            const double fc = 0.5 * (ca + 1.0), fcd = -0.5 * pir * sa;
            double de = 0.0;
            for (int n = 0; n < nfn; ++n) {
                const double d = r - M.mu[n];
                const double b = exp(-M.beta[n] * d * d);
                de = fma(b * (fcd - 2.0 * M.beta[n] * d * fc), hr[n], de);
            }
            const double ir = de / r;
            gx = ir * dx;
            gy = ir * dy;
            gz = ir * dz;
        }
        S.gpair[3 * p] = gx;
        S.gpair[3 * p + 1] = gy;
        S.gpair[3 * p + 2] = gz;
        v0 -= dx * gx;
        v1 -= dy * gy;
        v2 -= dz * gz;
        v3 -= dx * gy;
        v4 -= dx * gz;
        v5 -= dy * gz;
    }
    for (int off = 32; off > 0; off >>= 1) {
        v0 += __shfl_xor(v0, off);
        v1 += __shfl_xor(v1, off);
        v2 += __shfl_xor(v2, off);
        v3 += __shfl_xor(v3, off);
        v4 += __shfl_xor(v4, off);
        v5 += __shfl_xor(v5, off);
    }
    if (lane == 0) {
        double* vo = S.vown + 6 * static_cast<size_t>(atom);
        vo[0] = v0;
        vo[1] = v1;
        vo[2] = v2;
        vo[3] = v3;
        vo[4] = v4;
        vo[5] = v5;
    }
}

// Per directed pair (one wave per slot, lane = pair): energy share e_p =
// sum_n g_n(r) He_{tc,n} (He: the split derivative the polynomial kernel
// leaves in Hq) and the pair's virial del (x) (-g_p); the reference's
// half-pair evdwl is e_p + e_p' over the two directions
// (pair_mlip_pair.cpp:196-212).
__global__ __launch_bounds__(kPairThreads) void k_pair_model_energy(DevModel M, DevSystem S, double* epv) {
    const int slot = blockIdx.x;
    const int atom = S.atom_of_slot[slot];
    if (atom < 0) return;
    const int t = S.elem[atom], nfn = M.n_fn;
    const double* he = S.Hq + static_cast<size_t>(slot) * M.n_p;
    const double pir = kPiRef / M.cutoff;
    for (int64_t p = S.poff[atom] + threadIdx.x; p < S.pend[atom]; p += kPairThreads) {
        double dx, dy, dz, r;
        double e = 0.0, v[6] = {0, 0, 0, 0, 0, 0};
        if (pair_geom(M, S, atom, p, dx, dy, dz, r)) {
            const int s = S.elem[S.pnbr[p]];
            const double* hr = he + M.pair_tc[t][s] * nfn;
            const double fc = 0.5 * (cos(pir * r) + 1.0);
            for (int n = 0; n < nfn; ++n) {
                const double d = r - M.mu[n];
                e = fma(exp(-M.beta[n] * d * d) * fc, hr[n], e);
            }
            const double gx = S.gpair[3 * p], gy = S.gpair[3 * p + 1], gz = S.gpair[3 * p + 2];
            v[0] = -dx * gx;
            v[1] = -dy * gy;
            v[2] = -dz * gz;
            v[3] = -dx * gy;
            v[4] = -dx * gz;
            v[5] = -dy * gz;
        }
        epv[7 * p] = e;
        for (int c = 0; c < 6; ++c) epv[7 * p + 1 + c] = v[c];
    }
}

}  // namespace

hipError_t launch_pair_model_energy(const DevModel& m, const DevSystem& s, double* epv, hipStream_t st) {
    const int nslot = s.nblocks * kBlock;
    if (nslot == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_model_energy, dim3(nslot), dim3(kPairThreads), 0, st, m, s, epv);
    return launched();
}

hipError_t launch_pair_features(const DevModel& m, const DevSystem& s, hipStream_t st) {
    const int nslot = s.nblocks * kBlock;
    if (nslot == 0) return hipSuccess;
    const dim3 grid(nslot), block(kPairThreads);
    if (m.n_fn <= 8)
        hipLaunchKernelGGL(k_pair_feat<8>, grid, block, 0, st, m, s);
    else if (m.n_fn <= 16)
        hipLaunchKernelGGL(k_pair_feat<16>, grid, block, 0, st, m, s);
    else
        hipLaunchKernelGGL(k_pair_feat<32>, grid, block, 0, st, m, s);
    return launched();
}

hipError_t launch_pair_poly(const DevModel& m, const DevSystem& s, hipStream_t st) {
    const int nslot = s.nblocks * kBlock;
    if (nslot == 0) return hipSuccess;
    if (m.pd_cols > 0) {
        const int nf = m.n_type * m.n_fn, ntile = m.pd_cols / 16;
        const size_t lds = sizeof(double) * (16 * static_cast<size_t>((nf + 1) | 1) + 2 * ntile * kPolySplit * 256 +
                                             16 * static_cast<size_t>(m.pd_cols));
        if (lds > lds_limit()) return hipErrorInvalidConfiguration;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_pair_poly_dense),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_pair_poly_dense, dim3(nslot / 16), dim3(64 * ntile * kPolySplit), lds, st, m, s);
        return launched(lds);
    }
    hipLaunchKernelGGL(k_pair_poly, dim3((nslot + kPairThreads - 1) / kPairThreads), dim3(kPairThreads), 0, st, m, s);
    return launched();
}

hipError_t launch_pair_force(const DevModel& m, const DevSystem& s, hipStream_t st) {
    const int nslot = s.nblocks * kBlock;
    if (nslot == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_force, dim3(nslot), dim3(kPairThreads), 0, st, m, s);
    return launched();
}

}  // namespace mlip
