// Order-5/6 invariants of the gtinv model (the table's order-5 and order-6
// families; every factor has l <= 1 there, the kernel takes up to l = 4):
// polynomial features (FEAT) or their share of the adjoint G = dE/da and of
// the energy of linear families.  Reference: the same terms of
// compute_anlm_uniq_products / compute_anlm_linear_term /
// compute_anlm_polynomial_model_correction (src/USER-MLIP/
// pair_mlip_gtinv.cpp:260-343, 451-521) for irreps of order 5 and 6.
//
// Workgroup = one wave on (block of 64 same-species centres, radial index n),
// lane = centre.  The centre's a_{s,l<=lmaxh,m<=0} is staged in LDS (each
// lane reads only its own entries); a visit is one (family, factor position)
// with its terms listed: G_{S,L,-k} += H sum_terms C prod(other factors).
// Families outside the polynomial have the same weights for every centre and
// run merged (k_qhigh_rows), with their energy (1/q) sum_k w_k
// Re(G_k a_{S,L,-k}) (Euler's theorem summed over the q factor positions)
// added to the order-3/4 energy slot 0 of the centre after that kernel.
#include <hip/hip_runtime.h>

#include "device_api.h"
#include "device_common.h"

namespace mlip {

namespace {

using namespace dev;

struct HiTile {
    const double2* a;  // [s][lm][lane]
    int nh, lane;
    __device__ __forceinline__ void get(int s, int l, int m, double& re, double& im) const {
        const int am = m < 0 ? -m : m;
        const double2 v = a[(s * nh + l * (l + 1) / 2 + l - am) * kBlock + lane];
        re = v.x;
        im = v.y;
        if (m > 0) {  // a_{l,m} = (-1)^m conj(a_{l,-m})
            const double sg = (m & 1) ? -1.0 : 1.0;
            re *= sg;
            im *= -sg;
        }
    }
};

template <bool FEAT>
__global__ __launch_bounds__(64) void k_qhigh(DevModel M, DevSystem S) {
    extern __shared__ double2 hi_tile[];
    const int blk = blockIdx.x, n = blockIdx.y, lane = threadIdx.x;
    const int t = S.block_type[blk];
    const int nh = M.n_lmhh;
    for (int s = 0; s < M.n_type; ++s)
        for (int lm = 0; lm < nh; ++lm)
            hi_tile[(s * nh + lm) * kBlock + lane] =
                double2{S.A[a_index(M, blk, n, s, lm, 0, lane)], S.A[a_index(M, blk, n, s, lm, 1, lane)]};
    const HiTile T{hi_tile, nh, lane};
    const int slot = blk * kBlock + lane;
    const int64_t prow = (int64_t)slot * M.n_pr + pcol(M, t, n, 0);
    const int vb = FEAT ? M.hfeat_beg[t] : M.hadj_beg[t];
    const int ve = FEAT ? M.hfeat_end[t] : M.hadj_end[t];
    cptr<VisitHi> vis = as_const(M.hvis);
    cptr<int32_t> term = as_const(M.hterm);
    cptr<double> coef = as_const(M.hcoef);
    for (int vi = vb; vi < ve; ++vi) {
        const VisitHi v = vis[vi];
        const int L = uniform(v.L), Sx = uniform(v.S), pslot = uniform(v.pslot);
        const int no = uniform(v.order) - 1;
        double gr[kMaxLHi + 1], gi[kMaxLHi + 1];
#pragma unroll
        for (int k = 0; k <= kMaxLHi; ++k) gr[k] = gi[k] = 0.0;
        // the factors' (species, l) of the visit in one scalar: indexed in the record
        // they are a read of scratch memory per term and factor (864 atoms, two
        // species, orders 5 and 6 to l = 1 in the polynomial, 2 functions: adjoint
        // 51.4 and features 7.8 ms, now 38.8 and 6.1)
        static_assert(kMaxOrderGpu - 1 <= 5, "twelve bits each");
        uint64_t factors = 0;
#pragma unroll
        for (int o = 0; o < kMaxOrderGpu - 1; ++o) factors |= static_cast<uint64_t>(uniform(v.ls[o])) << (12 * o);
        double d = 0.0;
        for (int ti = uniform(v.tbeg); ti < uniform(v.tend); ++ti) {
            const int code = term[ti];
            const double c = coef[ti];
            const int k = code & 15;
            double pr = 1.0, pi = 0.0;
            for (int o = 0; o < no; ++o) {
                const int ls = static_cast<int>(factors >> (12 * o)) & 0xfff;
                const int mo = ((code >> (4 + 4 * o)) & 15) - 8;
                double yr, yi;
                T.get(ls >> 8, ls & 255, mo, yr, yi);
                const double tr = pr * yr - pi * yi;
                pi = pr * yi + pi * yr;
                pr = tr;
            }
            if (FEAT) {
                double ar, ai;
                T.get(Sx, L, -k, ar, ai);
                d = fma(c, ar * pr - ai * pi, d);
            } else {
#pragma unroll
                for (int kk = 0; kk <= kMaxLHi; ++kk)
                    if (kk == k) {
                        gr[kk] = fma(c, pr, gr[kk]);
                        gi[kk] = fma(c, pi, gi[kk]);
                    }
            }
        }
        if (FEAT) {
            S.D[prow + pslot] = d;
            continue;
        }
        const double H = S.H[prow + pslot];
#pragma unroll
        for (int k = 0; k <= kMaxLHi; ++k) {
            if (k > L) break;
            double* g = S.G + a_index(M, blk, n, Sx, lmh(L, -k), 0, lane);
            g[0] += H * gr[k];
            g[kBlock] += H * gi[k];  // imaginary part: next component, same lane
        }
    }
}

// Merged rows of the linear families (HiRow): the workgroup's four waves share
// the tile of a (block of centres, radial index), every m stored so that a
// factor is one LDS read; a row's terms are dealt over the waves (term ti to
// wave ti mod 4) and the four partial rows summed in wave order through LDS,
// kHiRows rows at a time.  G_{S,L,-k} += scale sum_terms coef prod, energy
// (1/q) w_k Re(G a) per row (Euler).  Bound: LDS reads and FP64 products of
// the terms (the table's order-5/6 invariants: 61,036 terms of 1,090 visits
// per species become the distinct products of 12 rows).  499 atoms of the
// order-6, l <= 20 model: orders 5/6 49.3 ms as one visit per (family, factor
// position) on one wave per (block, n), the evaluation 53.0 -> 3.1 ms.
constexpr int kHiWaves = 4;
constexpr int kHiRows = 8;

__global__ __launch_bounds__(64 * kHiWaves) void k_qhigh_rows(DevModel M, DevSystem S) {
    extern __shared__ double2 hi_tile[];
    const int blk = blockIdx.x, n = blockIdx.y, lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
    const int t = uniform(S.block_type[blk]);
    const int nh = M.n_lmhh, nl = (M.lmaxh + 1) * (M.lmaxh + 1);
    double2* part = hi_tile + M.n_type * nl * kBlock;  // [row of the group][wave][lane]
    for (int e = wave; e < M.n_type * nh; e += kHiWaves) {
        const int s = e / nh, lm = e % nh;
        int l = 0;
        while ((l + 1) * (l + 2) / 2 <= lm) ++l;
        const int m = l * (l + 1) / 2 + l - lm;  // entry of a_{l,-m}
        const double re = S.A[a_index(M, blk, n, s, lm, 0, lane)], im = S.A[a_index(M, blk, n, s, lm, 1, lane)];
        double2* row = hi_tile + (s * nl + l * l + l) * kBlock + lane;
        row[-m * kBlock] = double2{re, im};
        if (m > 0) row[m * kBlock] = (m & 1) ? double2{-re, im} : double2{re, -im};
    }
    __syncthreads();
    cptr<HiRow> rows = as_const(M.hrow);
    cptr<int32_t> term = as_const(M.hrterm) + uniform(M.hrt_off[t]);
    cptr<double> coef = as_const(M.hrcoef) + uniform(M.hrc_off[t] + n * M.hrt_num[t]);
    const double2* tile = hi_tile + lane;
    double eacc = 0.0;
    const int rb = uniform(M.hrow_beg[t]), re = uniform(M.hrow_end[t]);
    for (int r0 = rb; r0 < re; r0 += kHiRows) {
        const int rn = min(kHiRows, re - r0);
        for (int r = 0; r < rn; ++r) {
            const HiRow R = rows[r0 + r];
            const int no = uniform(R.order) - 1;
            double gr = 0.0, gi = 0.0;
            for (int ti = uniform(R.tbeg) + wave; ti < uniform(R.tend); ti += kHiWaves) {
                const int code = term[ti];
                const double c = coef[ti];
                double2 p = tile[(code & 63) * kBlock];
                for (int o = 1; o < no; ++o) {
                    const double2 y = tile[((code >> (6 * o)) & 63) * kBlock];
                    p = double2{p.x * y.x - p.y * y.y, p.x * y.y + p.y * y.x};
                }
                gr = fma(c, p.x, gr);
                gi = fma(c, p.y, gi);
            }
            part[(r * kHiWaves + wave) * kBlock + lane] = double2{gr, gi};
        }
        __syncthreads();
        for (int r = 0; r < rn; ++r) {
            const HiRow R = rows[r0 + r];
            // the rows of one output (orders 5 and 6) add to the same G entry
            if (uniform(R.out) % kHiWaves != wave) continue;
            const int Sx = uniform(R.S), L = uniform(R.L), k = uniform(R.k);
            const double iq = 1.0 / uniform(R.order), scale = M.split ? iq : 1.0;
            double gr = 0.0, gi = 0.0;
#pragma unroll
            for (int w = 0; w < kHiWaves; ++w) {
                const double2 v = part[(r * kHiWaves + w) * kBlock + lane];
                gr += v.x;
                gi += v.y;
            }
            gr *= scale;
            gi *= scale;
            double* g = S.G + a_index(M, blk, n, Sx, lmh(L, -k), 0, lane);
            g[0] += gr;
            g[kBlock] += gi;
            const double2 a = tile[(Sx * nl + L * L + L - k) * kBlock];
            eacc = fma((k == 0 ? 1.0 : 2.0) * iq, gr * a.x - gi * a.y, eacc);
        }
        __syncthreads();
    }
    part[wave * kBlock + lane].x = eacc;
    __syncthreads();
    if (wave == 0) {
        double e = 0.0;
#pragma unroll
        for (int w = 0; w < kHiWaves; ++w) e += part[w * kBlock + lane].x;
        S.Eq34[((size_t)blk * M.n_fn + n) * kWavesPerWg * kBlock + lane] += e;
    }
}

}  // namespace

hipError_t launch_qhigh(const DevModel& m, const DevSystem& s, bool feat, hipStream_t st) {
    if (s.nblocks == 0 || m.lmaxh < 0) return hipSuccess;
    const size_t lds = sizeof(double2) * m.n_type * m.n_lmhh * kBlock;
    if (lds > lds_limit()) return hipErrorInvalidConfiguration;
    if (feat)
        hipLaunchKernelGGL(k_qhigh<true>, dim3(s.nblocks, m.n_fn), dim3(64), lds, st, m, s);
    else if (m.hadj_end[0] > m.hadj_beg[0] || m.hadj_end[1] > m.hadj_beg[1])
        hipLaunchKernelGGL(k_qhigh<false>, dim3(s.nblocks, m.n_fn), dim3(64), lds, st, m, s);
    hipError_t e = launched(lds);
    if (feat || (m.hrow_end[0] == m.hrow_beg[0] && m.hrow_end[1] == m.hrow_beg[1])) return e;
    const size_t rlds = sizeof(double2) * kBlock *
                        (static_cast<size_t>(m.n_type) * (m.lmaxh + 1) * (m.lmaxh + 1) + kHiRows * kHiWaves);
    if (rlds > lds_limit()) return hipErrorInvalidConfiguration;
    const hipError_t ea = hipFuncSetAttribute(reinterpret_cast<const void*>(k_qhigh_rows),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(rlds));
    if (ea != hipSuccess) return first_error(e, ea);
    hipLaunchKernelGGL(k_qhigh_rows, dim3(s.nblocks, m.n_fn), dim3(64 * kHiWaves), rlds, st, m, s);
    return first_error(e, launched(rlds));
}

}  // namespace mlip
