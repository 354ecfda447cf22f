// a_nlm on the FP64 matrix cores, a centre per workgroup, a wave per neighbor
// species.  The product a[n][(l, m, re/im)] = sum_j g_n(r_j) Y(j)[(l, m, re/im)]
// takes four neighbors a step (v_mfma_f64_16x16x4f64: A[i][k] from lane 16 k + i,
// B[k][j] from lane 16 k + j, result r of lane l = D[l / 16 + 4 r][l % 16]), and
// both operands are formed in the lanes that feed them: lane 16 k + i holds
// g_i(r) of neighbor k, and the component i % 2 of column i / 2.  Column c runs
// up m = c and then, when that ends, up m = LT - c (LT = l_max + 1), so that
// eight columns (seven in use at l_max 12) of LT steps hold the whole triangle m
// <= l: one product per step and four neighbors, 13 for the 182 values, with no
// transposition through LDS and no barrier in the loop.  Y is the monic
// recursion P_{l+1} = z P_l - c_{l,m} P_{l-1}, linear in its start, so each lane
// runs it on its own component of (-conj(u))^m; the norm N_{lm} is applied to
// the sums.
//
// Neighbors come in batches of 64, a thread each: sorted by species on the way
// into LDS (ballots, so the order is that of the list), wave 0 writes z, r and
// the cutoff function, wave 1 the powers (-conj(u))^m.
//
// Bound: the FP64 pipe, which matrix and vector instructions share on this
// device (69 and 50 TFLOP/s alone, 56-67 together): per step of four neighbors
// 13 products of 64 cycles and ~90 vector instructions.  256k atoms (137 neighbors,
// l_max 12, 12 functions): 8.2 ms with the order-1/2 features (7.0 without),
// 3,991 atoms 177 us (features from tables in HBM, four barriers a round: 9.4 ms,
// 198 us).  Before: a workgroup of four waves
// with chunks of 16 mixed neighbors, a column per thread through LDS and two
// barriers per chunk, 11.9 ms, and a feature pass that re-read a_nlm, 2.6 ms
// (3,991 atoms: 250 + 62 us).  Also tried: columns formed a lane per neighbor
// and transposed through LDS, 16.1 ms (6,800 vector instructions a wave against
// 3,800).  Three waves a SIMD hold the 13 accumulators and 12 constants with no
// spill, as long as the compiler does not hoist the constants of exp and cos
// out of the loops (this file is built without machine loop-invariant motion).
//
// Reference: PairMLIPGtinv::compute_anlm (src/USER-MLIP/pair_mlip_gtinv.cpp:349-447).
#include <hip/hip_runtime.h>

#include <cstddef>

#include "device_api.h"
#include "device_common.h"

namespace mlip {

namespace {

using namespace dev;

typedef double dbl4 __attribute__((ext_vector_type(4)));

constexpr double kPiRef = 3.141592653589793;  // mlip_basis_function.cpp:26
constexpr int kBatch = 64;  // neighbors per batch
constexpr int kColsFeat = 48;  // order-1/2 features per species (41 for two species and l_max 12)

// T: type of z and the start powers (FP32 in the mixed mode; g, the recursion,
// products and sums are FP64)
template <typename T, int LT>
struct Lds {
    union {
        struct {
            double rr[kBatch], fc[kBatch];
            T z[kBatch];
            T w[kBatch][2 * LT + 1];  // (-conj(u))^m, m < LT; odd pitch
        };
        alignas(16) double buf[kColsBuf];  // a round of the epilogue, read as double2
    };
    double fw[kColsFeat][kQ12Weights];  // order-1/2 features of the centre's species: weights,
    uint32_t fd[kColsFeat];             // order | L | s0 | s1 in 4 bits each, column above
};

template <typename T, int LT, int NS>
__global__ __launch_bounds__(64 * NS) __attribute__((amdgpu_waves_per_eu(3))) void k_anlm_cols(DevModel M, DevSystem S,
                                                                                              int feat) {
    __shared__ Lds<T, LT> L;
    using Shared = Lds<T, LT>;
    static_assert(alignof(Shared) >= sizeof(double2) && offsetof(Shared, buf) == 0, "16-byte reads of buf");
    const int slot = xcd_slot(blockIdx.x, S.nblocks);
    if (slot < 0) return;
    const int atom = S.atom_of_slot[slot];
    if (atom < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int nfn = M.n_fn, nlmh = M.n_lmh;
    const int li = lane & 15, lq = lane >> 4;
    const double mu = li < nfn ? M.mu[li] : 0.0, beta = li < nfn ? M.beta[li] : 0.0;
    // start entries of this lane's two columns (the entry 1, Im w^0 = 0, where
    // it has none) and the step where the second begins
    const int col = li >> 1;
    const int i1 = col <= LT / 2 ? li : 1;
    const int sw = col >= 1 && col <= LT / 2 ? LT - col : LT;
    const int i2 = sw < LT ? 2 * sw + (li & 1) : 1;
    double cn[LT];
#pragma unroll
    for (int t = 1; t < LT; ++t) cn[t] = M.cols->c[t][li];
    dbl4 acc[LT];
#pragma unroll
    for (int t = 0; t < LT; ++t) acc[t] = dbl4{0.0, 0.0, 0.0, 0.0};
    // The features' tables, here because a read behind the stores of a_nlm waits for
    // them
    const int blk = slot / kBlock, slane = slot % kBlock;
    const int ty = S.block_type[blk];
    const int f0 = M.fq12_off[ty], nfe = feat ? M.fq12_off[ty + 1] - f0 : 0;
    for (int k = tid; k < nfe * kQ12Weights; k += 64 * NS)
        L.fw[k / kQ12Weights][k % kQ12Weights] = M.fq12w[static_cast<size_t>(f0) * kQ12Weights + k];
    for (int k = tid; k < nfe; k += 64 * NS) {
        const FeatQ12 f = M.fq12[f0 + k];
        L.fd[k] = f.order | f.L << 4 | f.s0 << 8 | f.s1 << 12 | f.col << 16;
    }
    const int p0 = S.poff[atom], p1 = S.pend[atom];
    const double pir = kPiRef / M.cutoff;
    for (int b0 = p0; b0 < p1; b0 += kBatch) {
        int spec = -1;
        PairDel g{};
        if (b0 + lane < p1) {
            g = pair_del(M, S, atom, b0 + lane);
            if (g.valid) spec = NS == 1 ? 0 : S.elem[S.pnbr[b0 + lane]];
        }
        const uint64_t m0 = __ballot(spec == 0), m1 = NS == 1 ? 0 : __ballot(spec == 1);
        const int n0 = __popcll(m0), n1 = __popcll(m1);
        if (b0 > p0) __syncthreads();
        if (spec >= 0) {
            const uint64_t below = (1ull << lane) - 1ull;
            const int k = spec == 0 ? __popcll(m0 & below) : n0 + __popcll(m1 & below);
            const double ir = 1.0 / g.r;
            if (NS == 1 || wave == 0) {
                L.z[k] = static_cast<T>(g.dz * ir);
                L.rr[k] = g.r;
                L.fc[k] = 0.5 * (cos(pir * g.r) + 1.0);
            }
            if (NS == 1 || wave == 1) {
                const double vx = -(g.dx * ir), vy = g.dy * ir;
                const double v2x = vx * vx - vy * vy, v2y = 2.0 * vx * vy;
                double ex = 1.0, ey = 0.0, ox = vx, oy = vy;  // even and odd powers
                T* w = L.w[k];
#pragma unroll
                for (int m = 0; m < LT; m += 2) {
                    w[2 * m] = static_cast<T>(ex);
                    w[2 * m + 1] = static_cast<T>(ey);
                    double t = ex * v2x - ey * v2y;
                    ey = ex * v2y + ey * v2x;
                    ex = t;
                    if (m + 1 < LT) {
                        w[2 * m + 2] = static_cast<T>(ox);
                        w[2 * m + 3] = static_cast<T>(oy);
                        t = ox * v2x - oy * v2y;
                        oy = ox * v2y + oy * v2x;
                        ox = t;
                    }
                }
            }
        }
        __syncthreads();
        const int b = wave == 0 ? 0 : n0, e = wave == 0 ? n0 : n0 + n1;
        // operands of the next step are read a step ahead
        int q = min(b + lq, kBatch - 1);
        double r = L.rr[q], fc = L.fc[q];
        T zt = L.z[q], s1t = L.w[q][i1], s2t = L.w[q][i2];
        for (int j = b; j < e; j += 4) {
            // the last step's surplus neighbors (stale or the other species') count as zero
            const bool ok = j + lq < e;
            const double d = r - mu;
            const double gn = ok ? exp(-beta * (d * d)) * fc : 0.0;
            const double z = ok ? static_cast<double>(zt) : 0.0, s2 = ok ? static_cast<double>(s2t) : 0.0;
            double y1 = ok ? static_cast<double>(s1t) : 0.0, y2 = 0.0;
            q = min(j + 4 + lq, kBatch - 1);
            r = L.rr[q];
            fc = L.fc[q];
            zt = L.z[q];
            s1t = L.w[q][i1];
            s2t = L.w[q][i2];
            acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(gn, y1, acc[0], 0, 0, 0);
#pragma unroll
            for (int t = 1; t < LT; ++t) {
                double yn = t == 1 ? z * y1 : fma(z, y1, cn[t] * y2);
                if (t > LT / 2) yn = sw == t ? s2 : yn;
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(gn, yn, acc[t], 0, 0, 0);
                y2 = y1;
                y1 = yn;
            }
        }
    }
    // norms, then a_nlm to HBM: result r of lane (lq, li) is radial index lq + 4 r.
    // Each step's table reads wait for the stores before them, which paces these
    // 8-byte stores so that the L2 gathers the lines of neighboring slots: all
    // tables first, then all stores, took 9.4 ms instead of 8.2.
    double* ab = S.A + a_index(M, blk, 0, wave, 0, 0, slane);
    const uint32_t np = static_cast<uint32_t>(NS * nlmh) * 2 * kBlock;  // stride of a radial index
    int lmc[LT];
#pragma unroll
    for (int t = 0; t < LT; ++t) {
        const double nrm = M.cols->norm[t][li];
        lmc[t] = M.cols->lmc[t][li];
        const uint32_t at = lq * np + static_cast<uint32_t>(lmc[t]) * kBlock;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[t][r] *= nrm;
            if (lmc[t] >= 0 && lq + 4 * r < nfn) (ab + 4 * r * np)[at] = acc[t][r];
        }
    }
    if (!feat) return;
    // Order-1/2 polynomial features of this centre from the a_nlm it holds, four
    // radial indices (one result register) a round: a of all species into LDS
    // as [n][s][lm](re, im), thread per (feature, n) with n fastest (the
    // features are listed by L, so a wave's items have nearly equal lengths),
    // the round's row segment (zero where no order-1/2 family writes) stored as
    // one run of the slot's compact row.  Two barriers a round: the segment
    // alternates between two places, so that it is stored while the next round
    // begins.
    const int w = M.prange[ty][1] - M.prange[ty][0];
    double* as = L.buf;                        // [n][s][lm] (re, im)
    double* segs = as + 4 * NS * nlmh * 2;     // two of [n][rank - lo]
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int r0 = 4 * r, rn = min(4, nfn - r0);
        if (rn <= 0) break;
        double* seg = segs + (r & 1) * 4 * w;
#pragma unroll
        for (int t = 0; t < LT; ++t)
            if (lmc[t] >= 0 && lq < rn) as[((lq * NS + wave) * nlmh) * 2 + lmc[t]] = acc[t][r];
        for (int e = tid; e < rn * w; e += 64 * NS) seg[e] = 0.0;
        __syncthreads();
        for (int it = tid; it < nfe * rn; it += 64 * NS) {
            const int fi = it / rn, nl = it - fi * rn;
            const uint32_t f = L.fd[fi];
            const double* wt = L.fw[fi];
            const double2* x = reinterpret_cast<const double2*>(as) + (nl * NS + (f >> 8 & 15)) * nlmh;
            double d;
            if ((f & 15) == 1) {
                d = wt[0] * x[0].x;
            } else {
                // the order-1/2 pass's pair-summed form, same order of terms;
                // four at a time (weights past L are zero), their reads together
                const double2* y = reinterpret_cast<const double2*>(as) + (nl * NS + (f >> 12 & 15)) * nlmh;
                const int fl = f >> 4 & 15, b = fl * (fl + 1) / 2 + fl;  // lmh(L, 0); lmh(L, -k) = b - k
                d = 0.0;
                for (int k = 0; k <= fl; k += 4) {
                    double2 xv[4], yv[4];
                    double wv[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int at = b - min(k + j, fl);
                        xv[j] = x[at];
                        yv[j] = y[at];
                        wv[j] = wt[k + j];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) d = fma(wv[j], xv[j].x * yv[j].x + xv[j].y * yv[j].y, d);
                }
            }
            seg[nl * w + (f >> 16)] = d;
        }
        __syncthreads();
        double* drow = S.D + static_cast<size_t>(slot) * M.n_pr + static_cast<size_t>(r0) * w;
        for (int e = tid; e < rn * w; e += 64 * NS) drow[e] = seg[e];
    }
}

// steps of the instance that holds l_max
int cols_steps(int maxl) { return maxl < 5 ? 5 : maxl < 9 ? 9 : kColsMaxL + 1; }

template <typename T, int NS>
hipError_t launch_cols(const DevModel& m, const DevSystem& s, int feat, hipStream_t st) {
    const int grid = 8 * kBlock * ((s.nblocks + 7) / 8), lt = cols_steps(m.maxl);
    const auto k = lt == 5 ? k_anlm_cols<T, 5, NS> : lt == 9 ? k_anlm_cols<T, 9, NS> : k_anlm_cols<T, 13, NS>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(64 * NS), 0, st, m, s, feat);
    return launched();
}

}  // namespace

void build_cols_tables(int maxl, ColsTab& t) {
    const int lt = cols_steps(maxl);
    // N_mm without the sign that (-conj(u))^m carries, N_lm = N_{l-1,m} sqrt((4
    // l^2 - 1) / (l^2 - m^2))
    long double norm[kColsMaxL + 1][kColsMaxL + 1], dg = 1.0L / sqrtl(4.0L * 3.14159265358979323846264338327950288L);
    for (int m = 0; m < lt; ++m) {
        if (m > 0) dg *= -sqrtl((2.0L * m + 1.0L) / (2.0L * m));
        norm[m][m] = dg;
        for (int l = m + 1; l < lt; ++l)
            norm[l][m] = norm[l - 1][m] * sqrtl((4.0L * l * l - 1.0L) / (1.0L * l * l - 1.0L * m * m));
    }
    for (int k = 0; k < kColsMaxL + 1; ++k)
        for (int i = 0; i < 16; ++i) {
            t.c[k][i] = t.norm[k][i] = 0.0;
            t.lmc[k][i] = -1;
            const int col = i / 2, m = k < lt - col ? col : lt - col, l = k < lt - col ? col + k : k;
            if (col > lt / 2 || k >= lt) continue;
            if (l > m) t.c[k][i] = -static_cast<double>((1.0L * (l - 1) * (l - 1) - 1.0L * m * m) / (4.0L * (l - 1) * (l - 1) - 1.0L));
            if (l > maxl) continue;
            t.norm[k][i] = static_cast<double>(norm[l][m]);
            t.lmc[k][i] = 2 * (l * (l + 1) / 2 + l - m) + i % 2;
        }
}

bool anlm_cols_fits(const DevModel& m) { return m.cols != nullptr && m.maxl <= kColsMaxL && m.n_fn <= 16 && m.n_type <= 2; }

// the features' tables, a round's a_nlm and two row segments fit the LDS
bool anlm_cols_features(const DevModel& m) {
    for (int t = 0; t < m.n_type; ++t) {
        const int features = m.fq12_off[t + 1] - m.fq12_off[t], w = m.prange[t][1] - m.prange[t][0];
        if (features > kColsFeat || w > 65535 || 4 * (2 * m.n_type * m.n_lmh + 2 * w) > kColsBuf) return false;
    }
    return true;
}

hipError_t launch_anlm_cols(const DevModel& m, const DevSystem& s, int feat, int precision, hipStream_t st) {
    if (precision == kMixed) return m.n_type == 1 ? launch_cols<float, 1>(m, s, feat, st) : launch_cols<float, 2>(m, s, feat, st);
    return m.n_type == 1 ? launch_cols<double, 1>(m, s, feat, st) : launch_cols<double, 2>(m, s, feat, st);
}

}  // namespace mlip
