// Forces on the matrix cores (l_max <= 12, up to 16 radial functions): a
// workgroup per centre, its neighbors sorted by species into tiles of 16, a wave
// per tile.  Per pair
//   Gq_lm = sum_n g_n G_nlm,  Gp_lm = sum_n g'_n G_nlm
//   dE/d(del) = sum_lm w_m Re(Gp Y) rhat + w_m Re(Gq . grad Y),  w_0 = 1, w_{m<0} = 2
// The two sums over n are products G^T [rows][n] x g [n][pair] of 16 rows and 16
// pairs, four n a step (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32: A[i][k]
// from lane 16 k + i, B[k][j] from lane 16 k + j; result r of lane l is row l /
// 16 + 4 r in FP64 and 4 (l / 16) + r in FP32, of pair l % 16).  Lane 16 k + j
// therefore forms g_n of pair j for n = 4 s + k, and quarter q of the wave gets
// four rows of each product: re and im of two entries.  The centre's G (both
// species, w_m and the norm of Y_lm multiplied in) is staged in LDS in operand
// order, with the rows of quarter q the entries l = m, m + 1, ... of its columns
// m = q, 4 + q, ...: every quarter runs the columns of one pass of four in step.
// With Q_l the monic column polynomial (Q_{l+1} = z Q_l - c_{l,m} Q_{l-1}) and D_l
// its z-derivative, a column keeps
//   Sp = sum_l Q Gp,  Sq = sum_l Q Gq,  Sd = sum_l D Gq
// in T, folded in FP64 with the column's power of u = x + i y:
//   er += Re(Sp ubar^m),  t += (Re(SE ubar^{m-1} - SB ubar^{m+1}) / 2,
//                               Im(SE ubar^{m-1} + SB ubar^{m+1}) / 2, -Re(SA ubar^m))
//   SA = m z Sq - (1-z^2) Sd, SB = m Sq + z Sd, SE = m (1+z^2) Sq - z (1-z^2) Sd
// (m = 0: SE ubar^{-1} = -z Sd u), and the quarters are added at the end.
//
// Bound: the FP64 pipe (vector and matrix instructions share it; 84 products of
// 64 cycles and ~700 vector instructions per tile at l_max 12 and 12 functions).
// 256k atoms (137 neighbors, l_max 12, 12 functions): 11.2 ms, matrix instructions
// busy 50 % and vector issue 33 % of the SIMD cycles;
// 3,991 atoms 202 us; mixed, 31k atoms: 0.96 ms.  Before: a thread per pair with G
// read as LDS broadcasts (bound by them: one 16-byte read per four FMAs), 14.9 ms,
// 293 us and 1.29 ms.  No spill is affordable here: with 464 bytes of scratch per
// lane 27 ms, 120 bytes 19.7 ms; the scheduler is therefore held to one product
// ahead, and the file is built without machine loop-invariant motion.  Waves per
// workgroup at 256k atoms: 20.4, 15.0, 13.0 and 11.2 ms with 1 to 4.
//
// Reference: PairMLIPGtinv::compute_partial_force (src/USER-MLIP/pair_mlip_gtinv.cpp:161-256).
#include <hip/hip_runtime.h>

#include "device_api.h"
#include "device_common.h"

namespace mlip {

namespace {

using namespace dev;

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

constexpr double kPiRef = 3.141592653589793;  // mlip_basis_function.cpp:26
constexpr int kFcBatch = 176;                 // neighbors per batch: three workgroups share a CU's LDS at 12 functions
constexpr int kFcChunks = (kFcBatch + 63) / 64;
constexpr int kFcMaxWaves = 4;

// passes of four columns, entries and product tiles for LT = l_max + 1 levels
template <int LT>
struct Shape {
    static constexpr int np = (LT + 3) / 4;
    static constexpr int start(int p) { return p * LT - 2 * p * (p - 1); }
    static constexpr int entries = start(np);
    static constexpr int tiles = (entries + 1) / 2;
};

template <typename T>
struct Quad;
template <>
struct Quad<double> {
    using type = dbl4;
    static __device__ __forceinline__ dbl4 mfma(double a, double b, dbl4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // (quarter, result) of product row i
    static __device__ __forceinline__ int quarter(int i) { return i & 3; }
    static __device__ __forceinline__ int result(int i) { return i >> 2; }
};
template <>
struct Quad<float> {
    using type = flt4;
    static __device__ __forceinline__ flt4 mfma(float a, float b, flt4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int quarter(int i) { return i >> 2; }
    static __device__ __forceinline__ int result(int i) { return i & 3; }
};

template <typename T>
struct FcLds {
    double x[kFcBatch], y[kFcBatch], z[kFcBatch], rr[kFcBatch], fc[kFcBatch], fd[kFcBatch];
    uint16_t order[kFcBatch];        // sorted position -> neighbor of the batch
    uint64_t mask[2][kFcChunks];     // neighbors of each species per 64
    double mu[16], beta[16];
    T c[kForceEntries][4];
    double vred[6][kFcMaxWaves];
};

// LT: levels; KS: steps of four radial functions
template <typename T, int LT, int KS>
__global__ __launch_bounds__(64 * kFcMaxWaves) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 3))) void
k_force_cols(DevModel M, DevSystem S) {
    using V4 = typename Quad<T>::type;
    using Sh = Shape<LT>;
    extern __shared__ __attribute__((aligned(16))) unsigned char fc_dyn[];
    T* Gs = reinterpret_cast<T*>(fc_dyn);  // [species][tile][step][lane]
    __shared__ FcLds<T> L;
    const int slot = xcd_slot(blockIdx.x, S.nblocks);
    if (slot < 0) return;
    const int atom = S.atom_of_slot[slot];
    if (atom < 0) return;
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = uniform(tid >> 6), nwave = nthr >> 6;
    const int lj = lane & 15, lq = lane >> 4;
    const int nfn = M.n_fn, ns = M.n_type;
    const ForceTab* tab = M.ftab;
    const int p0 = S.poff[atom], p1 = S.pend[atom];
    const double pir = kPiRef / M.cutoff;
    double va = 0.0, vb = 0.0;  // virial: xx, yy, zz and xy, xz, yz in quarters 0, 1, 2

    // G of four product tiles of this wave to registers and on to LDS; entries
    // past the model's read an in-range one and store zero, so that all reads
    // are in flight together
    constexpr int kHold = 4;
    const int blk = slot / kBlock, sl = slot % kBlock;
    const int q4 = 4 * Quad<T>::quarter(lj) + Quad<T>::result(lj);
    double gv[kHold][2][KS], fac[kHold];
    auto load_g = [&](int tb) __attribute__((always_inline)) {
        int row[kHold];
#pragma unroll
        for (int i = 0; i < kHold; ++i) {
            const int t = min(tb + i * nwave, Sh::tiles - 1);
            row[i] = tab->row[t][q4];
            fac[i] = tab->fac[t][q4];  // 0 where the entry is none of the model's
        }
#pragma unroll
        for (int i = 0; i < kHold; ++i)
#pragma unroll
            for (int k = 0; k < 2 * KS; ++k) {
                const int sp = k / KS, n = 4 * (k % KS) + lq, r = max(row[i], 0);
                gv[i][sp][k % KS] =
                    sp < ns ? S.G[a_index(M, blk, min(n, nfn - 1), sp, r >> 1, r & 1, sl)] : 0.0;
            }
    };
    auto store_g = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kHold; ++i) {
            const int t = tb + i * nwave;
            if (t >= Sh::tiles) break;
#pragma unroll
            for (int k = 0; k < 2 * KS; ++k)
                if (k / KS < ns)
                    Gs[64 * ((k / KS) * Sh::tiles * KS + t * KS + k % KS) + lane] =
                        4 * (k % KS) + lq < nfn && fac[i] != 0.0 ? static_cast<T>(gv[i][k / KS][k % KS] * fac[i]) : T(0);
        }
    };
    for (int tb = wave; tb < Sh::tiles; tb += kHold * nwave) {
        load_g(tb);
        store_g(tb);
    }
    for (int k = tid; k < Sh::entries * 4; k += nthr) L.c[k >> 2][k & 3] = static_cast<T>(tab->c[k >> 2][k & 3]);
    if (tid < 16) {
        L.mu[tid] = tid < nfn ? M.mu[tid] : 0.0;
        L.beta[tid] = tid < nfn ? M.beta[tid] : 0.0;
    }

    for (int b0 = p0; b0 < p1; b0 += kFcBatch) {
        const int nb = min(kFcBatch, p1 - b0);
        if (b0 > p0) __syncthreads();
        for (int c = wave; c < kFcChunks; c += nwave) {
            const int k = 64 * c + lane;
            int spec = -1;
            if (k < nb) {
                const PairDel g = pair_del(M, S, atom, b0 + k);
                if (g.valid) {
                    spec = S.elem[S.pnbr[b0 + k]];
                    const double ir = 1.0 / g.r;
                    L.x[k] = g.dx * ir;
                    L.y[k] = g.dy * ir;
                    L.z[k] = g.dz * ir;
                    L.rr[k] = g.r;
                    double sa, ca;
                    sincos(pir * g.r, &sa, &ca);
                    L.fc[k] = 0.5 * (ca + 1.0);
                    L.fd[k] = -0.5 * pir * sa;
                } else {
                    double* o = S.gpair + 3 * static_cast<size_t>(b0 + k);
                    o[0] = o[1] = o[2] = 0.0;
                }
            }
            const uint64_t m0 = __ballot(spec == 0), m1 = __ballot(spec == 1);
            if (lane == 0) {
                L.mask[0][c] = m0;
                L.mask[1][c] = m1;
            }
        }
        __syncthreads();
        int n0 = 0, n1 = 0;
#pragma unroll
        for (int c = 0; c < kFcChunks; ++c) {
            n0 += __popcll(L.mask[0][c]);
            n1 += __popcll(L.mask[1][c]);
        }
        for (int c = wave; c < kFcChunks; c += nwave) {
            int k0 = 0, k1 = n0;
            for (int e = 0; e < c; ++e) {
                k0 += __popcll(L.mask[0][e]);
                k1 += __popcll(L.mask[1][e]);
            }
            const uint64_t bit = 1ull << lane, m0 = L.mask[0][c], m1 = L.mask[1][c];
            if (m0 & bit) L.order[k0 + __popcll(m0 & (bit - 1))] = static_cast<uint16_t>(64 * c + lane);
            if (m1 & bit) L.order[k1 + __popcll(m1 & (bit - 1))] = static_cast<uint16_t>(64 * c + lane);
        }
        __syncthreads();
        const int t0 = uniform((n0 + 15) >> 4), tn = t0 + uniform((n1 + 15) >> 4);
        for (int tile = wave; tile < tn; tile += nwave) {
            const bool sp = tile >= t0;
            const int at = sp ? n0 + 16 * (tile - t0) + lj : 16 * tile + lj, end = sp ? n0 + n1 : n0;
            const bool ok = at < end;  // surplus lanes repeat the tile's first pair
            const int k = L.order[ok ? at : at - lj];
            const double x = L.x[k], y = L.y[k], zd = L.z[k];
            T g[KS], gd[KS];
            {
                const double r = L.rr[k], fc = L.fc[k], fd = L.fd[k];
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    // padded n >= n_fn meet zero rows of G
                    const double dd = r - L.mu[4 * s + lq], be = L.beta[4 * s + lq];
                    const double b = exp(-be * (dd * dd));
                    g[s] = static_cast<T>(b * fc);
                    gd[s] = static_cast<T>(b * (fd - 2.0 * be * dd * fc));
                }
            }
            const T* Ga = Gs + (sp ? Sh::tiles * KS * 64 : 0) + lane;
            auto product = [&](int t, V4& dq, V4& dp) __attribute__((always_inline)) {
                dq = V4{0, 0, 0, 0};
                dp = V4{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const T a = Ga[(t * KS + s) * 64];
                    dq = Quad<T>::mfma(a, g[s], dq);
                    dp = Quad<T>::mfma(a, gd[s], dp);
                }
            };
            const T z = static_cast<T>(zd);
            const double zz = 1.0 - zd * zd;
            const double u2x = x * x - y * y, u2y = -2.0 * x * y;  // ubar^2
            const double u4x = u2x * u2x - u2y * u2y, u4y = 2.0 * u2x * u2y;
            // ubar^{m-1} of the quarter's column (m = 0: u, see above)
            double cx = lq == 0 ? x : lq == 1 ? 1.0 : lq == 2 ? x : u2x;
            double cy = lq == 0 ? y : lq == 1 ? 0.0 : lq == 2 ? -y : u2y;
            double er = 0.0, tx = 0.0, ty = 0.0, tz = 0.0;
            V4 dq, dp, nq, np;
            product(0, nq, np);
#pragma unroll
            for (int p = 0; p < Sh::np; ++p) {
                T spr, spi, sqr, sqi, sdr = 0, sdi = 0;
                T q1 = 1, q2 = 0, d1 = 0, d2 = 0;  // Q and D of the last two levels
#pragma unroll
                for (int o = 0; o < LT - 4 * p; ++o) {
                    const int e = Sh::start(p) + o;
                    if (e % 2 == 0) {
                        __builtin_amdgcn_sched_barrier(0);  // one product ahead, not more: registers
                        dq = nq;
                        dp = np;
                        if (e / 2 + 1 < Sh::tiles) product(e / 2 + 1, nq, np);
                    }
                    const int r = 2 * (e % 2);
                    if (o == 0) {
                        spr = dp[r];
                        spi = dp[r + 1];
                        sqr = dq[r];
                        sqi = dq[r + 1];
                    } else {
                        if (o == 1) {
                            q2 = 1;
                            q1 = z;
                            d1 = 1;
                            sdr = dq[r];
                            sdi = dq[r + 1];
                        } else {
                            const T nc = L.c[e][lq];
                            const T qn = fma(z, q1, nc * q2);
                            const T dn = fma(z, d1, fma(nc, d2, q1));
                            q2 = q1;
                            q1 = qn;
                            d2 = d1;
                            d1 = dn;
                            sdr = fma(d1, dq[r], sdr);
                            sdi = fma(d1, dq[r + 1], sdi);
                        }
                        spr = fma(q1, dp[r], spr);
                        spi = fma(q1, dp[r + 1], spi);
                        sqr = fma(q1, dq[r], sqr);
                        sqi = fma(q1, dq[r + 1], sqi);
                    }
                }
                const double fm = 4 * p + lq;
                double c0x = cx * x + cy * y, c0y = cy * x - cx * y;  // ubar^m
                double kd = zd * zz;
                if (p == 0 && lq == 0) {
                    c0x = 1.0;
                    c0y = 0.0;
                    kd = zd;
                }
                const double cpx = c0x * x + c0y * y, cpy = c0y * x - c0x * y;
                const double Sqr = sqr, Sqi = sqi, Sdr = sdr, Sdi = sdi;
                er += static_cast<double>(spr) * c0x - static_cast<double>(spi) * c0y;
                const double mz = fm * zd, ke = fma(mz, zd, fm);
                const double sar = mz * Sqr - zz * Sdr, sai = mz * Sqi - zz * Sdi;
                const double sbr = fm * Sqr + zd * Sdr, sbi = fm * Sqi + zd * Sdi;
                const double ser = ke * Sqr - kd * Sdr, sei = ke * Sqi - kd * Sdi;
                tx += (ser * cx - sei * cy) - (sbr * cpx - sbi * cpy);
                ty += (ser * cy + sei * cx) + (sbr * cpy + sbi * cpx);
                tz -= sar * c0x - sai * c0y;
                if (p + 1 < Sh::np) {
                    const double t = cx * u4x - cy * u4y;
                    cy = cx * u4y + cy * u4x;
                    cx = t;
                    if (p == 0 && lq == 0) {  // ubar^3
                        cx = u2x * x + u2y * y;
                        cy = u2y * x - u2x * y;
                    }
                }
            }
#pragma unroll
            for (int off = 16; off < 64; off <<= 1) {
                er += __shfl_xor(er, off);
                tx += __shfl_xor(tx, off);
                ty += __shfl_xor(ty, off);
                tz += __shfl_xor(tz, off);
            }
            const double r = L.rr[k], ir = 1.0 / r;
            const double fx = er * x + 0.5 * tx * ir, fy = er * y + 0.5 * ty * ir, fz = er * zd + tz * ir;
            if (ok && lq < 3) {
                const double f = lq == 0 ? fx : lq == 1 ? fy : fz;
                S.gpair[3 * static_cast<size_t>(b0 + k) + lq] = f;
                // virial: del (x) F_centre with F_centre = -dE/d(del)
                va -= r * (lq == 0 ? x : lq == 1 ? y : zd) * f;
                vb -= r * (lq == 2 ? y : x) * (lq == 0 ? fy : fz);
            }
        }
    }
    // fixed-order reduction: butterfly within each quarter, then over waves
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        va += __shfl_xor(va, off);
        vb += __shfl_xor(vb, off);
    }
    if (lj == 0 && lq < 3) {
        L.vred[lq][wave] = va;
        L.vred[3 + lq][wave] = vb;
    }
    __syncthreads();
    if (tid < 6) {
        double s = 0.0;
        for (int k = 0; k < nwave; ++k) s += L.vred[tid][k];
        S.vown[6 * static_cast<size_t>(atom) + tid] = s;
    }
}

// levels of the instance that holds l_max
int force_levels(int maxl) { return maxl < 5 ? 5 : maxl < 9 ? 9 : kColsMaxL + 1; }

template <typename T, int LT, int KS>
hipError_t launch_fc(const DevModel& m, const DevSystem& s, int threads, hipStream_t st) {
    const size_t lds = sizeof(T) * 64 * KS * Shape<LT>::tiles * m.n_type;
    if (lds + sizeof(FcLds<T>) > lds_limit()) return hipErrorInvalidConfiguration;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_force_cols<T, LT, KS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_force_cols<T, LT, KS>), dim3(8 * kBlock * ((s.nblocks + 7) / 8)), dim3(threads), lds, st, m, s);
    return launched();
}

template <typename T, int LT>
hipError_t launch_fc_l(const DevModel& m, const DevSystem& s, int threads, hipStream_t st) {
    switch ((m.n_fn + 3) / 4) {
        case 1: return launch_fc<T, LT, 1>(m, s, threads, st);
        case 2: return launch_fc<T, LT, 2>(m, s, threads, st);
        case 3: return launch_fc<T, LT, 3>(m, s, threads, st);
        default: return launch_fc<T, LT, 4>(m, s, threads, st);
    }
}

template <typename T>
hipError_t launch_fc_t(const DevModel& m, const DevSystem& s, int threads, hipStream_t st) {
    const int lt = force_levels(m.maxl);
    if (lt == 5) return launch_fc_l<T, 5>(m, s, threads, st);
    if (lt == 9) return launch_fc_l<T, 9>(m, s, threads, st);
    return launch_fc_l<T, kColsMaxL + 1>(m, s, threads, st);
}

}  // namespace

void build_force_tables(int maxl, ForceTab& t) {
    const int lt = force_levels(maxl);
    for (int k = 0; k < (kForceEntries + 1) / 2; ++k)
        for (int i = 0; i < 16; ++i) {
            t.row[k][i] = -1;
            t.fac[k][i] = 0.0;
        }
    long double diag[kColsMaxL + 4];
    diag[0] = 1.0L / sqrtl(4.0L * 3.14159265358979323846264338327950288L);
    for (int m = 1; m <= maxl; ++m) diag[m] = diag[m - 1] * sqrtl((2.0L * m + 1.0L) / (2.0L * m));
    int e = 0;
    for (int p = 0; 4 * p < lt; ++p)
        for (int o = 0; o < lt - 4 * p; ++o, ++e)
            for (int q = 0; q < 4; ++q) {
                const int m = 4 * p + q, l = m + o;
                const long double b = 1.0L * (l - 1) * (l - 1);
                t.c[e][q] = o >= 2 ? -static_cast<double>((b - 1.0L * m * m) / (4.0L * b - 1.0L)) : 0.0;
                if (l > maxl) continue;
                long double n = diag[m];
                for (int j = m + 1; j <= l; ++j) n *= sqrtl((4.0L * j * j - 1.0L) / (1.0L * j * j - 1.0L * m * m));
                for (int c = 0; c < 2; ++c) {
                    t.row[e / 2][4 * q + 2 * (e % 2) + c] = 2 * (l * (l + 1) / 2 + l - m) + c;
                    t.fac[e / 2][4 * q + 2 * (e % 2) + c] = static_cast<double>(m == 0 ? n : 2.0L * n);
                }
            }
}

bool force_cols_fits(const DevModel& m) { return m.ftab != nullptr && m.n_fn <= 16 && m.n_type <= 2; }

hipError_t launch_force_cols(const DevModel& m, const DevSystem& s, int precision, int threads, hipStream_t st) {
    return precision == kMixed ? launch_fc_t<float>(m, s, threads, st) : launch_fc_t<double>(m, s, threads, st);
}

}  // namespace mlip
