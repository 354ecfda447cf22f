// Order-3 share of the adjoint G = dE/da of families outside the polynomial
// (their weights are the same for every centre of a species), by output m:
//   G_{S,L,-k} += sum_{la <= lb} sum_{sa,sb} w_{S,L,sa,sb}
//                 sum_{ma} C^L_{la,lb}(k, ma) a_{sa,la,ma} a_{sb,lb,k-ma}
// For fixed (la, lb, k) the products a_{sa,la,ma} a_{sb,lb,k-ma} do not depend
// on L, and the coefficient blocks of the species combinations and of both
// output species are multiples of one another (one irrep): so each product is
// formed once for every L >= k with |la - lb| <= L <= la + lb and both S, summed over ma
// into t_{L,(sa,sb)}, and only those sums meet the weights.  (Reference: the
// same terms of compute_anlm_linear_term and compute_anlm_uniq_products,
// src/USER-MLIP/pair_mlip_gtinv.cpp:300-317, 451-478.)
//
// Workgroup = 12 waves on one (block of 64 same-species centres, radial index);
// the a_nlm tile l <= lmaxq3, m <= 0, both species, in LDS.  A wave walks records
// (la, lb, up to kQ3N consecutive L of one parity) of one (k, parity of L) at a
// time, G_{S,L,-k} of that segment in registers.  The records of all segments
// in a row are cut into twelve ranges by modelled cost (model.cpp); a segment
// that a cut divides is written by the wave that holds its end and the other
// parts are added after a barrier, in order.  A step's factors come as tile
// offsets in the coefficient stream (Rec3), one step ahead.
//
// The waves also add the order-1/2 families to the rows they write (H of the
// block's centres staged in LDS) and form the rows above the tile.
//
// Bound: FP64 VALU with one 16-byte LDS read per product, latency at 3 waves
// per SIMD.  Per (atom, radial index) of the order-4 benchmark model (l <= 8) the
// order-3 terms were ~25,000 products of 6 FMA-rate instructions; here they are
// 5,500 products of 4, and 16,000 coefficient FMA pairs.  At 256k atoms orders 1-4
// took 36.4 ms as one visit per (family, factor position) with 3/4 of the
// instructions address, descriptor and product work; k_q3 takes 15.6 ms and k_q4
// 1.5 ms (vector issue 57 % of the SIMD cycles, the waves wait half of theirs); with
// the factors' addresses formed from m in each step and the divided rows read and
// written one by one it was 18.2 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_api.h"
#include "device_common.h"
#include "q3_rows.h"
#include "q4_terms.h"

namespace mlip {

namespace {

using namespace dev;

constexpr int kQ3Threads = 64 * kWavesPerWg;
constexpr int kHPitch = kBlock + 1;  // doubles between ranks of the staged H

// a_{l,m} for m > 0 is (-1)^m conj(a_{l,-m}): the sign is in the coefficients,
// the conjugation a flip of the imaginary part's sign bit.
__device__ __forceinline__ double flip(double v, unsigned mask) {
    return __hiloint2double(static_cast<int>(__double2hiint(v) ^ mask), __double2loint(v));
}

// One step's operands: both species' factors, the coefficients and the next
// step's factors (Rec3).
template <int NT, int N>
struct Step {
    double2 x[NT], y[NT];
    double c[N];
    unsigned fx, fy;   // sign masks
    unsigned nx, ny;   // next step's factors
    __device__ __forceinline__ void load(const double2* As, int ss, unsigned dx, unsigned dy, cptr<double> cp) {
        const char* base = reinterpret_cast<const char*>(As);
        const double2* px = reinterpret_cast<const double2*>(base + (dx & ~kQ3Conj));
        const double2* py = reinterpret_cast<const double2*>(base + (dy & ~kQ3Conj));
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            x[s] = px[s * ss];
            y[s] = py[s * ss];
        }
        fx = dx & kQ3Conj;
        fy = dy & kQ3Conj;
        const uint64_t code = reinterpret_cast<cptr<uint64_t>>(cp)[0];
        nx = static_cast<unsigned>(code);
        ny = static_cast<unsigned>(code >> 32);
#pragma unroll
        for (int j = 0; j < N; ++j) c[j] = cp[1 + j];
    }
    // FIRST: the sums start here
    template <int V, bool FIRST = false>
    __device__ __forceinline__ void use(double (&tr)[N][V], double (&ti)[N][V]) {
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            x[s].y = flip(x[s].y, fx);
            y[s].y = flip(y[s].y, fy);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            // V = 4: (sa, sb) = v / 2, v % 2; V = 3: (0,0), (0,1), (1,1)
            const int sa = V == 4 ? v / 2 : V == 3 ? v / 2 : 0, sb = V == 4 ? v % 2 : V == 3 ? (v + 1) / 2 : 0;
            const double pr = fma(x[sa].x, y[sb].x, -(x[sa].y * y[sb].y));
            const double pi = fma(x[sa].x, y[sb].y, x[sa].y * y[sb].x);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                tr[j][v] = FIRST ? c[j] * pr : fma(c[j], pr, tr[j][v]);
                ti[j][v] = FIRST ? c[j] * pi : fma(c[j], pi, ti[j][v]);
            }
        }
    }
};

// G_{S,L0 + 2 (I0 + j)} += sum_v w t_{j,v}, every index a compile-time constant
// from the start (recursion over j, S and v), and each case of the switch on i0
// closed by an assembler comment of its own: otherwise the compiler merges the
// cases' stores into one with a run-time address, and the rows go to scratch
// memory.
template <int NT, int LI, int N, int V, int I0, int J = 0, int SP = 0, int C = 0>
__device__ __forceinline__ void fold(cptr<double> w, const double (&tr)[N][V], const double (&ti)[N][V],
                                     double (&gr)[NT][LI], double (&gi)[NT][LI]) {
    if constexpr (I0 + N <= LI && J < N) {
        const double h = w[(J * 2 + SP) * 4 + C];
        gr[SP][I0 + J] = fma(h, tr[J][C], gr[SP][I0 + J]);
        gi[SP][I0 + J] = fma(h, ti[J][C], gi[SP][I0 + J]);
        constexpr int C1 = C + 1 < V ? C + 1 : 0, S1 = C1 > 0 ? SP : SP + 1 < NT ? SP + 1 : 0;
        fold<NT, LI, N, V, I0, (C1 == 0 && S1 == 0 ? J + 1 : J), S1, C1>(w, tr, ti, gr, gi);
    } else {
        asm volatile("; rows from %0" ::"n"(I0));
    }
}

// One record: all ma with |k - ma| <= lb, the next step's operands requested
// while this one is used (the loop is unrolled by two, so no copies).
template <int NT, int LI, int N, bool SYM>
__device__ __forceinline__ void record(const double2* As, int ss, unsigned x0, unsigned y0, int left, int i0,
                                       cptr<double> c, cptr<double> w, double (&gr)[NT][LI], double (&gi)[NT][LI]) {
    constexpr int V = NT == 1 ? 1 : SYM ? 3 : 4;
    double tr[N][V], ti[N][V];
    Step<NT, N> cur, nxt;
    cur.load(As, ss, x0, y0, c);
    c += N + 1;
    nxt.load(As, ss, cur.nx, cur.ny, c);
    cur.template use<V, true>(tr, ti);
    while (--left > 0) {
        c += N + 1;
        cur.load(As, ss, nxt.nx, nxt.ny, c);
        nxt.template use<V>(tr, ti);
        if (--left == 0) break;
        c += N + 1;
        nxt.load(As, ss, cur.nx, cur.ny, c);
        cur.template use<V>(tr, ti);
    }
    switch (i0) {
        case 0: fold<NT, LI, N, V, 0>(w, tr, ti, gr, gi); break;
        case 1: fold<NT, LI, N, V, 1>(w, tr, ti, gr, gi); break;
        case 2: fold<NT, LI, N, V, 2>(w, tr, ti, gr, gi); break;
        case 3: fold<NT, LI, N, V, 3>(w, tr, ti, gr, gi); break;
        case 4: fold<NT, LI, N, V, 4>(w, tr, ti, gr, gi); break;
        default: fold<NT, LI, N, V, 5>(w, tr, ti, gr, gi); break;
    }
}

// H (or weight) sources of the order-1/2 families of one output row
struct Row12 {
    const DevModel& M;
    const double* hs;      // staged H [rank - lo][lane] (pitch kHPitch), or null
    const double* hrow;    // H of this lane's slot at rank lo
    int n;
    __device__ __forceinline__ double value(int src) const {
        if (src < 0) return as_const(M.weight)[n * M.n_gtinv + (-1 - src)];
        return hs ? hs[src * kHPitch] : hrow[src];
    }
};

// The order-1/2 families of the rows (s, L): their sources, and their part of
// output m = -k: order 2 G_{s,L,-k} += H C_k a_{s',L,+k}, order 1 G_{s,0,0} += H C;
// a0 holds both species' a_{.,L,-k}.  add() returns the energy of families outside
// the polynomial (Euler: 1 / order of Re(G a)).
template <int NT>
struct Sources12 {
    int src[NT + 1], coef[NT + 1];
    double h[NT + 1];
    __device__ __forceinline__ void load(const Row12& R, int t, int s, int L) {
        cptr<int32_t> q = as_const(R.M.q12r) + uniform(((t * 2 + s) * (kMaxLQ12 + 1) + L) * 6);
#pragma unroll
        for (int i = 0; i <= NT; ++i) {
            const int at = i < NT ? 2 * i : 4;
            src[i] = i < NT || L == 0 ? q[at] : kNoSource;
            coef[i] = q[at + 1];
            h[i] = src[i] != kNoSource ? R.value(src[i]) : 0.0;
        }
    }
    __device__ __forceinline__ double add(const Row12& R, int s, int L, int k, const double2 (&a0)[NT], double& gr,
                                          double& gi) const {
        cptr<double> c = as_const(R.M.coef);
        double e = 0.0;
        const double wk = k == 0 ? 0.5 : 1.0, sg = (k & 1) ? -1.0 : 1.0;
#pragma unroll
        for (int sp = 0; sp < NT; ++sp) {
            if (src[sp] == kNoSource) continue;
            const double hc = h[sp] * (sg * c[coef[sp] + k]);
            gr = fma(hc, a0[sp].x, gr);
            gi = fma(-hc, a0[sp].y, gi);
            if (src[sp] < 0) e = fma(wk * hc, a0[sp].x * a0[s].x + a0[sp].y * a0[s].y, e);
        }
        if (src[NT] != kNoSource) {
            const double v = h[NT] * c[coef[NT]];
            gr += v;
            if (src[NT] < 0) e = fma(v, a0[s].x, e);
        }
        return e;
    }
};

template <int NT>
__device__ __forceinline__ double add12(const Row12& R, int t, int s, int L, int k, const double2 (&a0)[NT],
                                        double& gr, double& gi) {
    Sources12<NT> q;
    q.load(R, t, s, L);
    return q.add(R, s, L, k, a0, gr, gi);
}

template <int NT, int LI>
__global__ __launch_bounds__(kQ3Threads) void k_q3(DevModel M, DevSystem S, int stage) {
    extern __shared__ __attribute__((aligned(16))) double2 q3_tile[];
    const int blk = blockIdx.x, n = blockIdx.y;
    const int t = uniform(S.block_type[blk]);
    const int per_s = n_lmh_of(M.lmaxq3) * kBlock;  // entries per species
    const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int hw = M.prange[t][1] - M.prange[t][0];
    const double* hseg = S.H + static_cast<size_t>(blk) * kBlock * M.n_pr + static_cast<size_t>(n) * hw;
    double* hs = reinterpret_cast<double*>(q3_tile + NT * per_s);
    {
        // everything read from HBM before the first task is in flight together: the
        // tile (a thread's entries are kWavesPerWg values of lm apart) and H
        constexpr int kHold = (n_lmh_of(LI == 5 ? 8 : 10) + kWavesPerWg - 1) / kWavesPerWg, kHoldH = 4;
        const int top = per_s / kBlock - 1;
        double2 v[NT][kHold];
        double hv[kHoldH];
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            const double* src = S.A + a_index(M, blk, n, s, 0, 0, lane);
#pragma unroll
            for (int i = 0; i < kHold; ++i) {
                const int lm = min(wave + i * kWavesPerWg, top);
                v[s][i] = double2{src[2 * lm * kBlock], src[(2 * lm + 1) * kBlock]};
            }
        }
        const int hn = stage ? kBlock * hw : 0;
#pragma unroll
        for (int i = 0; i < kHoldH; ++i) {
            const int e = min(static_cast<int>(threadIdx.x) + i * kQ3Threads, hn - 1);
            hv[i] = hn > 0 ? hseg[static_cast<size_t>(e / hw) * M.n_pr + e % hw] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int i = 0; i < kHold; ++i)
                if (wave + i * kWavesPerWg <= top) q3_tile[s * per_s + i * kQ3Threads + threadIdx.x] = v[s][i];
#pragma unroll
        for (int i = 0; i < kHoldH; ++i) {
            const int e = threadIdx.x + i * kQ3Threads;
            if (e < hn) hs[(e % hw) * kHPitch + e / hw] = hv[i];
        }
        for (int e = threadIdx.x + kHoldH * kQ3Threads; e < hn; e += kQ3Threads)
            hs[(e % hw) * kHPitch + e / hw] = hseg[static_cast<size_t>(e / hw) * M.n_pr + e % hw];
    }
    __syncthreads();
    const double2* As = q3_tile + lane;
    cptr<Task3> tasks = as_const(M.t3);
    cptr<Rec3> recs = as_const(M.r3);
    cptr<double> coef = as_const(M.c3);
    cptr<double> wts = as_const(M.w3) + uniform(M.w3_off[t] + n * M.w3_ent[t] * 8);
    const int tb = uniform(M.t3_off[t][wave]), te = uniform(M.t3_off[t][wave + 1]);
    const Row12 rows{M, stage ? hs + lane : nullptr, hseg + static_cast<size_t>(lane) * M.n_pr, n};
    double* const G = S.G + a_index(M, blk, n, 0, 0, 0, lane);
    double eacc = 0.0;
    double gr[NT][LI], gi[NT][LI];
    int pend = 0, k = 0, L0 = 0, nL = 0;
    for (int ti = tb; ti < te; ++ti) {
        const Task3 T = tasks[ti];
        k = uniform(T.k);
        L0 = uniform(T.L0);
        nL = uniform(T.nL);
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int i = 0; i < LI; ++i) gr[s][i] = gi[s][i] = 0.0;
        const int rb = uniform(T.rbeg), re = uniform(T.rend);
        Rec3 nxt{};
        if (rb < re) nxt = recs[rb];
        for (int ri = rb; ri < re; ++ri) {
            const Rec3 cur = nxt;
            if (ri + 1 < re) nxt = recs[ri + 1];
            const int sig = uniform(cur.sig);
            const int i0 = (sig >> 12) & 15, steps = sig >> 16;
            const unsigned x0 = uniform(static_cast<int>(cur.x)), y0 = uniform(static_cast<int>(cur.y));
            cptr<double> c = coef + uniform(cur.coef);
            cptr<double> w = wts + uniform(cur.went) * 8;
            // N, and whether la = lb (one product for the two orders of a
            // species pair)
            switch ((sig >> 8) & 15) {
                case 1: record<NT, LI, 1, false>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 2: record<NT, LI, 2, false>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 3: record<NT, LI, 3, false>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 4: record<NT, LI, 4, false>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 9: record<NT, LI, 1, true>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 10: record<NT, LI, 2, true>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                case 11: record<NT, LI, 3, true>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
                default: record<NT, LI, 4, true>(As, per_s, x0, y0, steps, i0, c, w, gr, gi); break;
            }
        }
        pend = uniform(T.mode);
        // energy of the degree-3 families: (1/3) sum w_k Re(G a), w_0 = 1,
        // else 2; then, where this wave writes the rows, the order-1/2 families
        double e3 = 0.0;
#pragma unroll
        for (int i = 0; i < LI; ++i) {
            if (i >= nL) continue;
            const int L = L0 + 2 * i;
            double2 a[NT];
#pragma unroll
            for (int s = 0; s < NT; ++s) a[s] = As[s * per_s + (L * (L + 1) / 2 + L - k) * kBlock];
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                e3 = fma(gr[s][i], a[s].x, e3);
                e3 = fma(-gi[s][i], a[s].y, e3);
                if (M.split) {  // per-atom energy split: terms weighted by 1 / degree
                    gr[s][i] *= 1.0 / 3.0;
                    gi[s][i] *= 1.0 / 3.0;
                }
                if (pend == 0) {
                    eacc += add12<NT>(rows, t, s, L, k, a, gr[s][i], gi[s][i]);
                    double* g = G + static_cast<size_t>((s * M.n_lmh + L * (L + 1) / 2 + L - k) * 2) * kBlock;
                    g[0] = gr[s][i];
                    g[kBlock] = gi[s][i];
                }
            }
        }
        eacc = fma(k == 0 ? 1.0 / 3.0 : 2.0 / 3.0, e3, eacc);
    }
    // rows above the tile, order-1/2 families only: each L's m = -kk dealt over
    // `share` waves, a_nlm read from HBM an entry ahead
    const int nhi = q3_rows_above(M.lmaxq3, M.maxl), share = q3_row_share(M.lmaxq3, nhi);
    for (int it = wave; it < nhi * share; it += kWavesPerWg) {
        const int L = q3_row_level(it, share, M.lmaxq3);
        const double* src = S.A + a_index(M, blk, n, 0, L * (L + 1) / 2 + L, 0, lane);
        const int sp = M.n_lmh * 2 * kBlock;
        double2 an[NT];
        int kk = q3_row_first(it, share);  // (<= L)
#pragma unroll
        for (int s = 0; s < NT; ++s) an[s] = double2{src[s * sp - 2 * kk * kBlock], src[s * sp - (2 * kk - 1) * kBlock]};
        Sources12<NT> q12[NT];
#pragma unroll
        for (int s = 0; s < NT; ++s) q12[s].load(rows, t, s, L);
        for (; kk <= L; kk += share) {
            double2 a[NT];
            const int kn = min(kk + share, L);
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                a[s] = an[s];
                an[s] = double2{src[s * sp - 2 * kn * kBlock], src[s * sp - (2 * kn - 1) * kBlock]};
            }
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                double hr = 0.0, hi = 0.0;
                eacc += q12[s].add(rows, s, L, kk, a, hr, hi);
                double* g = G + static_cast<size_t>((s * M.n_lmh + L * (L + 1) / 2 + L - kk) * 2) * kBlock;
                g[0] = hr;
                g[kBlock] = hi;
            }
        }
    }
    // parts of divided segments: the last task of a wave
    for (int r = 1; r <= M.q3_rounds; ++r) {
        __syncthreads();
        if (pend != r) continue;
        // all rows read, then all written: one latency, not one per row
        double* g[NT][LI];
        double2 v[NT][LI];
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int i = 0; i < LI; ++i) {
                const int L = L0 + 2 * min(i, nL - 1);
                g[s][i] = G + static_cast<size_t>((s * M.n_lmh + L * (L + 1) / 2 + L - k) * 2) * kBlock;
                v[s][i] = double2{g[s][i][0], g[s][i][kBlock]};
            }
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int i = 0; i < LI; ++i) {
                if (i >= nL) continue;
                g[s][i][0] = v[s][i].x + gr[s][i];
                g[s][i][kBlock] = v[s][i].y + gi[s][i];
            }
    }
    S.Eq34[(((size_t)blk * M.n_fn + n) * kWavesPerWg + wave) * kBlock + lane] = eacc;
}

template <int NT, int LI>
hipError_t launch_k(const DevModel& m, const DevSystem& s, hipStream_t st) {
    size_t lds = sizeof(double2) * NT * n_lmh_of(m.lmaxq3) * kBlock;
    // the block's H segment beside the tile where both fit (l_max 20 with the
    // l = 10 tile does not: H is then read per lane from HBM)
    int hw = 0;
    for (int t = 0; t < NT; ++t) hw = std::max(hw, m.prange[t][1] - m.prange[t][0]);
    const size_t hl = sizeof(double) * hw * kHPitch;
    const int stage = hw > 0 && lds + hl <= lds_limit() ? 1 : 0;
    if (stage) lds += hl;
    if (lds > lds_limit()) return hipErrorInvalidConfiguration;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_q3<NT, LI>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_q3<NT, LI>), dim3(s.nblocks, m.n_fn), dim3(kQ3Threads), lds, st, m, s, stage);
    return launched(lds);
}

// ---------------------------------------------------------------- order 4
// Order-4 linear families (every factor l <= 2 in the table) as polynomials in
// the 9 a_{l<=2,m} of each species: the distinct products of three variables
// (Q4Terms) are formed once and added to every output (S, L) they reach, with
// one coefficient per (radial index, product, output) summed over families and
// factor positions on the host.  Wave `part` of the block's four takes every
// fourth pair (i, j) and its products with k >= j, fully unrolled, all
// variables and the 6 outputs per species in registers; the four partial sums
// meet in LDS.  Bound: FP64 VALU, ~4,900 instructions for two species against
// ~40,000 as one visit per (family, factor position).
template <int NT, int PART>
__device__ __forceinline__ void q4_part(const double (&ar)[NT][6], const double (&ai)[NT][6], cptr<double> c,
                                        double (&gr)[NT][6], double (&gi)[NT][6]) {
    int pair = 0, at = 0;
#pragma unroll
    for (int i = 0; i < 9 * NT; ++i)
#pragma unroll
        for (int j = i; j < 9 * NT; ++j) {
            if (!q4_pair_used(NT, i, j)) continue;
            if (pair++ % kQ4Parts != PART) continue;
            // variables: m <= 0 stored at l (l + 1) / 2 + l - |m|, m > 0 by
            // conjugation and sign
            auto var = [&](int v, double& re, double& im) __attribute__((always_inline)) {
                const int s = v / 9, l = q4_l(v), m = q4_m(v), am = m < 0 ? -m : m, e = l * (l + 1) / 2 + l - am;
                re = (m > 0 && (m & 1)) ? -ar[s][e] : ar[s][e];
                im = m > 0 ? ((m & 1) ? ai[s][e] : -ai[s][e]) : ai[s][e];
            };
            double xr, xi, yr, yi;
            var(i, xr, xi);
            var(j, yr, yi);
            const double qr = fma(xr, yr, -(xi * yi)), qi = fma(xr, yi, xi * yr);
#pragma unroll
            for (int k = j; k < 9 * NT; ++k) {
                if (!q4_used(i, j, k)) continue;
                double zr, zi;
                var(k, zr, zi);
                const double pr = fma(qr, zr, -(qi * zi)), pi = fma(qr, zi, qi * zr);
                const int M = q4_m(i) + q4_m(j) + q4_m(k), par = (q4_l(i) + q4_l(j) + q4_l(k)) & 1;
#pragma unroll
                for (int L = 0; L < 3; ++L) {
                    if (L < M || (L & 1) != par) continue;
#pragma unroll
                    for (int s = 0; s < NT; ++s) {
                        const double h = c[at++];
                        const int e = L * (L + 1) / 2 + L - M;
                        gr[s][e] = fma(h, pr, gr[s][e]);
                        gi[s][e] = fma(h, pi, gi[s][e]);
                    }
                }
            }
            // one pair's products per scheduling region (coefficient loads may
            // cross): all of them at once would not fit the registers
            __builtin_amdgcn_sched_barrier(4);
        }
}

template <int NT>
__global__ __launch_bounds__(64 * kQ4Parts) void k_q4(DevModel M, DevSystem S) {
    __shared__ double2 part[kQ4Parts - 1][NT][6][kBlock];
    const int blk = blockIdx.x, n = blockIdx.y;
    const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int t = uniform(S.block_type[blk]);
    double ar[NT][6], ai[NT][6], gr[NT][6], gi[NT][6];
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int e = 0; e < 6; ++e) {
            // (l_max < 2: the variables above it are zero)
            const bool in = e < M.n_lmh;
            const double* p = S.A + a_index(M, blk, n, s, in ? e : 0, 0, lane);
            ar[s][e] = in ? p[0] : 0.0;
            ai[s][e] = in ? p[kBlock] : 0.0;
            gr[s][e] = gi[s][e] = 0.0;
        }
    cptr<double> c = as_const(M.c4) + uniform((t * M.n_fn + n) * q4_total(NT) + q4_offset(NT, wave));
    switch (wave) {
        case 0: q4_part<NT, 0>(ar, ai, c, gr, gi); break;
        case 1: q4_part<NT, 1>(ar, ai, c, gr, gi); break;
        case 2: q4_part<NT, 2>(ar, ai, c, gr, gi); break;
        default: q4_part<NT, 3>(ar, ai, c, gr, gi); break;
    }
    if (wave > 0)
#pragma unroll
        for (int s = 0; s < NT; ++s)
#pragma unroll
            for (int e = 0; e < 6; ++e) part[wave - 1][s][e][lane] = double2{gr[s][e], gi[s][e]};
    __syncthreads();
    if (wave > 0) return;
    double e4 = 0.0;
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int e = 0; e < 6; ++e) {
            if (e >= M.n_lmh) continue;
            double hr = gr[s][e], hi = gi[s][e];
#pragma unroll
            for (int q = 0; q + 1 < kQ4Parts; ++q) {
                const double2 v = part[q][s][e][lane];
                hr += v.x;
                hi += v.y;
            }
            // degree 4 (Euler): (1/4) w_k Re(G a); e = 0, 2, 5 are m = 0
            e4 = fma(e == 0 || e == 2 || e == 5 ? 0.25 : 0.5, hr * ar[s][e] - hi * ai[s][e], e4);
            const double sc = M.split ? 0.25 : 1.0;
            double* g = S.G + a_index(M, blk, n, s, e, 0, lane);
            g[0] = fma(sc, hr, g[0]);
            g[kBlock] = fma(sc, hi, g[kBlock]);
        }
    S.Eq34[((size_t)blk * M.n_fn + n) * kWavesPerWg * kBlock + lane] += e4;
}

}  // namespace

// L of one parity per segment: up to 5 (l <= 8) or 6 (l <= 10, the table's
// largest order-3 l) rows per species in registers.
hipError_t launch_q3(const DevModel& m, const DevSystem& s, hipStream_t st) {
    if (s.nblocks == 0 || m.lmaxq3 < 0) return hipSuccess;
    hipError_t e;
    if (m.lmaxq3 > 8)
        e = m.n_type == 1 ? launch_k<1, 6>(m, s, st) : launch_k<2, 6>(m, s, st);
    else
        e = m.n_type == 1 ? launch_k<1, 5>(m, s, st) : launch_k<2, 5>(m, s, st);
    if (e != hipSuccess || !m.c4) return e;
    if (m.n_type == 1)
        hipLaunchKernelGGL(k_q4<1>, dim3(s.nblocks, m.n_fn), dim3(64 * kQ4Parts), 0, st, m, s);
    else
        hipLaunchKernelGGL(k_q4<2>, dim3(s.nblocks, m.n_fn), dim3(64 * kQ4Parts), 0, st, m, s);
    return launched();
}

}  // namespace mlip
