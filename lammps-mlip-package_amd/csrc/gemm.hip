// Quadratic form of the polynomial model on the matrix cores (FP64 MFMA).
//
// Per centre species t, for the species' slot rows (blocks are grouped by
// species, and a row holds only the features the species sees):
//   Hq[slot][a] = sum_b D[slot][b] W_t[b][a]
// with W_t the symmetric quadratic form of the species' features
// (reference: the comb2 part of compute_polynomial_model_uniq_products and
// compute_anlm_polynomial_model_correction, pair_mlip_gtinv.cpp:321-343,
// 481-521, and compute_polynomial_adjoints, mlipkk.cpp:668-731).
//
// Workgroup tile 64 rows x 128 columns, K staged through LDS 16 at a time
// (the next stage's global loads in flight while the current one computes);
// four waves of 32 x 64 each, i.e. 2 x 4 blocks of v_mfma_f64_16x16x4f64.
// Lane layout of that instruction (measured on gfx950): A[i][k] from lane
// 16 k + i, B[k][j] from lane 16 k + j, result register r of lane l is
// D[l / 16 + 4 r][l % 16].
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_api.h"
#include "device_common.h"

namespace mlip {

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// Per species: its rows of D, its form (w x w), the output rows, and for the
// fused polynomial step linear weights and energy partials (null: not wanted);
// ld = row pitch.
struct GemmArgs {
    const double* A[2];
    const double* B[2];
    double* C[2];
    const double* lin[2];
    double* epart[2];
    int w[2], mtiles[2];
    int ld, grid0;
};

constexpr int kGM = 64;        // rows per workgroup
constexpr int kGN = 128;       // columns per workgroup
constexpr int kGK = 16;        // K per LDS stage
constexpr int kGThreads = 256;
// LDS row padding (doubles): rows of the K slabs 80 and 144 doubles apart
// (measured 2.48 -> 2.35 ms per evaluation at 256k against a pad of 1)
constexpr int kGPad = 16;
constexpr int kGSmallTiles = 160;  // see gemm_small

// EPI: the polynomial step of a model without cubic terms in the epilogue,
// C = H = lin + A B and epart[row * ldep + nt] = sum over the tile's columns
// of A[row][col] (lin + (A B) / 2) (A holds the features d, K = N), each row's
// partial in a fixed order: four columns per lane, a butterfly over the 16
// lanes of the row, then the two column waves.  Held to 4 waves per SIMD
// (128 registers with the accumulators): unconstrained, the compiler issues
// every epilogue load at once (108 VGPRs), which halves the occupancy of
// the product loop (2.35 -> 2.97 ms at 256k).
template <bool EPI>
__global__ __launch_bounds__(kGThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_gemm_rows(GemmArgs G) {
    // the launch holds both species' tiles, species 1 from workgroup G.grid0
    const int t = static_cast<int>(blockIdx.x) >= G.grid0 ? 1 : 0;
    const double* __restrict__ A = G.A[t];
    const double* __restrict__ B = G.B[t];
    double* __restrict__ C = G.C[t];
    const double* __restrict__ lin = G.lin[t];
    double* __restrict__ epart = G.epart[t];
    const int lda = G.ld, ldc = G.ld, ldep = G.ld, ldb = G.w[t], K = G.w[t], N = G.w[t], mtiles = G.mtiles[t],
              ntiles = (N + kGN - 1) / kGN;
    __shared__ double As[kGK][kGM + kGPad];  // [k][row]
    __shared__ double Bs[kGK][kGN + kGPad];  // [k][column]
    // XCD-aware order: workgroups are dealt round-robin over the 8 XCDs, and
    // consecutive workgroups of one XCD take the column tiles of one row
    // tile, so its A rows are fetched into that XCD's L2 once
    const int g = blockIdx.x - (t ? G.grid0 : 0);
    const int xcd = g & 7, k8 = g >> 3;
    const int mt = xcd + 8 * (k8 / ntiles), nt = k8 % ntiles;
    if (mt >= mtiles) return;
    const int m0 = mt * kGM, n0 = nt * kGN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    // global -> register staging roles
    const int arow = tid >> 2, ak = (tid & 3) * 4;   // A: 64 rows x 16 k, 4 per thread
    // B: 16 k x 128 columns, 8 per thread, 16 apart (a row's 16 lanes store
    // consecutive doubles: no LDS bank conflicts; global reads stay 128-byte runs)
    const int bk = tid >> 4, bc = tid & 15;
    const double* arow_p = A + (size_t)(m0 + arow) * lda;
    double ra[4], rb[8];
    auto load = [&](int kb) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = kb + ak + q;
            ra[q] = k < K ? arow_p[k] : 0.0;
        }
        const int k = kb + bk;
        const double* brow = B + (size_t)k * ldb;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int c = n0 + bc + 16 * q;
            rb[q] = (k < K && c < N) ? brow[c] : 0.0;
        }
    };
    dbl4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    const int nk = (K + kGK - 1) / kGK;
    load(0);
    for (int kt = 0; kt < nk; ++kt) {
        if (kt) __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) As[ak + q][arow] = ra[q];
#pragma unroll
        for (int q = 0; q < 8; ++q) Bs[bk][bc + 16 * q] = rb[q];
        __syncthreads();
        if (kt + 1 < nk) load((kt + 1) * kGK);
#pragma unroll
        for (int kk = 0; kk < kGK / 4; ++kk) {
            const int ka = kk * 4 + (lane >> 4);
            double a[2], b[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = As[ka][wr * 32 + i * 16 + (lane & 15)];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[ka][wc * 64 + j * 16 + (lane & 15)];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    if constexpr (EPI) {
        __shared__ double esum[2][kGM];  // [column wave][row of the tile]
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int rt = wr * 32 + i * 16 + (lane >> 4) + 4 * r;
                const size_t row = static_cast<size_t>(m0 + rt);
                double e = 0.0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int col = n0 + wc * 64 + j * 16 + (lane & 15);
                    if (col < N) {
                        const double la = lin[col], hq = acc[i][j][r];
                        C[row * ldc + col] = la + hq;
                        e = fma(A[row * lda + col], la + 0.5 * hq, e);
                    }
                }
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) e += __shfl_xor(e, o);
                if ((lane & 15) == 0) esum[wc][rt] = e;
            }
        __syncthreads();
        if (epart && tid < kGM) epart[static_cast<size_t>(m0 + tid) * ldep + nt] = esum[0][tid] + esum[1][tid];
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + wc * 64 + j * 16 + (lane & 15);
            if (col >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wr * 32 + i * 16 + (lane >> 4) + 4 * r;
                C[(size_t)row * ldc + col] = acc[i][j][r];
            }
        }
}

// Few rows: workgroup tile 16 x 128, each of eight waves one 16 x 16 block over
// all of K; the 16 rows of A in LDS, B fragments (four 128-byte runs) straight
// from the caches, two rounds of kSAhead steps in flight.  Products, epilogue
// and energy partials are formed in the tiled kernel's order, so a row's
// results do not depend on which of the two ran (nor on the rows beside it).
// Bound: the latency of K / 64 load rounds.  The tiled kernel walks K / 16
// staged rounds on 28 workgroups per species at 864 atoms (K = 492); it is the
// better one once its tiles fill the device (gemm_small).
constexpr int kSM = 16;
constexpr int kSThreads = 512;
constexpr int kSAhead = 16;           // steps of 4 K per load round
constexpr int kSPitch = kSM + 1;

// rows of A in LDS, K padded with zeros to whole rounds
size_t small_lds(int w) {
    return sizeof(double) * kSPitch * (static_cast<size_t>(w + 4 * kSAhead - 1) / (4 * kSAhead) * (4 * kSAhead));
}

template <bool EPI>
__global__ __launch_bounds__(kSThreads) void k_gemm_small(GemmArgs G) {
    extern __shared__ double as[];  // [k][row]
    __shared__ double vs[EPI ? kSM : 1][kGN + 1];
    const int t = static_cast<int>(blockIdx.x) >= G.grid0 ? 1 : 0;
    const int g = blockIdx.x - (t ? G.grid0 : 0);
    const int w = G.w[t], ntiles = (w + kGN - 1) / kGN, ld = G.ld;
    const int mt = g / ntiles, nt = g % ntiles;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int col = nt * kGN + wave * 16 + li;
    const bool cin = col < w;
    const int rounds = (w + 4 * kSAhead - 1) / (4 * kSAhead);
    // columns and K past the form read its last entries: K meets zeros of A,
    // column results are not stored
    const double* b = G.B[t] + (cin ? col : w - 1);
    double bv[kSAhead], bw[kSAhead];
    auto load = [&](int s, double (&v)[kSAhead]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kSAhead; ++q) {
            const int k = 4 * (s * kSAhead + q) + lk;
            v[q] = b[static_cast<size_t>(k < w ? k : w - 1) * w];
        }
    };
    load(0, bv);
    for (int e = threadIdx.x; e < kSM * rounds * 4 * kSAhead; e += kSThreads) {
        const int r = e / (rounds * 4 * kSAhead), k = e % (rounds * 4 * kSAhead);
        as[k * kSPitch + r] = k < w ? G.A[t][static_cast<size_t>(mt * kSM + r) * ld + k] : 0.0;
    }
    __syncthreads();
    dbl4 acc = {0.0, 0.0, 0.0, 0.0};
    auto use = [&](int s, const double (&v)[kSAhead]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kSAhead; ++q)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(as[(4 * (s * kSAhead + q) + lk) * kSPitch + li], v[q], acc, 0,
                                                       0, 0);
    };
    for (int s = 0; s < rounds; s += 2) {
        if (s + 1 < rounds) load(s + 1, bw);
        use(s, bv);
        if (s + 1 >= rounds) break;
        if (s + 2 < rounds) load(s + 2, bv);
        use(s + 1, bw);
    }
    const double la = EPI && cin ? G.lin[t][col] : 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = lk + 4 * r;
        if (cin) G.C[t][static_cast<size_t>(mt * kSM + row) * ld + col] = EPI ? la + acc[r] : acc[r];
        if constexpr (EPI) vs[row][wave * 16 + li] = la + 0.5 * acc[r];
    }
    if constexpr (EPI) {
        // thread (row, column half, lane of 16): the tiled kernel's order
        __syncthreads();
        const int row = threadIdx.x >> 5, wc = (threadIdx.x >> 4) & 1, l = threadIdx.x & 15;
        double e = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = wc * 64 + j * 16 + l;
            if (nt * kGN + c < w) e = fma(G.A[t][static_cast<size_t>(mt * kSM + row) * ld + nt * kGN + c], vs[row][c], e);
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) e += __shfl_xor(e, o);
        const double other = __shfl_xor(e, 16);
        if (G.epart[t] && (threadIdx.x & 31) == 0) G.epart[t][static_cast<size_t>(mt * kSM + row) * ld + nt] = e + other;
    }
}

// Ep[slot] = the slot's partial energies of the fused epilogue, in column
// tile order (no tile for a species without polynomial features: 0)
__global__ __launch_bounds__(256) void k_ep_sum(DevModel M, DevSystem S) {
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= S.nblocks * kBlock) return;
    const int t = S.block_type[slot / kBlock];
    const int nt = (M.wdim[t] + kGN - 1) / kGN;
    const double* ep = S.Hq + static_cast<size_t>(slot) * M.n_pr;
    double e = 0.0;
    for (int k = 0; k < nt; ++k) e += ep[k];
    S.Ep[slot] = e;
}

}  // namespace

namespace {
// The small-tile kernel while the 64 x 128 tiles of both species leave more than
// a third of the compute units idle (order-4 model, both species in one launch,
// tiled / small: 864 atoms 69 / 26 us, 2,048 atoms = 128 tiles 73 / 48 us, 4,000
// atoms = 252 tiles 75 / 91 us; two launches of the tiled kernel took 110 us at
// 864 and 120 us at 4,000 atoms).
bool gemm_small(const DevModel& m, const DevSystem& s) {
    const int w = m.n_type > 1 && m.wdim[1] > m.wdim[0] ? m.wdim[1] : m.wdim[0];
    // (its A rows must fit the LDS beside the energy tile)
    if (small_lds(w) + sizeof(double) * kSM * (kGN + 1) > lds_limit()) return false;
    return static_cast<int64_t>(s.nblocks) * ((w + kGN - 1) / kGN) <= kGSmallTiles;
}
}  // namespace

hipError_t launch_poly_gemm(const DevModel& m, const DevSystem& s, const int* nblk_type, hipStream_t st) {
    GemmArgs g{};
    g.ld = m.n_pr;
    const bool small = gemm_small(m, s);
    size_t lds = 0;
    int b0 = 0, grid[2] = {0, 0};
    for (int t = 0; t < m.n_type && t < 2; ++t) {
        const int nb = nblk_type[t], w = m.wdim[t];
        const size_t r0 = static_cast<size_t>(b0) * kBlock * m.n_pr;
        b0 += nb;
        if (nb == 0 || w == 0) continue;
        g.A[t] = s.D + r0;
        g.B[t] = m.wmat + m.wofs[t];
        g.C[t] = (m.poly_fused ? s.H : s.Hq) + r0;
        g.lin[t] = m.lin_p + static_cast<size_t>(t) * m.n_pr;
        g.epart[t] = s.Hq ? s.Hq + r0 : nullptr;
        g.w[t] = w;
        if (small) {
            lds = std::max(lds, small_lds(w));
            g.mtiles[t] = nb * kBlock / kSM;
            grid[t] = g.mtiles[t] * ((w + kGN - 1) / kGN);
        } else {
            g.mtiles[t] = nb * kBlock / kGM;
            grid[t] = 8 * ((w + kGN - 1) / kGN) * ((g.mtiles[t] + 7) / 8);
        }
    }
    if (b0 != s.nblocks) return hipErrorInvalidValue;
    g.grid0 = grid[0];
    if (grid[0] + grid[1] == 0) return hipSuccess;
    const dim3 gr(grid[0] + grid[1]), blk(small ? kSThreads : kGThreads);
    if (small) {
        const void* f = m.poly_fused ? reinterpret_cast<const void*>(k_gemm_small<true>)
                                     : reinterpret_cast<const void*>(k_gemm_small<false>);
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
    }
    if (small && m.poly_fused)
        hipLaunchKernelGGL(k_gemm_small<true>, gr, blk, lds, st, g);
    else if (small)
        hipLaunchKernelGGL(k_gemm_small<false>, gr, blk, lds, st, g);
    else if (m.poly_fused)
        hipLaunchKernelGGL(k_gemm_rows<true>, gr, blk, 0, st, g);
    else
        hipLaunchKernelGGL(k_gemm_rows<false>, gr, blk, 0, st, g);
    return launched();
}

hipError_t launch_poly_sum(const DevModel& m, const DevSystem& s, hipStream_t st) {
    const int nslot = s.nblocks * kBlock;
    if (nslot == 0) return hipSuccess;
    hipLaunchKernelGGL(k_ep_sum, dim3((nslot + 255) / 256), dim3(256), 0, st, m, s);
    return launched();
}

}  // namespace mlip
