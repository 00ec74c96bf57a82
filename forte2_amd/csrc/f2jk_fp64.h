// FP64 exchange kernels (gfx950): the half-transform X = B C and the
// contraction K = sum_P X_P X_P^T on v_mfma_f64_16x16x4.
//
// One FP64 MFMA keeps a SIMD's matrix pipe busy for 64 cycles, so both are
// bound by how evenly the 16 x 16 output blocks are spread over the SIMDs as
// long as loads run a step ahead; LDS and L2 have room to spare.
//
// * The half-transform gives every wave whole rows (16 * IB of them) and all
//   the occupied columns of the tile (NB blocks of 16, exactly the job's
//   width): no wave holds padding columns, and A = B(P|mn) goes from global
//   memory straight into MFMA operands, each element loaded once by one lane.
//   Rates (random B): 65 TFLOP/s at nbf 1152 with 240 and 320 columns, where
//   the same kernel without its loads of B reaches 67-68 (the clock under FP64
//   MFMA load, not the 78.6 TFLOP/s of 2.4 GHz, is the ceiling) and the 128 x
//   320 tiles before it reached 46 (240 of 320 columns in use); 56 at nbf 384
//   with 80 columns (42 before: 80 of 128).  Below about 50 columns it is
//   bound by reading B: 4.2 TB/s of B and X at nbf 318.
// * The contraction splits the valid 16 x 16 blocks of a 128 x 128 tile over
//   its four waves (a diagonal tile's 36 lower blocks as 9 per wave, an edge
//   tile's rows in halves), and splits the P range of each kind of tile in
//   proportion to its cost, so the workgroups of a launch take about as long.
//   62 TFLOP/s of the lower triangle at nbf 1152 and 1536 (55 and 56 for the
//   uniform splits of whole tiles before it), 53 at nbf 384 (43), where 60 is
//   reached without any loads.
//
// Operand order.  A k step of 8 feeds two MFMAs: lane group g = lane / 16
// holds k = 2g and 2g + 1 and supplies the first to MFMA 0 and the second to
// MFMA 1.  The k sum is the same set of products in another order, and every
// lane's operands are 16 contiguous bytes, in global memory and in LDS.
//
// Tiles reach LDS by direct-to-LDS loads (lane l to slot l of 16 bytes) in the
// order in which the fragments are read: every LDS read is 1 KB of consecutive
// bytes.  A load into LDS is not ordered with register loads, so a step ends
// with a full drain before its barrier; the loads have had the whole step.
#pragma once
#include "f2jk_kernels.h"
#include "f2jk_tiles.h"

namespace f2jk {

typedef double dx2 __attribute__((ext_vector_type(2)));
// rows of B start at a multiple of 8 bytes only when nbf is odd
typedef double dx2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kDK = 16;         // k extent of one LDS stage
constexpr int kDMaxNB = 20;     // 16-column blocks of the widest tile
constexpr int kDMaxDens = 8;
constexpr int kDKsLds = 2 * 2 * 16 * 1024;                // two stages of 8 + 8 row blocks, 2 KB each
constexpr int kDKxLds(int nb) { return 2 * nb * 2048; }   // two stages of nb column blocks, 2 KB each

// 16-row blocks per wave.  More than one block shares a coefficient fragment
// among more MFMAs, fewer leave registers for more waves per SIMD, which covers
// the load latency better.  Measured (B 2.6 GB, nbf 384, 80 columns): 926, 933
// and 938 us with 3, 2 and 1; at nbf 1184 4045, 3733 and 3895 us; at nbf 318
// with 64 columns 226, 196 and 191 us with 4, 2 and 1, with 32 columns 170, 164
// and 162 us.  From 9 blocks on one row block already has enough MFMAs per step.
constexpr int kxd_ib(int nb) { return nb >= 5 && nb <= 8 ? 2 : 1; }

// a pointer that is the same in every lane, held in scalar registers
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* p) {
    const uint64_t u = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return (const T*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// columns of the densities side by side: density d is [ioff, ioff + width)
struct DCols {
    int nd;
    int nocc[kDMaxDens], width[kDMaxDens], ioff[kDMaxDens];
    __device__ __forceinline__ int count() const { return nd; }
    __device__ __forceinline__ int first(int d) const { return ioff[d]; }
    __device__ __forceinline__ int end(int d) const { return ioff[d] + width[d]; }
};
// the same of one or two densities, in registers
struct DCols2 {
    int nd, ioff0, end0, ioff1, end1;
    __device__ __forceinline__ int count() const { return nd; }
    __device__ __forceinline__ int first(int d) const { return d ? ioff1 : ioff0; }
    __device__ __forceinline__ int end(int d) const { return d ? end1 : end0; }
};

// ---------------------------------------------------------------------------
// Coefficients of all densities in the two forms the kernels read:
//   Cp[n][c]  row-major, the columns of all tiles (the gamma sums of the
//             half-transform; null without them);
//   Cq        [column tile][16-k step][block][k / 8 % 2][lane][2], the order
//             of the half-transform's LDS tiles; zero outside N x nocc.
// ---------------------------------------------------------------------------
struct DCoef {
    const double* C[kDMaxDens];
    int64_t ldc[kDMaxDens];
};
__device__ __forceinline__ void pack_cq_element(const double* const* C, const int64_t* ldc, int nd,
                                                const int* nocc, const int* ioff, int N, int ldcp, int nb, int nks,
                                                int64_t t, double* __restrict__ Cp, double* __restrict__ Cq) {
    const int tt = (int)(t & 1), lane = (int)((t >> 1) & 63);
    const int64_t u = t >> 7;                       // (ct * nks + s) * 2 nb + 2 j + h
    const int jh = (int)(u % (2 * nb));
    const int64_t v = u / (2 * nb);
    const int s = (int)(v % nks), ct = (int)(v / nks);
    const int k = kDK * s + 8 * (jh & 1) + 2 * (lane >> 4) + tt;
    const int c = (ct * nb + (jh >> 1)) * 16 + (lane & 15);
    double x = 0.0;
    for (int d = 0; d < nd; ++d) {
        const int i = c - ioff[d];
        if (i >= 0 && i < nocc[d] && k < N) x = C[d][(int64_t)k * ldc[d] + i];
    }
    Cq[t] = x;
    if (Cp && k < N) Cp[(int64_t)k * ldcp + c] = x;
}
__global__ void pack_cq_kernel(DCoef cs, DCols dc, int N, int ldcp, int nb, int nks, int64_t total,
                               double* __restrict__ Cp, double* __restrict__ Cq) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < total) pack_cq_element(cs.C, cs.ldc, dc.nd, dc.nocc, dc.ioff, N, ldcp, nb, nks, t, Cp, Cq);
}

// ---------------------------------------------------------------------------
// Half-transform: X[r][c] = sum_k A[r][k] C[k][c], r < R, for a tile of
// NB * 16 columns; 4 waves of 16 * IB rows each.
// With grow, the epilogue also forms the row sums
//   grow[ct * nd + d][r] = sum over the columns c of density d in the tile of X[r][c] C[r % N][c]
// whose sum over the N rows of one P is gamma_P = sum_mn B_Pmn D_mn (D = C C^T):
// the first J pass without another read of B and without D.  A row's sum does
// not depend on how rows are cut into tiles or P into chunks.
// ---------------------------------------------------------------------------
template <int NB, int IB, typename Cols>
__device__ __forceinline__ void kxd_body(char* lds, const double* __restrict__ A, int64_t R, int K,
                                         const double* __restrict__ Cq, int nks, double* __restrict__ X,
                                         int64_t ldx, int ncol, int ncolt, const double* __restrict__ Cp,
                                         const Cols& dc, double* __restrict__ grow, int64_t gstride, int b,
                                         int nblocks) {
    constexpr int STAGE = NB * 2048;  // bytes
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = xcd_remap(b, nblocks);
    const int ct = t % ncolt;
    const int64_t r0 = (int64_t)(t / ncolt) * (64 * IB);  // first row of the workgroup
    const int wr0 = wid * 16 * IB;
    const int lr = lane & 15, lg = lane >> 4;

    // rows past R are clamped onto the last row and never stored
    const double* At = A + r0 * K;
    uint32_t aoff[IB];
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        const int64_t row = r0 + wr0 + i * 16 + lr;
        aoff[i] = (uint32_t)((row < R ? row : R - 1) - r0) * (uint32_t)K + 2 * lg;
    }
    dx2 an[IB][2];
    auto load_a = [&](int s) {
        if ((s + 1) * kDK <= K) {
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    an[i][h] = *reinterpret_cast<const dx2u*>(At + (aoff[i] + (uint32_t)(s * kDK + 8 * h)));
        } else {  // the last step of a K that is not a multiple of 16: zeros past K
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k = s * kDK + 8 * h + 2 * lg;
                    const double* p = At + (aoff[i] + (uint32_t)(s * kDK + 8 * h));
                    an[i][h].x = k < K ? p[0] : 0.0;
                    an[i][h].y = k + 1 < K ? p[1] : 0.0;
                }
        }
    };
    const double* Ct = uniform_ptr(Cq + (int64_t)ct * nks * (NB * 256));
    auto load_c = [&](int s, int stg) {
        const double* base = Ct + (int64_t)s * (NB * 256);
        const uint32_t l0 = lds_addr(lds) + stg * STAGE;
        static_for<0, (2 * NB + 3) / 4>([&](auto Q) {
            const int q = wid + 4 * decltype(Q)::value;  // wave-uniform
            if (q < 2 * NB) lds_load16(base + q * 128, (uint32_t)lane * 16, l0 + q * 1024);
        });
    };

    dx4 acc[IB][NB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = dx4{0, 0, 0, 0};

    load_c(0, 0);
    load_a(0);
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(an[i][h]));
    drain_and_barrier();
    for (int s = 0; s < nks; ++s) {
        const int cur = s & 1;
        dx2 a[IB][2];
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) a[i][h] = an[i][h];
        if (s + 1 < nks) {
            load_c(s + 1, cur ^ 1);  // that stage was last read before the previous barrier
            load_a(s + 1);
        }
        // one column block of half a step at a time: the fragment three blocks
        // ahead is read, then the block's MFMAs; nothing moves across groups or
        // past the drain
        const char* st = lds + cur * STAGE + lane * 16;
        constexpr int NG = 2 * NB, AHEAD = NG > 3 ? 3 : NG - 1;
        dx2 c[4];
        auto frag = [&](auto G) {  // group G: half G / NB, block G % NB
            constexpr int g = decltype(G)::value;
            c[g & 3] = *reinterpret_cast<const dx2*>(st + (2 * (g % NB) + g / NB) * 1024);
        };
        static_for<0, AHEAD>(frag);
        static_for<0, NG>([&](auto G) {
            constexpr int g = decltype(G)::value, h = g / NB, j = g % NB;
            if constexpr (g + AHEAD < NG) frag(std::integral_constant<int, g + AHEAD>{});
#pragma unroll
            for (int i = 0; i < IB; ++i) acc[i][j] = mfma4(a[i][h].x, c[g & 3].x, acc[i][j]);
#pragma unroll
            for (int i = 0; i < IB; ++i) acc[i][j] = mfma4(a[i][h].y, c[g & 3].y, acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        });
        drain_and_barrier();
    }
    const int c0 = ct * NB * 16 + lr;
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = r0 + wr0 + i * 16 + acc_row<double>(lane, r);
            if (row < R) {
                double* dst = X + row * ldx + c0;
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    if (c0 + j * 16 < ncol) dst[j * 16] = acc[i][j][r];
            }
        }
    if (!grow) return;
    const int ldcp = ncolt * NB * 16, nd = dc.count();
    auto row_sums = [&](int d, auto masked) {
        const int lo = dc.first(d), hi = dc.end(d);
        double* gr = grow + (int64_t)(ct * nd + d) * gstride;
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = r0 + wr0 + i * 16 + acc_row<double>(lane, r);
                const double* cr = Cp + (int64_t)((uint32_t)(row < R ? row : R - 1) % (uint32_t)K) * ldcp + c0;
                double s = 0.0;
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const double x = cr[j * 16];
                    if constexpr (decltype(masked)::value) {
                        // the lanes of the density alone: its neighbour's sums may be
                        // infinite, and zero times them is not zero.  Kept a branch: as
                        // selects the copies of a whole row took up to 60 registers more
                        if ((uint32_t)(c0 + j * 16 - lo) < (uint32_t)(hi - lo)) {
                            s = fma(acc[i][j][r], x, s);
                            asm volatile("" : "+v"(s));
                        }
                    } else
                        s = fma(acc[i][j][r], x, s);
                }
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o);
                if (lr == 0 && row < R) gr[row] = s;
                __builtin_amdgcn_sched_barrier(0);  // one row's coefficients in registers at a time
            }
    };
    if (nd == 1)
        row_sums(0, std::false_type{});
    else
        for (int d = 0; d < nd; ++d) row_sums(d, std::true_type{});
}

template <int NB, int IB>
__global__ __launch_bounds__(256, 2) void kxd_kernel(const double* __restrict__ A, int64_t R, int K,
                                                     const double* __restrict__ Cq, int nks, double* __restrict__ X,
                                                     int64_t ldx, int ncol, int ncolt, const double* __restrict__ Cp,
                                                     DCols dc, double* __restrict__ grow, int64_t gstride) {
    __shared__ __attribute__((aligned(16))) char lds[kDKxLds(NB)];
    kxd_body<NB, IB>(lds, A, R, K, Cq, nks, X, ldx, ncol, ncolt, Cp, dc, grow, gstride,
                     blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// Transform of the row index: Y[P][i][n] = sum_k C[k][i] M[P][k][n], i < ni,
// n < ncol, for matrices M[P] of K rows with row stride ld: the half-transform
// with the operands exchanged (the coefficients of the same LDS tiles as A,
// M's rows as B, 16 consecutive n of a row per lane group), so the sum runs
// over M's rows and Y comes out with n contiguous, ready to be the A of
// kxd_kernel.  A wave holds IB blocks of 16 n for all NB * 16 rows i of the
// tile.
// ---------------------------------------------------------------------------
template <int NB, int IB>
__global__ __launch_bounds__(256, 2) void kxt_kernel(const double* __restrict__ M, int64_t pstride, int ld, int K,
                                                     int ncol, int64_t nblocks, const double* __restrict__ Cq, int nks,
                                                     double* __restrict__ Y, int ni, int ncolt) {
    __shared__ __attribute__((aligned(16))) char lds[kDKxLds(NB)];
    constexpr int STAGE = NB * 2048;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = t % ncolt;
    const int64_t q0 = ((int64_t)(t / ncolt) * 4 + wid) * IB;  // first block of the wave
    const int nblk = (ncol + 15) / 16;                         // blocks per P
    const int lr = lane & 15, lg = lane >> 4;

    const double* mp[IB];
    int64_t P[IB];
    int n[IB];
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        const int64_t q = q0 + i < nblocks ? q0 + i : nblocks - 1;  // past the end: computed, never stored
        P[i] = q / nblk;
        n[i] = (int)(q - P[i] * nblk) * 16 + lr;
        mp[i] = M + P[i] * pstride + (int64_t)(2 * lg) * ld + (n[i] < ncol ? n[i] : ncol - 1);
    }
    dx2 an[IB][2];
    auto load_m = [&](int s) {
        if ((s + 1) * kDK <= K) {
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const double* p = mp[i] + (int64_t)(s * kDK + 8 * h) * ld;
                    an[i][h].x = p[0];
                    an[i][h].y = p[ld];
                }
        } else {  // the last step of a K that is not a multiple of 16: zeros past K
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k = s * kDK + 8 * h + 2 * lg;
                    const double* p = mp[i] + (int64_t)(s * kDK + 8 * h) * ld;
                    an[i][h].x = k < K ? p[0] : 0.0;
                    an[i][h].y = k + 1 < K ? p[ld] : 0.0;
                }
        }
    };
    const double* Ct = uniform_ptr(Cq + (int64_t)ct * nks * (NB * 256));
    auto load_c = [&](int s, int stg) {
        const double* base = Ct + (int64_t)s * (NB * 256);
        const uint32_t l0 = lds_addr(lds) + stg * STAGE;
        static_for<0, (2 * NB + 3) / 4>([&](auto Q) {
            const int q = wid + 4 * decltype(Q)::value;
            if (q < 2 * NB) lds_load16(base + q * 128, (uint32_t)lane * 16, l0 + q * 1024);
        });
    };
    dx4 acc[IB][NB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = dx4{0, 0, 0, 0};
    load_c(0, 0);
    load_m(0);
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(an[i][h]));
    drain_and_barrier();
    for (int s = 0; s < nks; ++s) {
        const int cur = s & 1;
        dx2 a[IB][2];
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) a[i][h] = an[i][h];
        if (s + 1 < nks) {
            load_c(s + 1, cur ^ 1);
            load_m(s + 1);
        }
        const char* st = lds + cur * STAGE + lane * 16;
        constexpr int NG = 2 * NB, AHEAD = NG > 3 ? 3 : NG - 1;
        dx2 c[4];
        auto frag = [&](auto G) {
            constexpr int g = decltype(G)::value;
            c[g & 3] = *reinterpret_cast<const dx2*>(st + (2 * (g % NB) + g / NB) * 1024);
        };
        static_for<0, AHEAD>(frag);
        static_for<0, NG>([&](auto G) {
            constexpr int g = decltype(G)::value, h = g / NB, j = g % NB;
            if constexpr (g + AHEAD < NG) frag(std::integral_constant<int, g + AHEAD>{});
#pragma unroll
            for (int i = 0; i < IB; ++i) acc[i][j] = mfma4(c[g & 3].x, a[i][h].x, acc[i][j]);
#pragma unroll
            for (int i = 0; i < IB; ++i) acc[i][j] = mfma4(c[g & 3].y, a[i][h].y, acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        });
        drain_and_barrier();
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        if (q0 + i >= nblocks || n[i] >= ncol) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = (ct * NB + j) * 16 + acc_row<double>(lane, r);
                if (row < ni) Y[(P[i] * ni + row) * ncol + n[i]] = acc[i][j][r];
            }
    }
}

// gamma[d][P] = sum over column tiles and rows m of grow[ct * nd + d][P * N + m], one wave per (d, P)
__device__ __forceinline__ void gamma_rows_body(const double* __restrict__ grow, int64_t gstride, int nd, int ncolt,
                                                int N, double* __restrict__ gamma, int Q, int d, int P) {
    const int lane = threadIdx.x & 63;
    double s = 0.0;
    for (int ct = 0; ct < ncolt; ++ct) {
        const double* g = grow + (int64_t)(ct * nd + d) * gstride + (int64_t)P * N;
        for (int m = lane; m < N; m += 64) s += g[m];
    }
    s = wave_sum(s);
    if (lane == 0) gamma[(int64_t)d * Q + P] = s;
}
__global__ __launch_bounds__(256) void gamma_rows_kernel(const double* __restrict__ grow, int64_t gstride, int nd,
                                                         int ncolt, int N, int pc, double* __restrict__ gamma, int Q) {
    const int P = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (P < pc) gamma_rows_body(grow, gstride, nd, ncolt, N, gamma, Q, blockIdx.y, P);
}

// ---------------------------------------------------------------------------
// Contraction.  The lower triangle of K is cut into 128 x 128 tiles (DTiles).
// Tiles of kind k split the P range in ns[k] parts.  Workgroups are numbered by
// the position of their P range, so that those which read the same X run
// together.
// ---------------------------------------------------------------------------
static_assert(kDTileEdge == kTile, "one tile edge");
__host__ __device__ inline int dtile_kind(const DTiles& m, int mt, int nt) {
    return (mt == m.nt - 1 ? 2 : 0) + (mt == nt ? 1 : 0);
}
__host__ __device__ inline int dtile_cum(const DTiles& m, int g) {
    int c = 0;
    for (int k = 0; k < 4; ++k) c += m.cnt[k] * (int)((int64_t)m.ns[k] * g / m.G);
    return c;
}
// workgroup b -> tile (mt, nt), split s of ns
__host__ __device__ inline void dtile_decode(const DTiles& m, int b, int& mt, int& nt, int& s, int& ns) {
    int g = (int)((int64_t)b * m.G / m.total);
    while (dtile_cum(m, g + 1) <= b) ++g;
    while (dtile_cum(m, g) > b) --g;
    int x = b - dtile_cum(m, g);
    for (int k = 0; k < 4; ++k) {
        const int s0 = (int)((int64_t)m.ns[k] * g / m.G), s1 = (int)((int64_t)m.ns[k] * (g + 1) / m.G);
        const int n = m.cnt[k] * (s1 - s0);
        if (x >= n) {
            x -= n;
            continue;
        }
        const int q = x % m.cnt[k];
        s = s0 + x / m.cnt[k];
        ns = m.ns[k];
        if (k == 0) {
            mt = 1;
            while (mt * (mt + 1) / 2 <= q) ++mt;
            nt = q - mt * (mt - 1) / 2;
        } else if (k == 1) {
            mt = nt = q;
        } else {
            mt = m.nt - 1;
            nt = k == 2 ? q : mt;
        }
        return;
    }
}

__device__ __forceinline__ void ksd_body(char* lds, const double* __restrict__ X, int N, int OPAD, int ioff,
                                         int width, int Pc, const DTiles& tm, double* __restrict__ Kpart,
                                         int accumulate, int b) {
    constexpr int STAGE = 32 * 1024;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    int mt = 0, nt = 0, s = 0, ns = 1;
    dtile_decode(tm, xcd_remap(b, tm.total), mt, nt, s, ns);
    const bool diag = mt == nt;
    const int rbn = mt == tm.nt - 1 ? tm.rl : 8;
    const int m0 = mt * kTile, n0 = nt * kTile;
    const int Pa = (int)((int64_t)Pc * s / ns), Pb = (int)((int64_t)Pc * (s + 1) / ns);
    const int lr = lane & 15, lg = lane >> 4;

    // this wave's loads: row block (wid + 4 q) / 2 (0-7 of the tile's rows,
    // 8-15 of its columns), half (wid + 4 q) % 2 of the 16-k step
    int qrow[8];
    bool qon[8];
    uint32_t qoff[8];
    static_for<0, 8>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        const int rb = (wid + 4 * q) >> 1;
        const int row = (rb < 8 ? m0 : n0 - 128) + rb * 16;
        qon[q] = rb < 8 ? rb < rbn : !diag;
        qrow[q] = qon[q] ? row : 0;
        // rows past N are clamped onto row N - 1: they feed outputs that are never read
        const int lrow = qrow[q] + lr < N ? lr : N - 1 - qrow[q];
        qoff[q] = (uint32_t)(lrow * OPAD + 2 * lg) * 8;
    });
    // The k range runs in halves of 8 through the P of the split, one after the
    // other, and a step is any two of them: with steps that ended with their P,
    // an odd number of halves cost a half-empty step per P (nbf 318, two
    // densities of 3 halves: 109 us for both, the matrix pipes 44% busy).
    const int hp = width >> 3, nh = (Pb - Pa) * hp, nsteps = (nh + 1) >> 1;
    int Pn = Pa, kn = wid & 1, ln = wid & 1;  // the half this wave loads next: its P, place in P, number
    while (kn >= hp) kn -= hp, ++Pn;
    auto load = [&](int stg) {
        if (ln < nh) {
            const double* XP = X + (int64_t)Pn * N * OPAD + ioff + 8 * kn;
            const uint32_t l0 = lds_addr(lds) + stg * STAGE;
            static_for<0, 8>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                if (qon[q]) lds_load16(uniform_ptr(XP + (int64_t)qrow[q] * OPAD), qoff[q], l0 + (wid + 4 * q) * 1024);
            });
        }
        ln += 2;
        kn += 2;
        while (kn >= hp) kn -= hp, ++Pn;
    };
    // the steps of the P range, one after the other: compute(LDS of the step at
    // this lane's slot, halves of the step)
    auto sweep = [&](auto&& compute) {
        load(0);
        drain_and_barrier();
        for (int st = 0; st < nsteps; ++st) {
            const int cur = st & 1;
            if (st + 1 < nsteps) load(cur ^ 1);
            compute(lds + cur * STAGE + lane * 16, min(2, nh - 2 * st));
            __builtin_amdgcn_sched_barrier(0);  // no MFMA moves past the drain
            drain_and_barrier();
        }
    };
    auto frag = [&](const char* L, int rb, int h) {
        return *reinterpret_cast<const dx2*>(L + (2 * rb + h) * 1024);
    };
    double* Ks = Kpart + (int64_t)s * N * N;
    auto put = [&](const dx4& v, int rb, int cb) {
        const int col = n0 + cb * 16 + lr;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m0 + rb * 16 + acc_row<double>(lane, r);
            if (row < N && col < N) {
                double* dst = Ks + (int64_t)row * N + col;
                *dst = accumulate ? *dst + v[r] : v[r];
            }
        }
    };
    // NI x 4 blocks from row block i0 and column block j0
    auto rect = [&](auto NI_, int i0, int j0) {
        constexpr int NI = decltype(NI_)::value;
        dx4 acc[NI > 0 ? NI : 1][4];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = dx4{0, 0, 0, 0};
        sweep([&](const char* L, int halves) {
            for (int h = 0; h < halves; ++h) {
                dx2 a[NI > 0 ? NI : 1], c[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = frag(L, 8 + j0 + j, h);
#pragma unroll
                for (int i = 0; i < NI; ++i) a[i] = frag(L, i0 + i, h);
#pragma unroll
                for (int i = 0; i < NI; ++i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = mfma4(a[i].x, c[j].x, acc[i][j]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = mfma4(a[i].y, c[j].y, acc[i][j]);
                }
            }
        });
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) put(acc[i][j], i0 + i, j0 + j);
    };
    if (diag) {
        // the lower blocks, numbered row after row, in quarters
        const int nq = rbn * (rbn + 1) / 2;
        const int qa = nq * wid / 4, qn = nq * (wid + 1) / 4 - qa;
        int bi[9], bj[9];
        {
            int i = 0, q = qa;
            while (q > i) q -= ++i;
            static_for<0, 9>([&](auto T) {
                constexpr int t = decltype(T)::value;
                bi[t] = i < 8 ? i : 0;
                bj[t] = i < 8 ? q : 0;
                if (++q > i) q = 0, ++i;
            });
        }
        dx4 acc[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) acc[i] = dx4{0, 0, 0, 0};
        sweep([&](const char* L, int halves) {
            for (int h = 0; h < halves; ++h) {
                static_for<0, 3>([&](auto U) {  // three blocks at a time: consecutive MFMAs on different ones
                    constexpr int u = 3 * decltype(U)::value;
                    dx2 a[3], c[3];
                    static_for<0, 3>([&](auto T) {
                        a[T] = frag(L, bi[u + T], h);
                        c[T] = frag(L, bj[u + T], h);
                    });
                    static_for<0, 3>([&](auto T) {
                        if (u + T < qn) acc[u + T] = mfma4(a[T].x, c[T].x, acc[u + T]);
                    });
                    static_for<0, 3>([&](auto T) {
                        if (u + T < qn) acc[u + T] = mfma4(a[T].y, c[T].y, acc[u + T]);
                    });
                });
            }
        });
        static_for<0, 9>([&](auto T) {
            if (T < qn) put(acc[T], bi[T], bj[T]);
        });
    } else {
        // the rows in halves and the columns in halves, one quarter per wave
        const int nr0 = (rbn + 1) / 2;
        const int i0 = wid >> 1 ? nr0 : 0, ni = wid >> 1 ? rbn - nr0 : nr0, j0 = (wid & 1) * 4;
        switch (ni) {
            case 4: rect(std::integral_constant<int, 4>{}, i0, j0); break;
            case 3: rect(std::integral_constant<int, 3>{}, i0, j0); break;
            case 2: rect(std::integral_constant<int, 2>{}, i0, j0); break;
            case 1: rect(std::integral_constant<int, 1>{}, i0, j0); break;
            default: rect(std::integral_constant<int, 0>{}, i0, j0); break;
        }
    }
}
// all densities in one launch (the partials of one are dstride doubles)
__global__ __launch_bounds__(256, 2) void ksd_kernel(const double* __restrict__ X, int N, int OPAD, DCols dc, int Pc,
                                                     DTiles tm, double* __restrict__ Kpart, int64_t dstride,
                                                     int accumulate) {
    __shared__ __attribute__((aligned(16))) char lds[kDKsLds];
    const int d = blockIdx.x / tm.total;
    ksd_body(lds, X, N, OPAD, dc.ioff[d], dc.width[d], Pc, tm, Kpart + d * dstride, accumulate, blockIdx.x % tm.total);
}

// the reduction over the splits of the element's tile
__device__ __forceinline__ int dtile_splits(const DTiles& m, int m4, int n16) {
    return m.ns[dtile_kind(m, m4 * 4 / kTile, n16 * 16 / kTile)];
}
__global__ __launch_bounds__(256) void kred_kernel(const double* __restrict__ Kpart, int64_t dstride, DTiles tm,
                                                   int N, KPtrs K) {
    const int m4 = blockIdx.y, n16 = blockIdx.x;
    if (n16 * 16 > m4 * 4 + 3) return;
    k_reduce_body(Kpart + blockIdx.z * dstride, dtile_splits(tm, m4, n16), N, K.p[blockIdx.z], m4, n16);
}

// both reductions of a small build in one launch: nbj blocks of J, the rest K
template <int VEC, int ND>
__global__ __launch_bounds__(256) void jkred_kernel(const double* __restrict__ jpart, int nchunks, int N,
                                                    const int* __restrict__ rowoff, const int* __restrict__ jinv,
                                                    int nlist, int nvec, JPtrs<ND> J, int nbj,
                                                    const double* __restrict__ Kpart, int64_t dstride, DTiles tm,
                                                    KPtrs K) {
    if ((int)blockIdx.x < nbj) {
        j_reduce_body<VEC, ND>(jpart, nchunks, N, rowoff, jinv, nlist, nvec, J, blockIdx.x);
        return;
    }
    const int per = k_reduce_blocks(N), b = blockIdx.x - nbj, d = b / per;
    const int nb = (N + 15) / 16, m4 = b % per / nb, n16 = b % per % nb;
    if (n16 * 16 > m4 * 4 + 3) return;
    k_reduce_body(Kpart + d * dstride, dtile_splits(tm, m4, n16), N, K.p[d], m4, n16);
}

// The second J pass of a small build with gamma formed by its own blocks from
// the half-transform's row sums (gamma_rows_kernel's sums in the same order),
// which saves a launch; a block has at most kGBlock values of P.
template <int VEC, int EPT, int ND>
__global__ __launch_bounds__(kJThreads) void j_accum_rows_kernel(const double* __restrict__ B, int N, int Q,
                                                                 const double* __restrict__ grow, int64_t gstride,
                                                                 int ncolt, const int* __restrict__ rowoff,
                                                                 const uint32_t* __restrict__ elist, int nvec, int ppw,
                                                                 double* __restrict__ jpart) {
    __shared__ double g[ND * kGBlock];
    const int P0 = blockIdx.y * ppw, np = min(Q, P0 + ppw) - P0;
    const int lane = threadIdx.x & 63;
    for (int t = threadIdx.x >> 6; t < ND * np; t += kJThreads / 64) {
        const int d = t / np, p = t % np;
        double s = 0.0;
        for (int ct = 0; ct < ncolt; ++ct) {
            const double* r = grow + (int64_t)(ct * ND + d) * gstride + (int64_t)(P0 + p) * N;
            for (int m = lane; m < N; m += 64) s += r[m];
        }
        s = wave_sum(s);
        if (lane == 0) g[d * kGBlock + p] = s;
    }
    __syncthreads();
    const auto gamma = [&](int d, int P) { return g[d * kGBlock + P - P0]; };
    j_accum_kernel_body<double, VEC, EPT, ND, true>(B, N, Q, gamma, rowoff, nvec, ppw, jpart, blockIdx.x, blockIdx.y,
                                                    elist);
}

// ---------------------------------------------------------------------------
// Coefficients and D of the builds whose J needs D (FP32 and BF16x3 forms, J
// alone from C): one launch for every copy and density, and one for D.
// Rounds of launches bound both: at nbf 384 with 80 columns in BF16x3 five
// launches took 43 us (D's 128 x 128 tiles, six workgroups: 23 us, and its
// mirror); with these two the build went from 751 to 735 us, builds of 90 us
// lost 9 (one density) and 26 us (two).
// ---------------------------------------------------------------------------
struct PackOut {
    double* Cp;     // N x OPAD, or null
    float* Cp32;    // the same in FP32, or null
    u16 *Th, *Tl;   // transposed hi/lo bf16 planes, rows x KP with zeros past nocc and N, or null
    int rows, KP;
};
__global__ void pack_c_kernel(DCoef cs, DCols dc, int N, int OPAD, PackOut out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int c, k;
    if (out.Th) {
        if (t >= (int64_t)out.rows * out.KP) return;
        c = (int)(t / out.KP), k = (int)(t % out.KP);
    } else {
        if (t >= (int64_t)N * OPAD) return;
        k = (int)(t / OPAD), c = (int)(t % OPAD);
    }
    double x = 0.0;
    for (int d = 0; d < dc.nd; ++d) {
        const int i = c - dc.ioff[d];
        if (i >= 0 && i < dc.nocc[d] && k < N) x = cs.C[d][(int64_t)k * cs.ldc[d] + i];
    }
    if (out.Th) {
        __bf16 h, l;
        split_bf16_from_double(x, h, l);
        out.Th[t] = __builtin_bit_cast(u16, h);
        out.Tl[t] = __builtin_bit_cast(u16, l);
    }
    if (k < N && c < OPAD) {
        if (out.Cp) out.Cp[(int64_t)k * OPAD + c] = x;
        if (out.Cp32) out.Cp32[(int64_t)k * OPAD + c] = (float)x;
    }
}

// D = Cp Cp^T over the columns [ioff, ioff + width) (a multiple of 16): one
// 32 x 32 tile of the lower triangle per wave, operands from global memory
// (Cp is small enough for L2), a 16-k step ahead.  No mirror: J reads the lower
// triangle only.
constexpr int kDTile = 32;
__host__ __device__ inline int d_blocks(int N) {  // of four waves
    const int nt = (N + kDTile - 1) / kDTile;
    return (nt * (nt + 1) / 2 + 3) / 4;
}
__device__ __forceinline__ void d_body(const double* __restrict__ Cp, int N, int OPAD, int ioff, int width,
                                       double* __restrict__ D, int b) {
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int t = b * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nt = (N + kDTile - 1) / kDTile;
    if (t >= nt * (nt + 1) / 2) return;
    int mt = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (mt * (mt + 1) / 2 > t) --mt;
    while ((mt + 1) * (mt + 2) / 2 <= t) ++mt;
    const int m0 = mt * kDTile, n0 = (t - mt * (mt + 1) / 2) * kDTile;
    const double *ap[2], *bp[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // rows past N are clamped onto the last and never stored
        const int r = m0 + i * 16 + lr, c = n0 + i * 16 + lr;
        ap[i] = Cp + (int64_t)(r < N ? r : N - 1) * OPAD + ioff + 2 * lg;
        bp[i] = Cp + (int64_t)(c < N ? c : N - 1) * OPAD + ioff + 2 * lg;
    }
    dx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = dx4{0, 0, 0, 0};
    dx2 an[2][2], bn[2][2];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                an[i][h] = *reinterpret_cast<const dx2*>(ap[i] + k0 + 8 * h);
                bn[i][h] = *reinterpret_cast<const dx2*>(bp[i] + k0 + 8 * h);
            }
    };
    load(0);
    for (int k0 = 0; k0 < width; k0 += 16) {
        dx2 a[2][2], c[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) a[i][h] = an[i][h], c[i][h] = bn[i][h];
        if (k0 + 16 < width) load(k0 + 16);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma4(a[i][h].x, c[j][h].x, acc[i][j]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma4(a[i][h].y, c[j][h].y, acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + i * 16 + acc_row<double>(lane, r), n = n0 + j * 16 + lr;
                if (m < N && n < N) D[(int64_t)m * N + n] = acc[i][j][r];
            }
}
__global__ __launch_bounds__(256) void d_kernel(const double* __restrict__ Cp, int N, int OPAD, DCols dc,
                                                double* __restrict__ D) {
    const int d = blockIdx.y;
    d_body(Cp, N, OPAD, dc.ioff[d], dc.width[d], D + (int64_t)d * N * N, blockIdx.x);
}

}  // namespace f2jk
