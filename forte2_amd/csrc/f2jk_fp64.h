// FP64 half-transform X = B C (gfx950) on v_mfma_f64_16x16x4.
//
// Rates (random B): 65 TFLOP/s at nbf 1152 with 240 and 320 columns, where the
// same kernel without its loads of B reaches 67-68 (the clock under FP64 MFMA
// load, not the 78.6 TFLOP/s of 2.4 GHz, is the ceiling) and the 128 x 320
// tiles before it reached 46 (240 of 320 columns in use); 56 at nbf 384 with 80
// columns (42 before: 80 of 128).  Below about 50 columns it is bound by
// reading B: 4.2 TB/s of B and X at nbf 318.
//
// One FP64 MFMA keeps a SIMD's matrix pipe busy for 64 cycles, so the kernel
// is bound by how evenly the 16 x 16 output blocks are spread over the SIMDs
// as long as loads run a step ahead; LDS and L2 have room to spare.  So every
// wave gets whole rows (16 * IB of them) and all the occupied columns of the
// tile (NB blocks of 16, exactly the job's width): no wave holds padding
// columns, and A = B(P|mn) goes from global memory straight into MFMA operands,
// each element loaded once by one lane.
//
// Operand order.  A k step of 8 feeds two MFMAs: lane group g = lane / 16
// holds k = 2g and 2g + 1 and supplies the first to MFMA 0 and the second to
// MFMA 1.  The k sum is the same set of products in another order, and every
// lane's operands are 16 contiguous bytes, in global memory and in LDS.
//
// The coefficients reach LDS by direct-to-LDS loads (lane l to slot l of 16
// bytes) in the order in which the fragments are read: every LDS read is 1 KB
// of consecutive bytes.  A load into LDS is not ordered with register loads, so a step ends
// with a full drain before its barrier; the loads have had the whole step.
#pragma once
#include "f2jk_kernels.h"

namespace f2jk {

typedef double dx2 __attribute__((ext_vector_type(2)));
// rows of B start at a multiple of 8 bytes only when nbf is odd
typedef double dx2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kDK = 16;         // k extent of one LDS stage
constexpr int kDMaxNB = 20;     // 16-column blocks of the widest tile
constexpr int kDMaxDens = 8;
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
};

// ---------------------------------------------------------------------------
// Coefficients of all densities in the two forms the kernels read:
//   Cp[n][c]  row-major, OPAD columns (D = C C^T);
//   Cq        [column tile][16-k step][block][k / 8 % 2][lane][2], the order
//             of the half-transform's LDS tiles; zero outside N x nocc.
// ---------------------------------------------------------------------------
struct DCoef {
    const double* C[kDMaxDens];
    int64_t ldc[kDMaxDens];
};
__device__ __forceinline__ void pack_cq_element(const double* const* C, const int64_t* ldc, int nd,
                                                const int* nocc, const int* ioff, int N, int OPAD, int nb, int nks,
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
    if (k < N && c < OPAD) Cp[(int64_t)k * OPAD + c] = x;
}
__global__ void pack_cq_kernel(DCoef cs, DCols dc, int N, int OPAD, int nb, int nks, int64_t total,
                               double* __restrict__ Cp, double* __restrict__ Cq) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < total) pack_cq_element(cs.C, cs.ldc, dc.nd, dc.nocc, dc.ioff, N, OPAD, nb, nks, t, Cp, Cq);
}

// ---------------------------------------------------------------------------
// Half-transform: X[r][c] = sum_k A[r][k] C[k][c], r < R, for a tile of
// NB * 16 columns; 4 waves of 16 * IB rows each.
// ---------------------------------------------------------------------------
template <int NB, int IB>
__device__ __forceinline__ void kxd_body(char* lds, const double* __restrict__ A, int64_t R, int K,
                                         const double* __restrict__ Cq, int nks, double* __restrict__ X,
                                         int64_t ldx, int ncol, int ncolt, int b, int nblocks) {
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
}

template <int NB, int IB>
__global__ __launch_bounds__(256, 2) void kxd_kernel(const double* __restrict__ A, int64_t R, int K,
                                                     const double* __restrict__ Cq, int nks, double* __restrict__ X,
                                                     int64_t ldx, int ncol, int ncolt) {
    __shared__ __attribute__((aligned(16))) char lds[kDKxLds(NB)];
    kxd_body<NB, IB>(lds, A, R, K, Cq, nks, X, ldx, ncol, ncolt, blockIdx.x, gridDim.x);
}

}  // namespace f2jk
