// Grouped (multi-job) J/K launches for the serving layer.
//
// One persistent launch per phase covers the blocks of every job in the
// group.  A block walks the concatenated block index space with a stride of
// gridDim.x, finds its job from the launch's table of first blocks (a short
// uniform scan, at most kMaxGroup jobs) and runs the same device body as the
// single-job kernels with the job's own plan.  The decomposition of a job
// (element groups, P chunks, K splits) is its own plan, independent of the
// other jobs; the tile width of the BF16x3 half-transform is the group's
// (the widest job's), which changes which block computes an element of X but
// not the order of its k-sum.  So a job's J/K are bitwise the same alone and
// in any mix.
//
// Precisions: FP64 (J and K from the FP64 B), FP32 and BF16x3 (J from the
// FP32 B with FP64 accumulation, K on MFMA from the FP32 B), one precision
// per group.  A job computes J and K, or K only.
//
// The job table travels by value in the kernel arguments (kMaxGroup jobs fit
// the 4 KiB argument limit), so a launch needs no descriptor upload.
// Restrictions of the grouped path: nbf even, one X chunk per job.
#pragma once
#include <type_traits>

#include "f2jk.h"
#include "f2jk_kernels.h"
#include "f2jk_fp64.h"

namespace f2jk {

constexpr int kMaxGroup = 12;

enum GroupPhase {
    GP_PAD = 0,      // Cp[n][ioff+i] = C[n][i] (FP64; also the half-transform's copy of
                     // FP64 K, the FP32 copy, or the transposed hi/lo bf16 copies)
    GP_D = 1,        // D[d] = Cp_d Cp_d^T, lower tiles (precision forms)
    GP_GAMMA = 2,    // J pass 1 (precision forms)
    GP_GRED = 3,     // gamma reduction (FP64: of the half-transform's row sums)
    GP_JACC = 4,     // J pass 2
    GP_JRED = 5,     // J reduction + mirror
    GP_KX = 6,       // half-transform (whole B: one chunk)
    GP_KS = 7,       // contraction, splits of P
    GP_KRED = 8,     // K reduction + mirror
    GP_NPHASE = 9
};

struct GJob {
    const void* B;        // FP64 B (FP64 groups) or the FP32 copy (FP32 / BF16x3 groups)
    const int* rowoff;
    const double* C[2];
    double *Cp, *D, *gpart, *gamma, *jpart, *Kpart;
    double *Cq, *grow;    // FP64: coefficients in the half-transform's order, its row sums
    float* Cp32;          // FP32 coefficients (FP32 K)
    u16 *Cth, *Ctl;       // transposed hi/lo coefficients (BF16x3 K)
    void* X;              // half-transformed chunk: FP64, FP32, or hi then lo bf16
    double* J[2];
    double* K[2];
    int64_t ldc[2];
    int N, Q, nd, nocc[2], width[2], ioff[2], OPAD, KP;
    int nvec, neg, npc1, npc2, ppw2;
    int nlower, nsplit, ncolt;
    int dnb, dncolt, dnks, drows;  // FP64 half-transform; rows of a workgroup
    DTiles dt;              // FP64 contraction
    int want_j;
};

struct GArgs {
    int njobs;
    int first[kMaxGroup + 1];  // first block of each job in the launch's phase, then the total
    GJob job[kMaxGroup];
};
static_assert(sizeof(GArgs) <= 4096, "the job table must fit the kernel argument limit");

__host__ __device__ inline int gcdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

// blocks of one job in one phase (256 threads per block everywhere)
template <int PREC>
__host__ __device__ inline int phase_blocks(const GJob& g, int phase) {
    const int j = g.want_j ? 1 : 0;
    switch (phase) {
        case GP_PAD:
            if (PREC == F2JK_PREC_FP64) return g.dncolt * g.dnks * g.dnb;
            return gcdiv((long long)(PREC == F2JK_PREC_BF16X3 ? g.KP : g.N) * g.OPAD, 256);
        case GP_D: return j * d_blocks(g.N) * g.nd;
        case GP_GAMMA: return j * g.neg * g.npc1;
        case GP_GRED: return j * gcdiv((long long)g.nd * g.Q, PREC == F2JK_PREC_FP64 ? 4 : 256);
        case GP_JACC: return j * g.neg * g.npc2;
        case GP_JRED: return j * gcdiv(g.nvec, kJRedElems);
        case GP_KX:
            if (PREC == F2JK_PREC_FP64) return gcdiv((long long)g.Q * g.N, g.drows) * g.dncolt;
            return gcdiv((long long)g.Q * g.N, kTile) * g.ncolt;
        case GP_KS: return (PREC == F2JK_PREC_FP64 ? g.dt.total : g.nlower * g.nsplit) * g.nd;
        case GP_KRED: return k_reduce_blocks(g.N) * g.nd;
    }
    return 0;
}

// the FP64 half-transform of one job: the body of its width.  The job's fields
// are read once, before the choice: with a use in every body the compiler
// would copy the whole job table to scratch memory.
struct GKxd {
    const double *B, *Cq, *Cp;
    double *X, *grow;
    int64_t R;
    int N, nks, OPAD, ncolt;
    DCols2 dc;
};
// MAXNB 8: narrow jobs only, one row block per wave (116 registers and 32 KB of
// LDS: four workgroups per CU); 20: every width (235 registers, two).  A group
// with one job of more than 128 columns runs all its jobs in the second.
constexpr int kGroupNarrowNB = 8;
constexpr int grouped_kxd_ib(int maxnb, int nb) { return maxnb == kGroupNarrowNB ? 1 : kxd_ib(nb); }
template <int MAXNB, int NB = 1>
__device__ __forceinline__ void grouped_kxd(char* lds, int nb, const GKxd& k, int b, int nblocks) {
    if constexpr (NB <= MAXNB) {
        if (nb == NB)
            kxd_body<NB, grouped_kxd_ib(MAXNB, NB)>(lds, k.B, k.R, k.N, k.Cq, k.nks, k.X, k.OPAD, k.OPAD, k.ncolt, k.Cp, k.dc, k.grow,
                                     k.R, b, nblocks);
        else
            grouped_kxd<MAXNB, NB + 1>(lds, nb, k, b, nblocks);
    }
}

// PREC: the group's precision; NBW, VA: tile width and load width of the
// BF16x3 half-transform; NBW of the FP64 one: its widest column tile, in blocks.
template <int PHASE, int PREC, int NBW = 2, int VA = 2>
__global__ __launch_bounds__(256, PREC == F2JK_PREC_FP64 && PHASE == GP_KX && NBW == kGroupNarrowNB ? 4
                                  : PREC != F2JK_PREC_BF16X3 ? (PHASE == GP_KX || PHASE == GP_KS ? 2 : 1)
                                  : PHASE == GP_KX ? kx_bf16_waves_per_eu<NBW>()
                                  : PHASE == GP_KS ? 2 : 1)
void grouped_kernel(const GArgs a) {
    using TB = typename std::conditional<PREC == F2JK_PREC_FP64, double, float>::type;
    const int total = a.first[a.njobs];
    for (int lb = blockIdx.x; lb < total; lb += gridDim.x) {
        int j = 0;
        while (lb >= a.first[j + 1]) ++j;
        const GJob& g = a.job[j];
        const int local = lb - a.first[j], nblocks = a.first[j + 1] - a.first[j];
        const int tid = threadIdx.x;
        if constexpr (PHASE == GP_PAD) {
            const long long t = (long long)local * 256 + tid;
            if constexpr (PREC == F2JK_PREC_BF16X3) {
                // one thread per (row n, column c) of Cp and per (c, k) of the
                // transposed hi/lo copy, k < KP (zero past N)
                if (t < (long long)g.KP * g.OPAD) {
                    const int c = (int)(t / g.KP), k = (int)(t % g.KP);
                    const int d = (g.nd == 2 && c >= g.ioff[1]) ? 1 : 0;
                    const int i = c - g.ioff[d];
                    const double x = (i < g.nocc[d] && k < g.N) ? g.C[d][(long long)k * g.ldc[d] + i] : 0.0;
                    __bf16 h, l;
                    split_bf16_from_double(x, h, l);
                    g.Cth[t] = __builtin_bit_cast(u16, h);
                    g.Ctl[t] = __builtin_bit_cast(u16, l);
                    if (k < g.N) g.Cp[(long long)k * g.OPAD + c] = x;
                }
            } else if constexpr (PREC == F2JK_PREC_FP64) {
                pack_cq_element(g.C, g.ldc, g.nd, g.nocc, g.ioff, g.N, g.dncolt * g.dnb * 16, g.dnb, g.dnks, t, g.Cp, g.Cq);
            } else if (t < (long long)g.N * g.OPAD) {
                const int n = (int)(t / g.OPAD), c = (int)(t % g.OPAD);
                const int d = (g.nd == 2 && c >= g.ioff[1]) ? 1 : 0;
                const int i = c - g.ioff[d];
                const double x = (i < g.nocc[d]) ? g.C[d][(long long)n * g.ldc[d] + i] : 0.0;
                g.Cp[t] = x;
                g.Cp32[t] = (float)x;
            }
        } else if constexpr (PHASE == GP_D) {
            const int per = d_blocks(g.N), d = local / per;
            d_body(g.Cp, g.N, g.OPAD, g.ioff[d], g.width[d], g.D + (long long)d * g.N * g.N, local % per);
        } else if constexpr (PHASE == GP_KRED) {
            const int per = k_reduce_blocks(g.N), nb = gcdiv(g.N, 16);
            const int d = local / per, m4 = local % per / nb, n16 = local % per % nb;
            const long long NN = (long long)g.N * g.N;
            if (n16 * 16 <= m4 * 4 + 3)
                k_reduce_body(g.Kpart + d * g.nsplit * NN,
                              PREC == F2JK_PREC_FP64 ? dtile_splits(g.dt, m4, n16) : g.nsplit, g.N, g.K[d], m4, n16);
        } else if constexpr (PHASE == GP_GAMMA) {
            const int bx = local % g.neg, by = local / g.neg;
            const long long NN = (long long)g.N * g.N;
            const TB* B = (const TB*)g.B;
            if (g.nd == 2) {
                DPtrs<2> dp{{g.D, g.D + NN}};
                j_gamma_kernel_body<TB, 2, 4, 2, true>(B, g.N, g.Q, dp, g.N, g.rowoff, g.nvec, 32, g.gpart, bx, by);
            } else {
                DPtrs<1> dp{{g.D}};
                j_gamma_kernel_body<TB, 2, 4, 1, true>(B, g.N, g.Q, dp, g.N, g.rowoff, g.nvec, 32, g.gpart, bx, by);
            }
        } else if constexpr (PHASE == GP_GRED && PREC == F2JK_PREC_FP64) {
            const long long t = (long long)local * 4 + (tid >> 6);
            if (t < (long long)g.nd * g.Q)
                gamma_rows_body(g.grow, (long long)g.Q * g.N, g.nd, g.dncolt, g.N, g.gamma, g.Q, (int)(t / g.Q),
                                (int)(t % g.Q));
        } else if constexpr (PHASE == GP_GRED) {
            const long long t = (long long)local * 256 + tid;
            if (t < (long long)g.nd * g.Q) {
                const int dd = (int)(t / g.Q), P = (int)(t % g.Q);
                double s = 0.0;
#pragma unroll 8
                for (int q = 0; q < g.neg; ++q) s += g.gpart[((long long)q * g.nd + dd) * g.Q + P];
                g.gamma[t] = s;
            }
        } else if constexpr (PHASE == GP_JACC) {
            const int bx = local % g.neg, by = local / g.neg;
            const TB* B = (const TB*)g.B;
            if (g.nd == 2)
                j_accum_kernel_body<TB, 2, 4, 2, true>(B, g.N, g.Q, GammaAll{g.gamma, g.Q}, g.rowoff, g.nvec, g.ppw2, g.jpart, bx, by);
            else
                j_accum_kernel_body<TB, 2, 4, 1, true>(B, g.N, g.Q, GammaAll{g.gamma, g.Q}, g.rowoff, g.nvec, g.ppw2, g.jpart, bx, by);
        } else if constexpr (PHASE == GP_JRED) {
            if (g.nd == 2) {
                JPtrs<2> jp{{g.J[0], g.J[1]}};
                j_reduce_body<2, 2>(g.jpart, g.npc2, g.N, g.rowoff, nullptr, g.nvec, g.nvec, jp, local);
            } else {
                JPtrs<1> jp{{g.J[0]}};
                j_reduce_body<2, 1>(g.jpart, g.npc2, g.N, g.rowoff, nullptr, g.nvec, g.nvec, jp, local);
            }
        } else if constexpr (PHASE == GP_KX) {
            const int nb = nblocks;
            const long long R = (long long)g.Q * g.N;
            if constexpr (PREC == F2JK_PREC_FP64) {
                __shared__ __attribute__((aligned(16))) char lds[kDKxLds(NBW)];
                const GKxd k{(const double*)g.B, g.Cq, g.Cp, (double*)g.X, g.want_j ? g.grow : nullptr, R, g.N, g.dnks,
                             g.OPAD, g.dncolt,
                             DCols2{g.nd, g.ioff[0], g.ioff[0] + g.width[0], g.ioff[1], g.ioff[1] + g.width[1]}};
                grouped_kxd<NBW>(lds, g.dnb, k, local, nb);
            } else if constexpr (PREC == F2JK_PREC_FP32) {
                kx_kernel_body<2>((const float*)g.B, R, g.N, g.Cp32, g.OPAD, (float*)g.X, g.ncolt, local, nb);
            } else {
                u16* xh = (u16*)g.X;
                kx_bf16x3_kernel_body<NBW, VA>((const float*)g.B, R, g.N, g.KP, g.Cth, g.Ctl, g.OPAD, xh,
                                               xh + R * g.OPAD, g.ncolt, local, nb);
            }
        } else if constexpr (PHASE == GP_KS) {
            const int per = PREC == F2JK_PREC_FP64 ? g.dt.total : g.nlower * g.nsplit;
            const int d = local / per, b = local % per;
            double* kp = g.Kpart + (long long)d * g.nsplit * g.N * g.N;
            if constexpr (PREC == F2JK_PREC_BF16X3) {
                const u16* xh = (const u16*)g.X;
                ks_bf16x3_kernel_body<kTile, 2, 2>(xh, xh + (long long)g.Q * g.N * g.OPAD, g.N, g.OPAD, g.ioff[d], g.width[d],
                                      g.Q, g.nsplit, g.nlower, kp, 0, b, per);
            } else if constexpr (PREC == F2JK_PREC_FP64) {
                __shared__ __attribute__((aligned(16))) char lds[kDKsLds];
                ksd_body(lds, (const double*)g.X, g.N, g.OPAD, g.ioff[d], g.width[d], g.Q, g.dt, kp, 0, b);
            } else {
                ks_kernel_body((const float*)g.X, g.N, g.OPAD, g.ioff[d], g.width[d], g.Q, g.nsplit, g.nlower,
                                   kp, 0, b, per);
            }
        }
    }
}

}  // namespace f2jk
