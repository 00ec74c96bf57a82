// Device kernels of the density-fitted J/K builder (gfx950 / CDNA4).
//
// Data layout in HBM
//   B[P][m][n]   naux x nbf x nbf, row-major, symmetric in (m, n) -- the
//                reference layout of FockBuilder.B_Pmn
//                (forte2/jkbuilder/jkbuilder.py:52-72).
//   Cp[n][i]     nbf x OPAD, occupied coefficients of all densities side by
//                side, each density's block padded with zero columns to a
//                multiple of 16 (the MFMA k step of the contraction).
//   X[P][m][i]   half-transformed tensor of one P chunk, Pc x nbf x OPAD.
//
// J (two passes over the lower triangle of B, HBM-bound):
//   pass 1  gamma_P = sum_{m>=n} w_mn B_Pmn D_mn,  w = 2 (m>n), 1 (m=n)
//   pass 2  J_mn    = sum_P gamma_P B_Pmn           (m >= n, mirrored)
//   The lower triangle is walked as "vector elements": row m is cut into
//   ceil((m+1)/VEC) aligned VEC-wide pieces (16-byte loads), numbered
//   row after row; rowoff[m] is the number of pieces in rows < m.
// K (MFMA, compute-bound):
//   KX  X = B_chunk Cp           one tall GEMM, (Pc*N) x N x OPAD
//   KS  Kpart[s] += sum_{P in split s} X_P X_P^T   lower 128x128 tiles only
//   KR  K = sum_s Kpart[s], lower triangle mirrored to the upper one
// All reductions run in a fixed order (no atomics): the result of a build is
// a function of its inputs and shapes only.
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace f2jk {

constexpr int kWave = 64;
constexpr int kJThreads = 256;
constexpr int kJFlush = 32;  // P values reduced across waves per LDS flush

typedef double dx4 __attribute__((ext_vector_type(4)));
typedef float fx4 __attribute__((ext_vector_type(4)));

template <typename T, int V>
struct alignas(sizeof(T) * V) Vec {
    T v[V];
};

template <typename T, int V>
__device__ __forceinline__ Vec<T, V> load_vec(const T* p) {
    return *reinterpret_cast<const Vec<T, V>*>(p);
}

template <typename T, int V>
struct NTVec {
    typedef T type __attribute__((ext_vector_type(V)));
};

// streaming load that bypasses cache retention (data read once per pass)
template <typename T, int V, bool NT>
__device__ __forceinline__ Vec<T, V> stream_vec(const T* p) {
    if constexpr (NT && V > 1) {
        typedef typename NTVec<T, V>::type vt;
        const vt x = __builtin_nontemporal_load(reinterpret_cast<const vt*>(p));
        Vec<T, V> r;
#pragma unroll
        for (int v = 0; v < V; ++v) r.v[v] = x[v];
        return r;
    } else if constexpr (NT) {
        Vec<T, V> r;
        r.v[0] = __builtin_nontemporal_load(p);
        return r;
    } else {
        return load_vec<T, V>(p);
    }
}

template <int ND>
struct DPtrs {
    const double* p[ND];
};
template <int ND>
struct JPtrs {
    double* p[ND];
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// largest m in [0, n) with rowoff[m] <= e  (rowoff[0] = 0, rowoff[n] = total)
__device__ __forceinline__ int find_row(const int* __restrict__ rowoff, int n, int e) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (rowoff[mid] <= e)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Blocks are dispatched round-robin over the 8 XCDs (each with its own L2).
// Give every XCD a contiguous range of logical tile ids so that tiles that
// share operands run on the same L2.
__device__ __forceinline__ int xcd_remap(int b, int nblocks) {
    constexpr int NX = 8;
    const int xcd = b % NX, local = b / NX;
    const int base = nblocks / NX, rem = nblocks % NX;
    return xcd * base + (xcd < rem ? xcd : rem) + local;
}

// ---------------------------------------------------------------------------
// J pass 1: partial gamma per (element group, density, P).
// grid = (n_element_groups, ceil(Q / ppw)), block = 256.
// ---------------------------------------------------------------------------
// Vector element e of the lower triangle: row m and first column col.  With
// an element list (only the elements where B is nonzero for some P, packed
// as m << 16 | col) e indexes the list; otherwise elements are numbered row
// after row through rowoff.
template <int VEC>
__device__ __forceinline__ void j_element(const int* __restrict__ rowoff, const uint32_t* __restrict__ elist, int N,
                                          int e, int& m, int& col) {
    if (elist) {
        const uint32_t x = elist[e];
        m = (int)(x >> 16);
        col = (int)(x & 0xffffu);
    } else {
        m = find_row(rowoff, N, e);
        col = (e - rowoff[m]) * VEC;
    }
}

template <typename TB, int VEC, int EPT, int ND, bool NT = false>
__device__ __forceinline__ void j_gamma_kernel_body(
    const TB* __restrict__ B, int N, int Q, DPtrs<ND> D, int64_t ldd,
    const int* __restrict__ rowoff, int nvec, int ppw, double* __restrict__ gpart, int bx, int by,
    const uint32_t* __restrict__ elist = nullptr, const TB* __restrict__ packed = nullptr) {
    __shared__ double red[kJThreads / kWave][kJFlush][ND];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
    const int64_t NN = packed ? (int64_t)nvec * VEC : (int64_t)N * N;
    if (packed) B = packed;

    int64_t off[EPT];
    double d[EPT][ND][VEC];
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const int e = bx * (kJThreads * EPT) + k * kJThreads + tid;
        off[k] = 0;
#pragma unroll
        for (int dd = 0; dd < ND; ++dd)
#pragma unroll
            for (int v = 0; v < VEC; ++v) d[k][dd][v] = 0.0;
        if (e < nvec) {
            int m, col;
            j_element<VEC>(rowoff, elist, N, e, m, col);
            off[k] = packed ? (int64_t)e * VEC : (int64_t)m * N + col;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const int c = col + v;
                const double w = (c < m) ? 2.0 : (c == m ? 1.0 : 0.0);
#pragma unroll
                for (int dd = 0; dd < ND; ++dd)
                    d[k][dd][v] = (w != 0.0) ? w * D.p[dd][(int64_t)m * ldd + c] : 0.0;
            }
        }
    }

    const int P0 = by * ppw;
    const int P1 = min(Q, P0 + ppw);
    for (int Pb = P0; Pb < P1; Pb += kJFlush) {
        const int np = min(kJFlush, P1 - Pb);
        int j = 0;
        for (; j + 1 < np; j += 2) {
            const TB* B0 = B + (int64_t)(Pb + j) * NN;
            const TB* B1 = B0 + NN;
            Vec<TB, VEC> b0[EPT], b1[EPT];
#pragma unroll
            for (int k = 0; k < EPT; ++k) {
                b0[k] = stream_vec<TB, VEC, NT>(B0 + off[k]);
                b1[k] = stream_vec<TB, VEC, NT>(B1 + off[k]);
            }
            double a0[ND], a1[ND];
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) a0[dd] = a1[dd] = 0.0;
#pragma unroll
            for (int k = 0; k < EPT; ++k)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
#pragma unroll
                    for (int dd = 0; dd < ND; ++dd) {
                        a0[dd] = fma((double)b0[k].v[v], d[k][dd][v], a0[dd]);
                        a1[dd] = fma((double)b1[k].v[v], d[k][dd][v], a1[dd]);
                    }
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) {
                a0[dd] = wave_sum(a0[dd]);
                a1[dd] = wave_sum(a1[dd]);
            }
            if (lane == 0) {
#pragma unroll
                for (int dd = 0; dd < ND; ++dd) {
                    red[wid][j][dd] = a0[dd];
                    red[wid][j + 1][dd] = a1[dd];
                }
            }
        }
        if (j < np) {
            const TB* B0 = B + (int64_t)(Pb + j) * NN;
            double a0[ND];
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) a0[dd] = 0.0;
#pragma unroll
            for (int k = 0; k < EPT; ++k) {
                Vec<TB, VEC> b0 = stream_vec<TB, VEC, NT>(B0 + off[k]);
#pragma unroll
                for (int v = 0; v < VEC; ++v)
#pragma unroll
                    for (int dd = 0; dd < ND; ++dd)
                        a0[dd] = fma((double)b0.v[v], d[k][dd][v], a0[dd]);
            }
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) a0[dd] = wave_sum(a0[dd]);
            if (lane == 0) {
#pragma unroll
                for (int dd = 0; dd < ND; ++dd) red[wid][j][dd] = a0[dd];
            }
        }
        __syncthreads();
        for (int t = tid; t < np * ND; t += kJThreads) {
            const int jj = t / ND, dd = t % ND;
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < kJThreads / kWave; ++w) s += red[w][jj][dd];
            gpart[((int64_t)bx * ND + dd) * Q + Pb + jj] = s;
        }
        __syncthreads();
    }
}
template <typename TB, int VEC, int EPT, int ND, bool NT = false>
__global__ __launch_bounds__(kJThreads) void j_gamma_kernel(
    const TB* __restrict__ B, int N, int Q, DPtrs<ND> D, int64_t ldd,
    const int* __restrict__ rowoff, const uint32_t* __restrict__ elist, const TB* __restrict__ packed, int nvec,
    int ppw, double* __restrict__ gpart) {
    j_gamma_kernel_body<TB, VEC, EPT, ND, NT>(B, N, Q, D, ldd, rowoff, nvec, ppw, gpart, blockIdx.x, blockIdx.y,
                                              elist, packed);
}


// gamma[dd][P] = sum_g gpart[g][dd][P], g in a fixed order.
__global__ void j_gamma_reduce_kernel(const double* __restrict__ gpart, int ngroups,
                                      int ND, int Q, double* __restrict__ gamma) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)ND * Q) return;
    const int dd = (int)(t / Q), P = (int)(t % Q);
    double s = 0.0;
#pragma unroll 8
    for (int g = 0; g < ngroups; ++g) s += gpart[((int64_t)g * ND + dd) * Q + P];
    gamma[t] = s;
}

constexpr int kGBlock = 16;  // most P values of a block that forms its own gamma
// ---------------------------------------------------------------------------
// J pass 2: partial J per (P chunk, density, element).
// grid = (n_element_groups, n_p_chunks), block = 256.
// ---------------------------------------------------------------------------
// gamma(d, P): gamma of every P in global memory, or a block's own in LDS
struct GammaAll {
    const double* g;
    int Q;
    __device__ __forceinline__ double operator()(int d, int P) const { return g[(int64_t)d * Q + P]; }
};
template <typename TB, int VEC, int EPT, int ND, bool NT = false, typename Gamma>
__device__ __forceinline__ void j_accum_kernel_body(
    const TB* __restrict__ B, int N, int Q, const Gamma& gamma,
    const int* __restrict__ rowoff, int nvec, int ppw, double* __restrict__ jpart, int bx, int by,
    const uint32_t* __restrict__ elist = nullptr, const TB* __restrict__ packed = nullptr) {
    const int tid = threadIdx.x;
    const int64_t NN = packed ? (int64_t)nvec * VEC : (int64_t)N * N;
    if (packed) B = packed;
    const int P0 = by * ppw;
    const int P1 = min(Q, P0 + ppw);
    int64_t off[EPT];
    int eidx[EPT];
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const int e = bx * (kJThreads * EPT) + k * kJThreads + tid;
        eidx[k] = e;
        off[k] = 0;
        if (e < nvec) {
            if (packed) {
                off[k] = (int64_t)e * VEC;
            } else {
                int m, col;
                j_element<VEC>(rowoff, elist, N, e, m, col);
                off[k] = (int64_t)m * N + col;
            }
        }
    }
    double acc[EPT][ND][VEC];
#pragma unroll
    for (int k = 0; k < EPT; ++k)
#pragma unroll
        for (int dd = 0; dd < ND; ++dd)
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[k][dd][v] = 0.0;

    int P = P0;
    for (; P + 1 < P1; P += 2) {
        const TB* B0 = B + (int64_t)P * NN;
        const TB* B1 = B0 + NN;
        Vec<TB, VEC> b0[EPT], b1[EPT];
#pragma unroll
        for (int k = 0; k < EPT; ++k) {
            b0[k] = stream_vec<TB, VEC, NT>(B0 + off[k]);
            b1[k] = stream_vec<TB, VEC, NT>(B1 + off[k]);
        }
        double g0[ND], g1[ND];
#pragma unroll
        for (int dd = 0; dd < ND; ++dd) {
            g0[dd] = gamma(dd, P);
            g1[dd] = gamma(dd, P + 1);
        }
#pragma unroll
        for (int k = 0; k < EPT; ++k)
#pragma unroll
            for (int dd = 0; dd < ND; ++dd)
#pragma unroll
                for (int v = 0; v < VEC; ++v) {
                    acc[k][dd][v] = fma(g0[dd], (double)b0[k].v[v], acc[k][dd][v]);
                    acc[k][dd][v] = fma(g1[dd], (double)b1[k].v[v], acc[k][dd][v]);
                }
    }
    if (P < P1) {
        const TB* B0 = B + (int64_t)P * NN;
#pragma unroll
        for (int k = 0; k < EPT; ++k) {
            Vec<TB, VEC> b0 = stream_vec<TB, VEC, NT>(B0 + off[k]);
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) {
                const double g = gamma(dd, P);
#pragma unroll
                for (int v = 0; v < VEC; ++v) acc[k][dd][v] = fma(g, (double)b0.v[v], acc[k][dd][v]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        if (eidx[k] >= nvec) continue;
#pragma unroll
        for (int dd = 0; dd < ND; ++dd) {
            double* dst = jpart + (((int64_t)by * ND + dd) * nvec + eidx[k]) * VEC;
#pragma unroll
            for (int v = 0; v < VEC; ++v) dst[v] = acc[k][dd][v];
        }
    }
}
template <typename TB, int VEC, int EPT, int ND, bool NT = false>
__global__ __launch_bounds__(kJThreads) void j_accum_kernel(
    const TB* __restrict__ B, int N, int Q, const double* __restrict__ gamma,
    const int* __restrict__ rowoff, const uint32_t* __restrict__ elist, const TB* __restrict__ packed, int nvec,
    int ppw, double* __restrict__ jpart) {
    j_accum_kernel_body<TB, VEC, EPT, ND, NT>(B, N, Q, GammaAll{gamma, Q}, rowoff, nvec, ppw, jpart, blockIdx.x, blockIdx.y,
                                              elist, packed);
}


// J[dd][m][c] = J[dd][c][m] = sum_chunk jpart[chunk][dd][e][v]  (c = col+v <= m)
// for every lower-triangle vector element; with a list of the elements that
// the passes ran over, jinv[element] is its place in the list (-1: B is zero
// there for every P, so is J).  A block holds 64 elements; its four waves sum
// every fourth chunk each and are added in order: the chunks of a small nbf
// are many (one per P or two), and one thread per element left the launch a
// serial chain (33 us at nbf 24 with 139 chunks, 5 us with four waves).
constexpr int kJRedElems = 64;
template <int VEC, int ND>
__device__ __forceinline__ void j_reduce_body(const double* __restrict__ jpart, int nchunks, int N,
                                              const int* __restrict__ rowoff, const int* __restrict__ jinv,
                                              int nlist, int nvec, const JPtrs<ND>& J, int b) {
    __shared__ double red[3][kJRedElems][ND * VEC];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = b * kJRedElems + lane;
    const int le = e < nvec ? (jinv ? jinv[e] : e) : -1;
    double s[ND][VEC];
#pragma unroll
    for (int dd = 0; dd < ND; ++dd)
#pragma unroll
        for (int v = 0; v < VEC; ++v) s[dd][v] = 0.0;
    if (le >= 0) {
#pragma unroll 8
        for (int c = w; c < nchunks; c += 4)
#pragma unroll
            for (int dd = 0; dd < ND; ++dd) {
                const Vec<double, VEC> x =
                    load_vec<double, VEC>(jpart + (((int64_t)c * ND + dd) * nlist + le) * VEC);
#pragma unroll
                for (int v = 0; v < VEC; ++v) s[dd][v] += x.v[v];
            }
    }
    if (w > 0)
#pragma unroll
        for (int dd = 0; dd < ND; ++dd)
#pragma unroll
            for (int v = 0; v < VEC; ++v) red[w - 1][lane][dd * VEC + v] = s[dd][v];
    __syncthreads();
    if (w == 0 && e < nvec) {
        const int m = find_row(rowoff, N, e);
        const int col = (e - rowoff[m]) * VEC;
#pragma unroll
        for (int dd = 0; dd < ND; ++dd)
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const int i = dd * VEC + v, cc = col + v;
                const double x = ((s[dd][v] + red[0][lane][i]) + red[1][lane][i]) + red[2][lane][i];
                if (cc <= m) {
                    J.p[dd][(int64_t)m * N + cc] = x;
                    J.p[dd][(int64_t)cc * N + m] = x;
                }
            }
    }
    __syncthreads();  // red is free again (a persistent block goes on to its next 64 elements)
}
template <int VEC, int ND>
__global__ __launch_bounds__(kJThreads) void j_reduce_kernel(const double* __restrict__ jpart, int nchunks, int N,
                                                             const int* __restrict__ rowoff,
                                                             const int* __restrict__ jinv, int nlist, int nvec,
                                                             JPtrs<ND> J) {
    j_reduce_body<VEC, ND>(jpart, nchunks, N, rowoff, jinv, nlist, nvec, J, blockIdx.y * gridDim.x + blockIdx.x);
}

// flag[e] = 1 when B[P][m][c] != 0 for some P and some c <= m of vector
// element e (lower triangle, numbered row after row): the elements the J
// passes have to read.  One thread per element and range of P (blockIdx.y);
// flag starts at zero and a thread that finds its element flagged by another
// range stops (one range over all P left most of the chip idle: 1.2 ms at nbf
// 384, 2224 P).
template <typename TB, int VEC>
__global__ void j_scan_kernel(const TB* __restrict__ B, int N, int Q, const int* __restrict__ rowoff, int nvec,
                              volatile unsigned char* flag) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nvec) return;
    const int m = find_row(rowoff, N, e);
    const int col = (e - rowoff[m]) * VEC;
    const int64_t NN = (int64_t)N * N;
    const TB* p = B + (int64_t)m * N + col;
    const int P0 = (int)((int64_t)Q * blockIdx.y / gridDim.y), P1 = (int)((int64_t)Q * (blockIdx.y + 1) / gridDim.y);
    for (int P = P0; P < P1; P += 8) {
        if (flag[e]) return;
        int nz = 0;
        const int np = min(8, P1 - P);
        for (int i = 0; i < np; ++i) {
            const Vec<TB, VEC> b = load_vec<TB, VEC>(p + (P + i) * NN);
#pragma unroll
            for (int v = 0; v < VEC; ++v) nz |= (col + v <= m) && (b.v[v] != TB(0));
        }
        if (nz) {
            flag[e] = 1;
            return;
        }
    }
}
__global__ void fill_bytes_kernel(unsigned char* __restrict__ x, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0;
}
// out[P][i] = the listed vector element i of B_P: what the J passes read, one
// after the other.  In B the listed elements lie scattered in 16-byte pieces,
// and whole 128-byte lines come from memory for them.
template <typename TB, int VEC>
__global__ void j_pack_kernel(const TB* __restrict__ B, int N, int Q, const uint32_t* __restrict__ elist, int n,
                              TB* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t x = elist[i];
    const TB* p = B + (int64_t)(x >> 16) * N + (x & 0xffffu);
    const int64_t NN = (int64_t)N * N;
    for (int P = blockIdx.y; P < Q; P += gridDim.y)
        *reinterpret_cast<Vec<TB, VEC>*>(out + ((int64_t)P * n + i) * VEC) = load_vec<TB, VEC>(p + P * NN);
}

// ---------------------------------------------------------------------------
// MFMA helpers.  v_mfma_{f64,f32}_16x16x4: lane l supplies A[l%16][l/16] and
// B[l/16][l%16].  Accumulator element r of lane l holds D[i][l%16] with
//   f32:  i = 4*(l/16) + r
//   f64:  i = (l/16) + 4*r          (measured on gfx950)
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ int acc_row(int lane, int r) {
    if constexpr (sizeof(T) == 8)
        return (lane >> 4) + 4 * r;
    else
        return 4 * (lane >> 4) + r;
}

__device__ __forceinline__ dx4 mfma4(double a, double b, dx4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ fx4 mfma4(float a, float b, fx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kTile = 128;   // output tile edge (rows and columns)
constexpr int kBK = 16;      // k extent of one LDS stage
constexpr int kGThreads = 256;

// ---------------------------------------------------------------------------
// KX (FP32):  X[r][c] = sum_k A[r][k] Cp[k][c]
//   A  = B of the chunk viewed as R x K row-major (R = Pc*N rows, K = N)
//   Cp = K x OPAD row-major (zero-padded columns), X = R x OPAD row-major.
// Tile 128 x 128, 4 waves as 2 x 2 blocks of 64 x 64 (4 x 4 MFMA blocks each).
// VA: elements per global load of A (16 B when the row length allows).
// ---------------------------------------------------------------------------
template <int VA>
__device__ __forceinline__ void kx_kernel_body(const float* __restrict__ A, int64_t R,
                                                       int K, const float* __restrict__ Cp,
                                                       int OPAD, float* __restrict__ X,
                                                       int ncolt, int b, int nblocks) {
    constexpr int VB = 4;       // B tile loads are always 16 B (OPAD % 16 == 0)
    __shared__ float As[2][kTile][kBK + 1];  // two stages: MFMAs read one, the next k-step fills the other
    __shared__ float Bs[2][kBK][kTile];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int t = xcd_remap(b, nblocks);
    const int64_t r0 = (int64_t)(t / ncolt) * kTile;
    const int c0 = (t % ncolt) * kTile;
    const int wr = wid >> 1, wc = wid & 1;
    const int wcol0 = c0 + wc * 64;
    int nbv = (OPAD - wcol0) / 16;
    nbv = nbv < 0 ? 0 : (nbv > 4 ? 4 : nbv);

    constexpr int A_LD = (kTile * kBK) / (kGThreads * VA);  // loads per thread
    constexpr int B_LD = (kTile * kBK) / (kGThreads * VB);
    Vec<float, VA> ra[A_LD];
    Vec<float, VB> rb[B_LD];

    auto load_tiles = [&](int k0) {
#pragma unroll
        for (int s = 0; s < A_LD; ++s) {
            const int idx = tid + kGThreads * s;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
            const int64_t gr = r0 + row;
            const int gk = k0 + kc;
            if (gr < R && gk < K) {
                ra[s] = load_vec<float, VA>(A + gr * K + gk);
            } else {
#pragma unroll
                for (int v = 0; v < VA; ++v) ra[s].v[v] = 0.0f;
            }
        }
#pragma unroll
        for (int s = 0; s < B_LD; ++s) {
            const int idx = tid + kGThreads * s;
            const int kr = idx / (kTile / VB), cc = (idx % (kTile / VB)) * VB;
            const int gk = k0 + kr, gc = c0 + cc;
            if (gk < K && gc < OPAD) {
                rb[s] = load_vec<float, VB>(Cp + (int64_t)gk * OPAD + gc);
            } else {
#pragma unroll
                for (int v = 0; v < VB; ++v) rb[s].v[v] = 0.0f;
            }
        }
    };
    auto store_tiles = [&](int stg) {
#pragma unroll
        for (int s = 0; s < A_LD; ++s) {
            const int idx = tid + kGThreads * s;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
#pragma unroll
            for (int v = 0; v < VA; ++v) As[stg][row][kc + v] = ra[s].v[v];
        }
#pragma unroll
        for (int s = 0; s < B_LD; ++s) {
            const int idx = tid + kGThreads * s;
            const int kr = idx / (kTile / VB), cc = (idx % (kTile / VB)) * VB;
#pragma unroll
            for (int v = 0; v < VB; ++v) Bs[stg][kr][cc + v] = rb[s].v[v];
        }
    };

    fx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nk = (K + kBK - 1) / kBK;
    load_tiles(0);
    store_tiles(0);
    __syncthreads();
    if (nk > 1) load_tiles(kBK);
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 4) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[cur][wr * 64 + i * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[cur][kk + (lane >> 4)][wc * 64 + j * 16 + (lane & 15)];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j < nbv) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i][j] = mfma4(a[i], b[j], acc[i][j]);
                }
            }
        }
        if (kt + 1 < nk) store_tiles(cur ^ 1);  // the other stage was last read before the previous barrier
        if (kt + 2 < nk) load_tiles((kt + 2) * kBK);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j >= nbv) continue;
            const int col = wcol0 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = r0 + wr * 64 + i * 16 + acc_row<float>(lane, r);
                if (row < R) X[row * OPAD + col] = acc[i][j][r];
            }
        }
}
template <int VA>
__global__ __launch_bounds__(kGThreads) void kx_kernel(const float* __restrict__ A, int64_t R,
                                                       int K, const float* __restrict__ Cp,
                                                       int OPAD, float* __restrict__ X,
                                                       int ncolt) {
    kx_kernel_body<VA>(A, R, K, Cp, OPAD, X, ncolt, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// KX, wide tiles: the product of kx_kernel with 128 x 320 output tiles, so that
// a 128-row block of B is read once for up to 320 occupied columns (the
// 128-column kernel reads it once per column tile: 3x at 320 columns).  8 waves
// as 2 x 4, each 64 x 80 (4 x 5 MFMA blocks), one workgroup per CU.  The k
// loop, the MFMA and each output element's accumulation order are those of
// kx_kernel, so X is bitwise the same.  The k-major coefficient tile is padded by 16
// elements per row: its fragment reads (4 k rows x 16 columns per wave
// instruction) then fall in distinct LDS banks.
// ---------------------------------------------------------------------------
constexpr int kWideCols = 320;
constexpr int kWideThreads = 512;

template <int VA>
__device__ __forceinline__ void kx_wide_body(const float* __restrict__ A, int64_t R, int K,
                                             const float* __restrict__ Cp, int OPAD, float* __restrict__ X,
                                             int ncolt, int b, int nblocks) {
    constexpr int TN = kWideCols, BS = TN + 16;
    constexpr int WC = 4, NB = TN / WC / 16;       // 5 column blocks per wave
    constexpr int VB = 2;                          // coefficient loads: 2 elements each
    constexpr int A_LD = (kTile * kBK) / (kWideThreads * VA);
    constexpr int B_LD = (kBK * TN) / (kWideThreads * VB);
    static_assert(A_LD * kWideThreads * VA == kTile * kBK && B_LD * kWideThreads * VB == kBK * TN,
                  "tiles must split evenly over the threads");
    __shared__ float As[2][kTile][kBK + 1];
    __shared__ float Bs[2][kBK][BS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = xcd_remap(b, nblocks);
    const int64_t r0 = (int64_t)(t / ncolt) * kTile;
    const int c0 = (t % ncolt) * TN;
    const int wr = wid / WC, wc = wid % WC;
    const int wcol0 = c0 + wc * 16 * NB;
    int nbv = (OPAD - wcol0) / 16;
    nbv = nbv < 0 ? 0 : (nbv > NB ? NB : nbv);

    Vec<float, VA> ra[A_LD];
    Vec<float, VB> rb[B_LD];
    auto load_tiles = [&](int k0) {
#pragma unroll
        for (int s = 0; s < A_LD; ++s) {
            const int idx = tid + kWideThreads * s;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
            const int64_t gr = r0 + row;
            const int gk = k0 + kc;
            if (gr < R && gk < K) {
                ra[s] = load_vec<float, VA>(A + gr * K + gk);
            } else {
#pragma unroll
                for (int v = 0; v < VA; ++v) ra[s].v[v] = 0.0f;
            }
        }
#pragma unroll
        for (int s = 0; s < B_LD; ++s) {
            const int idx = tid + kWideThreads * s;
            const int kr = idx / (TN / VB), cc = (idx % (TN / VB)) * VB;
            const int gk = k0 + kr, gc = c0 + cc;
            if (gk < K && gc < OPAD) {
                rb[s] = load_vec<float, VB>(Cp + (int64_t)gk * OPAD + gc);
            } else {
#pragma unroll
                for (int v = 0; v < VB; ++v) rb[s].v[v] = 0.0f;
            }
        }
    };
    auto store_tiles = [&](int stg) {
#pragma unroll
        for (int s = 0; s < A_LD; ++s) {
            const int idx = tid + kWideThreads * s;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
#pragma unroll
            for (int v = 0; v < VA; ++v) As[stg][row][kc + v] = ra[s].v[v];
        }
#pragma unroll
        for (int s = 0; s < B_LD; ++s) {
            const int idx = tid + kWideThreads * s;
            const int kr = idx / (TN / VB), cc = (idx % (TN / VB)) * VB;
#pragma unroll
            for (int v = 0; v < VB; ++v) Bs[stg][kr][cc + v] = rb[s].v[v];
        }
    };

    fx4 acc[4][NB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nk = (K + kBK - 1) / kBK;
    load_tiles(0);
    store_tiles(0);
    __syncthreads();
    if (nk > 1) load_tiles(kBK);
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 4) {
            float a[4], bv[NB];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[cur][wr * 64 + i * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
            for (int j = 0; j < NB; ++j) bv[j] = Bs[cur][kk + (lane >> 4)][wc * 16 * NB + j * 16 + (lane & 15)];
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                if (j < nbv) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i][j] = mfma4(a[i], bv[j], acc[i][j]);
                }
            }
        }
        if (kt + 1 < nk) store_tiles(cur ^ 1);  // the other stage was last read before the previous barrier
        if (kt + 2 < nk) load_tiles((kt + 2) * kBK);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j >= nbv) continue;
            const int col = wcol0 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = r0 + wr * 64 + i * 16 + acc_row<float>(lane, r);
                if (row < R) X[row * OPAD + col] = acc[i][j][r];
            }
        }
}
template <int VA>
__global__ __launch_bounds__(kWideThreads) void kx_wide_kernel(const float* __restrict__ A, int64_t R, int K,
                                                               const float* __restrict__ Cp, int OPAD,
                                                               float* __restrict__ X, int ncolt) {
    kx_wide_body<VA>(A, R, K, Cp, OPAD, X, ncolt, blockIdx.x, gridDim.x);
}


// ---------------------------------------------------------------------------
// KS (FP32):  Kpart[s][m][n] (+)= sum_{P in split s} sum_{i < width} X[P][m][ioff+i] X[P][n][ioff+i]
// Only lower tiles (mt >= nt) are computed.  grid = nlower * nsplit.
// Each P is accumulated in FP32 and folded into FP64 registers.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ks_kernel_body(const float* __restrict__ X, int N, int OPAD,
                                                       int ioff, int width, int Pc, int nsplit,
                                                       int nlower, double* __restrict__ Kpart,
                                                       int accumulate, int b, int nblocks) {
    constexpr int VA = 4;
    __shared__ float As[2][kTile][kBK + 1];  // two LDS stages
    __shared__ float Bs[2][kTile][kBK + 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int lt = xcd_remap(b, nblocks);
    const int s = lt / nlower;
    int tl = lt % nlower;
    int mt = 0;
    while ((mt + 1) * (mt + 2) / 2 <= tl) ++mt;
    const int nt = tl - mt * (mt + 1) / 2;
    const int m0 = mt * kTile, n0 = nt * kTile;
    const int wr = wid >> 1, wc = wid & 1;
    const int Pa = (int)(((int64_t)Pc * s) / nsplit);
    const int Pb = (int)(((int64_t)Pc * (s + 1)) / nsplit);

    constexpr int LD = (kTile * kBK) / (kGThreads * VA);
    Vec<float, VA> ra[LD], rb[LD];

    auto load_tiles = [&](int P, int i0) {
        const float* XP = X + (int64_t)P * N * OPAD + ioff + i0;
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + kGThreads * q;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
            if (m0 + row < N) {
                ra[q] = load_vec<float, VA>(XP + (int64_t)(m0 + row) * OPAD + kc);
            } else {
#pragma unroll
                for (int v = 0; v < VA; ++v) ra[q].v[v] = 0.0f;
            }
            if (n0 + row < N) {
                rb[q] = load_vec<float, VA>(XP + (int64_t)(n0 + row) * OPAD + kc);
            } else {
#pragma unroll
                for (int v = 0; v < VA; ++v) rb[q].v[v] = 0.0f;
            }
        }
    };
    auto store_tiles = [&](int stg) {
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + kGThreads * q;
            const int row = idx / (kBK / VA), kc = (idx % (kBK / VA)) * VA;
#pragma unroll
            for (int v = 0; v < VA; ++v) {
                As[stg][row][kc + v] = ra[q].v[v];
                Bs[stg][row][kc + v] = rb[q].v[v];
            }
        }
    };

    dx4 acc64[4][4];
    fx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc64[i][j] = dx4{0, 0, 0, 0};
            acc[i][j] = fx4{0, 0, 0, 0};
        }

    const int nkp = width / kBK;  // k steps per P (width % 16 == 0)
    const int nsteps = (Pb - Pa) * nkp;
    auto load_step = [&](int st) { load_tiles(Pa + st / nkp, (st % nkp) * kBK); };
    if (nsteps > 0) {
        load_step(0);
        store_tiles(0);
    }
    __syncthreads();
    if (nsteps > 1) load_step(1);
    for (int st = 0; st < nsteps; ++st) {
        const int cur = st & 1;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 4) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[cur][wr * 64 + i * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[cur][wc * 64 + j * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mfma4(a[i], b[j], acc[i][j]);
        }
        if (st + 1 < nsteps) store_tiles(cur ^ 1);
        if (st + 2 < nsteps) load_step(st + 2);
        __syncthreads();
        if ((st + 1) % nkp == 0) {  // end of one P: fold FP32 partials into FP64
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc64[i][j][r] += (double)acc[i][j][r];
                    acc[i][j] = fx4{0, 0, 0, 0};
                }
        }
    }
    double* Ks = Kpart + (int64_t)s * N * N;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + wc * 64 + j * 16 + (lane & 15);
            if (col >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wr * 64 + i * 16 + acc_row<float>(lane, r);
                if (row >= N) continue;
                double* dst = Ks + (int64_t)row * N + col;
                const double v = acc64[i][j][r];
                *dst = accumulate ? (*dst + v) : v;
            }
        }
}
// two workgroups per CU: 4 waves of one workgroup leave each SIMD idle at the
// k-step barrier and the LDS-read latency
__global__ __launch_bounds__(kGThreads, 2) void ks_kernel(const float* __restrict__ X, int N, int OPAD,
                                                       int ioff, int width, int Pc, int nsplit,
                                                       int nlower, double* __restrict__ Kpart,
                                                       int accumulate) {
    ks_kernel_body(X, N, OPAD, ioff, width, Pc, nsplit, nlower, Kpart, accumulate, blockIdx.x, gridDim.x);
}


// ---------------------------------------------------------------------------
// BF16x3 precision form.  An FP32 value x is carried as the bf16 pair
//   hi = rne_bf16(x),  lo = rne_bf16(x - hi)      (x - hi is exact in FP32)
// which keeps ~16 significant bits; a product is formed from three bf16 MFMAs
//   a*b ~ hi_a*hi_b + hi_a*lo_b + lo_a*hi_b     (lo_a*lo_b ~ 2^-32 relative, dropped)
// with FP32 accumulation.  v_mfma_f32_16x16x32_bf16: lane l supplies
// A[l%16][8*(l/16) + 0..7] and B[8*(l/16) + 0..7][l%16]; accumulator element
// r holds D[4*(l/16) + r][l%16].
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;
// 16-byte staging registers: a native vector (plain loads/stores, no struct copies)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK16 = 32;              // k extent of one LDS stage = one MFMA k step

// LDS rows of the bf16 tiles are 32 elements (64 B) with the 16-byte chunks
// swizzled: chunk c of row r sits at element (c ^ ((r >> 2) & 2)) * 8.  gfx950
// serves a ds_read_b128 in passes of 32 lanes over 128 banks (512 B); a
// fragment read (lanes 0..31 = rows 0..15, chunks 0..1) would hit rows r and
// r + 8 in the same banks with plain 64 B (or 80 B) rows.  With the swizzle
// both those reads and row-ordered 16-byte stores are conflict-free.
__device__ __forceinline__ int swz16(int row, int chunk) { return (chunk ^ ((row >> 2) & 2)) << 3; }

// f(integral_constant<int, I>) for I = B..E-1: loop bodies whose register
// arrays are indexed by compile-time constants before any loop unrolling, so
// that the arrays are split into registers and never placed in memory.
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// A register prefetched in one iteration and consumed in the next is a phi of
// two loads (prologue and loop body); the compiler folds such a phi into one
// load at the loop head, right before the use, which removes the prefetch
// distance.  Passing the prologue's values through an empty asm that claims
// to modify them keeps the phi from being made of loads only (the cost is one
// wait for the prologue loads).
__device__ __forceinline__ void pin(u32x4& v) { asm volatile("" : "+v"(v)); }
template <int VA>
__device__ __forceinline__ void pin(Vec<float, VA>& v) {
#pragma unroll
    for (int i = 0; i < VA; ++i) asm volatile("" : "+v"(v.v[i]));
}

__device__ __forceinline__ fx4 mfma_bf16(bf16x8 a, bf16x8 b, fx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void split_bf16(float x, __bf16& hi, __bf16& lo) {
    hi = (__bf16)x;
    lo = (__bf16)(x - (float)hi);
}

// A double rounded to float and then split.  The asm keeps the compiler from
// merging the two roundings (double -> float -> bf16) into one, which can give
// another hi for a few values: every pad of the coefficients rounds the same way.
__device__ __forceinline__ void split_bf16_from_double(double x, __bf16& hi, __bf16& lo) {
    float f = (float)x;
    asm volatile("" : "+v"(f));
    split_bf16(f, hi, lo);
}

// KX (bf16x3): X[r][c] = sum_k A[r][k] Ct[c][k]
//   A  = FP32 B chunk, R x K row-major, split into hi/lo while staged to LDS
//   Ct = pre-split transposed coefficients, OPAD x KP (KP = K rounded up to 32)
//   X  = hi/lo bf16 pairs, R x OPAD.
// Tile 128 x (32*NBW): one block holds up to 320 occupied columns so that B is
// read from HBM once.  WAVES waves as 2 x (WAVES/2), each 64 rows x NB blocks
// of 16 columns (NB = 4*NBW/WAVES).  With 8 waves (two per SIMD, ~190
// registers each) the tile's staging is shared by twice the waves.
template <int NBW, int VA, int WAVES = 4>
__device__ __forceinline__ void kx_bf16x3_kernel_body(
    const float* __restrict__ A, int64_t R, int K, int KP, const u16* __restrict__ Cth,
    const u16* __restrict__ Ctl, int OPAD, u16* __restrict__ Xh, u16* __restrict__ Xl, int ncolt, int b, int nblocks) {
    constexpr int BN = 32 * NBW;
    constexpr int T = 64 * WAVES;       // threads
    constexpr int WC = WAVES / 2;       // waves across the columns
    constexpr int NB = 2 * NBW / WC;    // 16-column blocks per wave
    static_assert((2 * NBW) % WC == 0 && NB >= 1, "tile must split over the waves");
    // two LDS stages: the MFMAs read one while the next k-step is written to the other
    __shared__ __bf16 Ah[2][kTile][kBK16];
    __shared__ __bf16 Al[2][kTile][kBK16];
    __shared__ __bf16 Bh[2][BN][kBK16];
    __shared__ __bf16 Bl[2][BN][kBK16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int t = xcd_remap(b, nblocks);
    const int64_t r0 = (int64_t)(t / ncolt) * kTile;
    const int c0 = (t % ncolt) * BN;
    const int wr = wid / WC, wc = wid % WC;
    const int wcol0 = c0 + wc * 16 * NB;
    int nbv = (OPAD - wcol0) / 16;
    nbv = nbv < 0 ? 0 : (nbv > NB ? NB : nbv);

    constexpr int A_LD = (kTile * kBK16) / (T * VA);
    // the B tile (hi and lo arrays, BN rows of four 16-byte chunks each) is
    // staged as NB chunks per thread over both arrays (one per MFMA group); a
    // wave's 64 chunks lie in one array
    constexpr int BCH = BN * (kBK16 / 8);
    constexpr int B_LD = 2 * BCH / T;
    static_assert((2 * BCH) % T == 0 && BCH % 64 == 0 && B_LD == NB, "B tile must split evenly");
    Vec<float, VA> ra[A_LD];
    u32x4 rb[B_LD];

    // The loads carry no branches: rows past R (or columns past OPAD) are
    // clamped onto the last valid row and feed only output rows/columns that
    // are never stored; k past K is clamped onto the row's last VA elements,
    // finite values that meet the zero padding of Ct.
    // parts [S0, S1) of the A tile; the MFMA loop stores and reloads it in two halves
    auto load_a = [&](int k0, auto S0, auto S1) {
        static_for<decltype(S0)::value, decltype(S1)::value>([&](auto S) {
            constexpr int s = decltype(S)::value;
            const int idx = tid + T * s;
            const int row = idx / (kBK16 / VA), kc = (idx % (kBK16 / VA)) * VA;
            const int64_t gr = min(r0 + row, R - 1);
            const int gk = min(k0 + kc, K - VA);
            ra[s] = load_vec<float, VA>(A + gr * K + gk);
        });
    };
    auto load_b = [&](auto q, int k0) {
        const int idx = tid + T * q;
        const int lo = idx >= BCH, rem = idx - (lo ? BCH : 0);
        const int row = rem >> 2, kc = (rem & 3) * 8;
        const int64_t o = (int64_t)min(c0 + row, OPAD - 1) * KP + k0 + kc;
        rb[q] = *reinterpret_cast<const u32x4*>((lo ? Ctl : Cth) + o);
    };
    auto store_a = [&](int stg, auto S0, auto S1) {
        static_for<decltype(S0)::value, decltype(S1)::value>([&](auto S) {
            constexpr int s = decltype(S)::value;
            const int idx = tid + T * s;
            const int row = idx / (kBK16 / VA), kc = (idx % (kBK16 / VA)) * VA;
            const int e = swz16(row, kc >> 3) + (kc & 7);
#pragma unroll
            for (int v = 0; v < VA; ++v) split_bf16(ra[s].v[v], Ah[stg][row][e + v], Al[stg][row][e + v]);
        });
    };
    using A0 = std::integral_constant<int, 0>;
    using AH = std::integral_constant<int, (NB > 2 ? A_LD / 2 : A_LD)>;
    using AE = std::integral_constant<int, A_LD>;
    auto store_b = [&](auto q, int stg) {
        const int idx = tid + T * q;
        const int lo = idx >= BCH, rem = idx - (lo ? BCH : 0);
        const int row = rem >> 2, e = swz16(row, rem & 3);
        *reinterpret_cast<u32x4*>(lo ? &Bl[stg][row][e] : &Bh[stg][row][e]) = rb[q];
    };

    fx4 acc[4][NB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nk = KP / kBK16;
    load_a(0, A0{}, AE{});
#pragma unroll
    for (int q = 0; q < B_LD; ++q) load_b(q, 0);
    store_a(0, A0{}, AE{});
#pragma unroll
    for (int q = 0; q < B_LD; ++q) store_b(q, 0);
    __syncthreads();
    {
        const int k1 = (nk > 1 ? 1 : 0) * kBK16;
        load_a(k1, A0{}, AE{});
#pragma unroll
        for (int q = 0; q < B_LD; ++q) load_b(q, k1);
#pragma unroll
        for (int s = 0; s < A_LD; ++s) pin(ra[s]);
#pragma unroll
        for (int q = 0; q < B_LD; ++q) pin(rb[q]);
    }
    const int fr = lane & 15, fc = lane >> 4;  // fragment row / 16-byte chunk of this lane
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1, nxt = cur ^ 1;
        // registers hold step kt+1 (loaded one step ago); they are stored to the
        // other stage and refilled with step kt+2 (a clamped repeat near the end)
        const int kpre = min(kt + 2, nk - 1) * kBK16;
        // fragment reads in the order the first group consumes them (bh, al for
        // the first sweep, then bl, ah), so its first MFMA waits for two reads
        bf16x8 ah[4], al[4], bh[2], bl[2];
        const int rb0 = wc * 16 * NB + fr;
        bh[0] = *reinterpret_cast<const bf16x8*>(&Bh[cur][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = wr * 64 + i * 16 + fr;
            al[i] = *reinterpret_cast<const bf16x8*>(&Al[cur][r][swz16(r, fc)]);
        }
        bl[0] = *reinterpret_cast<const bf16x8*>(&Bl[cur][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = wr * 64 + i * 16 + fr;
            ah[i] = *reinterpret_cast<const bf16x8*>(&Ah[cur][r][swz16(r, fc)]);
        }
        // One group per 16-column block j: the fragments of block j+1 are read
        // while the 12 MFMAs of block j run (three sweeps, so consecutive MFMAs
        // never depend on each other), and the staging work of the next steps
        // sits in fixed groups so that it issues under the MFMAs.  Every block
        // is computed, also those past OPAD (their B rows are clamped copies).
        static_for<0, NB>([&](auto J) {
            constexpr int j = decltype(J)::value;
            if constexpr (j + 1 < NB) {
                const int r = wc * 16 * NB + (j + 1) * 16 + fr;
                bh[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Bh[cur][r][swz16(r, fc)]);
                bl[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Bl[cur][r][swz16(r, fc)]);
            }
            static_for<0, 4>([&](auto I) { acc[I][j] = mfma_bf16(al[I], bh[j & 1], acc[I][j]); });
            static_for<0, 4>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bl[j & 1], acc[I][j]); });
            static_for<0, 4>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bh[j & 1], acc[I][j]); });
            // the other stage was last read before the previous barrier
            if constexpr (j == 0) {
                store_a(nxt, A0{}, AH{});
                load_a(kpre, A0{}, AH{});
            }
            if constexpr (j == 2 && AH::value < A_LD) {
                store_a(nxt, AH{}, AE{});
                load_a(kpre, AH{}, AE{});
            }
            // one B chunk per group
            store_b(std::integral_constant<int, j>{}, nxt);
            load_b(std::integral_constant<int, j>{}, kpre);
            __builtin_amdgcn_sched_barrier(0);
        });
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j >= nbv) continue;
            const int col = wcol0 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = r0 + wr * 64 + i * 16 + 4 * (lane >> 4) + r;
                if (row < R) {
                    __bf16 h, l;
                    split_bf16(acc[i][j][r], h, l);
                    Xh[row * OPAD + col] = __builtin_bit_cast(u16, h);
                    Xl[row * OPAD + col] = __builtin_bit_cast(u16, l);
                }
            }
        }
}
// Waves of at most 5 column blocks need at most 256 registers: two waves per
// SIMD (two 4-wave workgroups per CU, or one 8-wave workgroup).
template <int NBW, int WAVES = 4>
constexpr int kx_bf16_waves_per_eu() { return (WAVES == 8 || NBW <= 5) ? 2 : 1; }

template <int NBW, int VA, int WAVES>
__global__ __launch_bounds__(64 * WAVES, (kx_bf16_waves_per_eu<NBW, WAVES>())) void kx_bf16x3_kernel(
    const float* __restrict__ A, int64_t R, int K, int KP, const u16* __restrict__ Cth,
    const u16* __restrict__ Ctl, int OPAD, u16* __restrict__ Xh, u16* __restrict__ Xl, int ncolt) {
    kx_bf16x3_kernel_body<NBW, VA, WAVES>(A, R, K, KP, Cth, Ctl, OPAD, Xh, Xl, ncolt, blockIdx.x, gridDim.x);
}


// ---------------------------------------------------------------------------
// KX (bf16x3), tall tiles: the same product as kx_bf16x3_kernel with 256-row
// tiles, so that each staged coefficient tile feeds twice the rows (the
// coefficient tile, 2.5x the bytes of a 128-row A tile at 320 columns, is
// what the 128-row kernel spends most of its staging on).  Per k-step:
//   * A (FP32 rows of B) is loaded into registers one step ahead, split into
//     bf16 hi/lo and stored to the next LDS stage at the start of the step;
//   * the pre-split coefficient tile (hi and lo planes) goes from global
//     memory straight into the next LDS stage (global_load_lds_dwordx4, no
//     registers): a wave's instruction fills 1 KB = 16 swizzled 64-byte rows,
//     lane l writing slot l, so lane l fetches the logical chunk that the
//     swizzle puts in slot l (the XOR swizzle is its own inverse);
//   * the MFMAs of the current stage run under both.
// The direct-to-LDS loads are issued from inline asm: the compiler does not
// track them, so it never waits for them before unrelated LDS reads (its own
// tracking waits for every pending one before any LDS read).  The kernel
// waits for them itself, with vmcnt(0) at the end of each step (the register
// loads of A are waited for too: a direct-to-LDS load need not complete in
// order with register loads, so no partial count is relied on); the barrier
// then publishes them.  Both kinds of load are issued at the start of the
// step, a full step ahead of their use.
// WR x WC waves; each wave holds a (256/WR) x (32*NBW/WC) block of the tile.
// ---------------------------------------------------------------------------
constexpr int kTallRows = 256;

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes per lane from global memory (wave-uniform base + per-lane 32-bit
// byte offset) into LDS at m0 + 16 * lane
__device__ __forceinline__ void lds_load16(const void* base, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
// Every global load (direct-to-LDS ones included) and LDS access of this wave
// has completed, then the workgroup barrier.  One asm statement with a memory
// clobber: the compiler moves no memory access across it.
__device__ __forceinline__ void drain_and_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// every global load of this wave has completed
__device__ __forceinline__ void drain_vm() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int NBW, int WR, int WC>
__device__ __forceinline__ void kx_bf16x3_tall_body(
    const float* __restrict__ A, int64_t R, int K, int KP, const u16* __restrict__ Cth,
    const u16* __restrict__ Ctl, int OPAD, u16* __restrict__ Xh, u16* __restrict__ Xl, int ncolt, int b,
    int nblocks) {
    constexpr int TM = kTallRows;
    constexpr int BN = 32 * NBW;
    constexpr int NW = WR * WC;
    constexpr int T = 64 * NW;
    constexpr int IB = TM / WR / 16;     // 16-row blocks per wave
    constexpr int NB = BN / WC / 16;     // 16-column blocks per wave
    static_assert(TM % (16 * WR) == 0 && BN % (16 * WC) == 0 && NB >= 1, "tile must split over the waves");
    // A: TM x 32 FP32 = TM*8 16-byte chunks, VA = 4 elements per chunk
    constexpr int A_LD = TM * 8 / T;
    static_assert(A_LD * T == TM * 8 && A_LD <= 15, "A tile must split evenly");
    // coefficient tile: 2 planes x BN rows x 4 chunks, in wave instructions of 16 rows
    constexpr int B_INS = 2 * BN / 16;
    constexpr int B_LD = (B_INS + NW - 1) / NW;
    __shared__ __attribute__((aligned(16))) __bf16 Ah[2][TM][kBK16];
    __shared__ __attribute__((aligned(16))) __bf16 Al[2][TM][kBK16];
    __shared__ __attribute__((aligned(16))) __bf16 Bt[2][2][BN][kBK16];  // [stage][hi, lo][row][k]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = xcd_remap(b, nblocks);
    const int64_t r0 = (int64_t)(t / ncolt) * TM;
    const int c0 = (t % ncolt) * BN;
    const int wr = wid / WC, wc = wid % WC;
    const int wcol0 = c0 + wc * 16 * NB;
    int nbv = (OPAD - wcol0) / 16;
    nbv = nbv < 0 ? 0 : (nbv > NB ? NB : nbv);

    Vec<float, 4> ra[A_LD];
    // Rows past R are clamped onto the last row (their outputs are never
    // stored); k past K is clamped onto the row's last 4 elements, finite
    // values that meet the zero padding of Ct.  The tile's base is
    // wave-uniform; each load adds a loop-invariant 32-bit row offset.
    const float* Atile = A + r0 * K;
    uint32_t aoff[A_LD];
    static_for<0, A_LD>([&](auto S) {
        constexpr int s = decltype(S)::value;
        const int row = (tid + T * s) >> 3;
        aoff[s] = (uint32_t)((min(r0 + row, R - 1) - r0) * K);
    });
    auto load_a = [&](int k0) {
        static_for<0, A_LD>([&](auto S) {
            constexpr int s = decltype(S)::value;
            const int kc = ((tid + T * s) & 7) * 4;
            ra[s] = load_vec<float, 4>(Atile + aoff[s] + min(k0 + kc, K - 4));
        });
    };
    auto store_a = [&](int stg) {
        static_for<0, A_LD>([&](auto S) {
            constexpr int s = decltype(S)::value;
            const int idx = tid + T * s;
            const int row = idx >> 3, kc = (idx & 7) * 4;
            const int e = swz16(row, kc >> 3) + (kc & 7);
#pragma unroll
            for (int v = 0; v < 4; ++v) split_bf16(ra[s].v[v], Ah[stg][row][e + v], Al[stg][row][e + v]);
        });
    };
    // This wave's direct-to-LDS loads of the coefficient tile of step k0.
    // Ct has ncolt * BN rows (zero past OPAD), so no row is clamped: a load's
    // address is a wave-uniform base (plane, 16-row group, k0) plus the
    // lane's offset, the same for every load (the swizzle of row 16g + lrow
    // depends on lrow only).
    const int lrow = lane >> 2, lpos = lane & 3;
    const uint32_t boff = (uint32_t)(lrow * KP + (lpos ^ ((lrow >> 2) & 2)) * 8) * 2;
    auto load_b = [&](int k0, int stg) {
        static_for<0, B_LD>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const int g = wid + NW * q;                // wave instruction index (wave-uniform)
            if (B_INS % NW == 0 || g < B_INS) {
                const int plane = g / (BN / 16), grp = g % (BN / 16);
                const u16* base = (plane ? Ctl : Cth) + (int64_t)(c0 + grp * 16) * KP + k0;
                lds_load16(base, boff, __builtin_amdgcn_readfirstlane(lds_addr(&Bt[stg][plane][grp * 16][0])));
            }
        });
    };

    fx4 acc[IB][NB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nk = KP / kBK16;
    load_a(0);
    store_a(0);
    load_b(0, 0);
    load_a((nk > 1 ? 1 : 0) * kBK16);
    drain_and_barrier();

    const int fr = lane & 15, fc = lane >> 4;
    const int ra0 = wr * (TM / WR), rb0 = wc * 16 * NB;
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1, nxt = cur ^ 1;
        const int k1 = min(kt + 1, nk - 1) * kBK16;  // clamped: the last steps repeat harmless loads
        const int k2 = min(kt + 2, nk - 1) * kBK16;
        bf16x8 bh[NB], bl[NB], ah[2], al[2];
        // row block 0 streams the column fragments in; later row blocks reuse them
        {
            const int r = ra0 + fr;
            al[0] = *reinterpret_cast<const bf16x8*>(&Al[cur][r][swz16(r, fc)]);
            ah[0] = *reinterpret_cast<const bf16x8*>(&Ah[cur][r][swz16(r, fc)]);
        }
        static_for<0, NB>([&](auto J) {
            constexpr int j = decltype(J)::value;
            const int r = rb0 + j * 16 + fr;
            bh[j] = *reinterpret_cast<const bf16x8*>(&Bt[cur][0][r][swz16(r, fc)]);
            bl[j] = *reinterpret_cast<const bf16x8*>(&Bt[cur][1][r][swz16(r, fc)]);
        });
        static_for<0, IB>([&](auto I) {
            constexpr int i = decltype(I)::value;
            if constexpr (i + 1 < IB) {
                const int r = ra0 + (i + 1) * 16 + fr;
                al[(i + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Al[cur][r][swz16(r, fc)]);
                ah[(i + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Ah[cur][r][swz16(r, fc)]);
            }
            // three sweeps over the column blocks: consecutive MFMAs never share an accumulator
            static_for<0, NB>([&](auto J) { acc[i][J] = mfma_bf16(al[i & 1], bh[J], acc[i][J]); });
            static_for<0, NB>([&](auto J) { acc[i][J] = mfma_bf16(ah[i & 1], bl[J], acc[i][J]); });
            static_for<0, NB>([&](auto J) { acc[i][J] = mfma_bf16(ah[i & 1], bh[J], acc[i][J]); });
            // staging of the next steps, under the MFMAs of row block 0: the
            // split of A(kt+1) (loaded in the previous step), the register
            // loads of A(kt+2), the LDS loads of Ct(kt+1)
            if constexpr (i == 0) {
                store_a(nxt);
                load_a(k2);
                load_b(k1, nxt);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        // every load and LDS store of this wave has landed, then publish
        drain_and_barrier();
    }
    // no direct-to-LDS load may outlive the workgroup
    drain_vm();
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (j >= nbv) continue;
            const int col = wcol0 + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = r0 + ra0 + i * 16 + 4 * (lane >> 4) + r;
                if (row < R) {
                    __bf16 h, l;
                    split_bf16(acc[i][j][r], h, l);
                    Xh[row * OPAD + col] = __builtin_bit_cast(u16, h);
                    Xl[row * OPAD + col] = __builtin_bit_cast(u16, l);
                }
            }
        }
}

template <int NBW, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, (WR * WC == 8 ? 2 : 1)) void kx_bf16x3_tall_kernel(
    const float* __restrict__ A, int64_t R, int K, int KP, const u16* __restrict__ Cth,
    const u16* __restrict__ Ctl, int OPAD, u16* __restrict__ Xh, u16* __restrict__ Xl, int ncolt) {
    kx_bf16x3_tall_body<NBW, WR, WC>(A, R, K, KP, Cth, Ctl, OPAD, Xh, Xl, ncolt, blockIdx.x, gridDim.x);
}

// KS (bf16x3): Kpart[s][m][n] (+)= sum_{P in split s} sum_{i < width} X[P][m][ioff+i] X[P][n][ioff+i]
// with X given as hi/lo bf16 pairs; width % 32 == 0.  FP32 accumulation over
// the P range of a split (the MFMA rounds once per 32 products), FP64 across
// splits.  Lower TS x TS tiles; WR x WC waves, each holding a (TS/WR) x
// (TS/WC) block of the tile.  TS = 128 with 2 x 2 waves fits two workgroups
// per CU (no FP64 registers); TS = 256 with 4 x 2 waves is one 8-wave
// workgroup per CU that reads half the LDS bytes per MFMA (each fragment
// feeds more blocks), for large nbf.  The split length (target_blocks) sets
// the length of the FP32 sums.
template <int TS, int WR, int WC>
__device__ __forceinline__ void ks_bf16x3_kernel_body(
    const u16* __restrict__ Xh, const u16* __restrict__ Xl, int N, int OPAD, int ioff, int width,
    int Pc, int nsplit, int nlower, double* __restrict__ Kpart, int accumulate, int b, int nblocks) {
    constexpr int T = 64 * WR * WC;        // threads
    constexpr int IB = TS / WR / 16;       // 16-row blocks per wave
    constexpr int JB = TS / WC / 16;       // 16-column blocks per wave
    static_assert(JB >= 2, "staging is spread over the first two column blocks");
    __shared__ __bf16 Ah[2][TS][kBK16];
    __shared__ __bf16 Al[2][TS][kBK16];
    __shared__ __bf16 Bh[2][TS][kBK16];
    __shared__ __bf16 Bl[2][TS][kBK16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int lt = xcd_remap(b, nblocks);
    const int s = lt / nlower;
    const int tl = lt % nlower;
    int mt = 0;
    while ((mt + 1) * (mt + 2) / 2 <= tl) ++mt;
    const int nt = tl - mt * (mt + 1) / 2;
    const int m0 = mt * TS, n0 = nt * TS;
    const int wr = wid / WC, wc = wid % WC;
    const int Pa = (int)(((int64_t)Pc * s) / nsplit);
    const int Pb = (int)(((int64_t)Pc * (s + 1)) / nsplit);

    constexpr int LD = (TS * kBK16 / 8) / T;  // 16-byte loads per array (= 2)
    static_assert(LD * T * 8 == TS * kBK16, "tile rows must split evenly over the threads");
    u32x4 rah[LD], ral[LD], rbh[LD], rbl[LD];

    // Branch-free loads: rows past N are clamped onto row N-1 and feed only
    // rows/columns of the tile that are never stored.
    auto load_a = [&](int P, int i0) {
        const int64_t base = (int64_t)P * N * OPAD + ioff + i0;
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + T * q;
            const int row = idx >> 2, kc = (idx & 3) * 8;
            const int64_t o = base + (int64_t)min(m0 + row, N - 1) * OPAD + kc;
            rah[q] = *reinterpret_cast<const u32x4*>(Xh + o);
            ral[q] = *reinterpret_cast<const u32x4*>(Xl + o);
        }
    };
    auto load_b = [&](int P, int i0) {
        const int64_t base = (int64_t)P * N * OPAD + ioff + i0;
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + T * q;
            const int row = idx >> 2, kc = (idx & 3) * 8;
            const int64_t o = base + (int64_t)min(n0 + row, N - 1) * OPAD + kc;
            rbh[q] = *reinterpret_cast<const u32x4*>(Xh + o);
            rbl[q] = *reinterpret_cast<const u32x4*>(Xl + o);
        }
    };
    auto store_a = [&](int stg) {
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + T * q;
            const int row = idx >> 2, e = swz16(row, idx & 3);
            *reinterpret_cast<u32x4*>(&Ah[stg][row][e]) = rah[q];
            *reinterpret_cast<u32x4*>(&Al[stg][row][e]) = ral[q];
        }
    };
    auto store_b = [&](int stg) {
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            const int idx = tid + T * q;
            const int row = idx >> 2, e = swz16(row, idx & 3);
            *reinterpret_cast<u32x4*>(&Bh[stg][row][e]) = rbh[q];
            *reinterpret_cast<u32x4*>(&Bl[stg][row][e]) = rbl[q];
        }
    };

    fx4 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nkp = width / kBK16;
    // steps are numbered across P; step st+1's tiles are written to the other
    // LDS stage while the MFMAs of step st run, and step st+2 is loaded
    const int nsteps = (Pb - Pa) * nkp;
    if (nsteps > 0) {
        load_a(Pa, 0);
        load_b(Pa, 0);
        store_a(0);
        store_b(0);
        const int s1 = nsteps > 1 ? 1 : 0;
        load_a(Pa + s1 / nkp, (s1 % nkp) * kBK16);
        load_b(Pa + s1 / nkp, (s1 % nkp) * kBK16);
#pragma unroll
        for (int q = 0; q < LD; ++q) {
            pin(rah[q]);
            pin(ral[q]);
            pin(rbh[q]);
            pin(rbl[q]);
        }
    }
    __syncthreads();
    const int fr = lane & 15, fc = lane >> 4;  // fragment row / 16-byte chunk of this lane
    const int ra0 = wr * (TS / WR), rb0w = wc * (TS / WC);
    int st = 0;
    for (int P = Pa; P < Pb; ++P) {
    for (int kt = 0; kt < nkp; ++kt, ++st) {
        const int cur = st & 1, nxt = cur ^ 1;
        const int sp = min(st + 2, nsteps - 1);  // clamped prefetch: the last loads are harmless repeats
        const int Ppre = Pa + sp / nkp, ipre = (sp % nkp) * kBK16;
        // fragment reads in the order the first group consumes them
        bf16x8 ah[IB], al[IB], bh[2], bl[2];
        const int rb0 = rb0w + fr;
        bh[0] = *reinterpret_cast<const bf16x8*>(&Bh[cur][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            const int r = ra0 + i * 16 + fr;
            al[i] = *reinterpret_cast<const bf16x8*>(&Al[cur][r][swz16(r, fc)]);
        }
        bl[0] = *reinterpret_cast<const bf16x8*>(&Bl[cur][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            const int r = ra0 + i * 16 + fr;
            ah[i] = *reinterpret_cast<const bf16x8*>(&Ah[cur][r][swz16(r, fc)]);
        }
        // one group per 16-column block j (as in the half-transform): block
        // j+1's fragments are read and one staging task is issued under the
        // 3 * IB MFMAs of block j
        static_for<0, JB>([&](auto J) {
            constexpr int j = decltype(J)::value;
            if constexpr (j + 1 < JB) {
                const int r = rb0w + (j + 1) * 16 + fr;
                bh[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Bh[cur][r][swz16(r, fc)]);
                bl[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Bl[cur][r][swz16(r, fc)]);
            }
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(al[I], bh[j & 1], acc[I][j]); });
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bl[j & 1], acc[I][j]); });
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bh[j & 1], acc[I][j]); });
            if constexpr (j == 0) {
                store_a(nxt);
                load_a(Ppre, ipre);
            }
            if constexpr (j == 1) {
                store_b(nxt);
                load_b(Ppre, ipre);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        __syncthreads();
    }
    }
    double* Ks = Kpart + (int64_t)s * N * N;
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int col = n0 + rb0w + j * 16 + (lane & 15);
            if (col >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + ra0 + i * 16 + 4 * (lane >> 4) + r;
                if (row >= N) continue;
                double* dst = Ks + (int64_t)row * N + col;
                const double v = (double)acc[i][j][r];
                *dst = accumulate ? (*dst + v) : v;
            }
        }
}
template <int TS, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, (TS == 128 ? 2 : 1)) void ks_bf16x3_kernel(
    const u16* __restrict__ Xh, const u16* __restrict__ Xl, int N, int OPAD, int ioff, int width,
    int Pc, int nsplit, int nlower, double* __restrict__ Kpart, int accumulate) {
    ks_bf16x3_kernel_body<TS, WR, WC>(Xh, Xl, N, OPAD, ioff, width, Pc, nsplit, nlower, Kpart, accumulate,
                                      blockIdx.x, gridDim.x);
}


// KS (bf16x3) with the tiles of X brought into LDS by direct-to-LDS loads:
// the same product, tiles, split ranges and MFMA sequence as
// ks_bf16x3_kernel (so the same Kpart, bitwise), without staging registers
// or LDS stores.  Each step issues the loads of the next step into the other
// stage right after the barrier and waits for them (vmcnt 0: no other global
// loads are in flight in the loop) at the end of the step.  A wave
// instruction fills 16 swizzled 64-byte rows of one plane (A hi, A lo, B hi,
// B lo); rows past N are clamped onto row N-1 (per lane, loop-invariant).
template <int TS, int WR, int WC>
__device__ __forceinline__ void ks_bf16x3_dma_body(
    const u16* __restrict__ Xh, const u16* __restrict__ Xl, int N, int OPAD, int ioff, int width,
    int Pc, int nsplit, int nlower, double* __restrict__ Kpart, int accumulate, int b, int nblocks) {
    constexpr int NW = WR * WC;
    constexpr int IB = TS / WR / 16;
    constexpr int JB = TS / WC / 16;
    constexpr int INS = 4 * TS / 16;   // wave instructions per step: 4 planes x TS/16 row groups
    constexpr int LD = INS / NW;
    static_assert(LD * NW == INS && JB >= 2, "tile must split over the waves");
    __shared__ __attribute__((aligned(16))) __bf16 Xt[2][4][TS][kBK16];  // [stage][Ah, Al, Bh, Bl][row][k]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lt = xcd_remap(b, nblocks);
    const int s = lt / nlower;
    const int tl = lt % nlower;
    int mt = 0;
    while ((mt + 1) * (mt + 2) / 2 <= tl) ++mt;
    const int nt = tl - mt * (mt + 1) / 2;
    const int m0 = mt * TS, n0 = nt * TS;
    const int wr = wid / WC, wc = wid % WC;
    const int Pa = (int)(((int64_t)Pc * s) / nsplit);
    const int Pb = (int)(((int64_t)Pc * (s + 1)) / nsplit);

    // per load q: wave-uniform row of its 16-row group (clamped) and the
    // lane's 32-bit byte offset from it (clamped row, swizzled chunk)
    const int lrow = lane >> 2, lpos = lane & 3;
    const int lchunk = lpos ^ ((lrow >> 2) & 2);
    int qrow[LD];
    uint32_t qoff[LD];
    static_for<0, LD>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        const int g = wid + NW * q;
        const int plane = g / (TS / 16), grp = g % (TS / 16);
        const int r0 = (plane < 2 ? m0 : n0) + grp * 16;
        const int rb = min(r0, N - 1);
        qrow[q] = rb;
        qoff[q] = (uint32_t)(((min(r0 + lrow, N - 1) - rb) * OPAD + lchunk * 8) * 2);
    });
    auto load = [&](int P, int i0, int stg) {
        static_for<0, LD>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const int g = wid + NW * q;
            const int plane = g / (TS / 16), grp = g % (TS / 16);
            const u16* base = ((plane & 1) ? Xl : Xh) + ((int64_t)P * N + qrow[q]) * OPAD + ioff + i0;
            lds_load16(base, qoff[q], lds_addr(&Xt[stg][plane][grp * 16][0]));
        });
    };

    fx4 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[i][j] = fx4{0, 0, 0, 0};

    const int nkp = width / kBK16;
    const int nsteps = (Pb - Pa) * nkp;
    if (nsteps > 0) load(Pa, 0, 0);
    drain_and_barrier();
    const int fr = lane & 15, fc = lane >> 4;
    const int ra0 = wr * (TS / WR), rb0w = wc * (TS / WC);
    // a wave whose block lies above the diagonal or past row N loads its share
    // and multiplies nothing
    const bool active = m0 + ra0 < N && n0 + rb0w <= m0 + ra0 + TS / WR - 1;
    int st = 0;
    for (int P = Pa; P < Pb; ++P) {
    for (int kt = 0; kt < nkp; ++kt, ++st) {
        const int cur = st & 1, nxt = cur ^ 1;
        const int sp = min(st + 1, nsteps - 1);  // clamped: the last loads are harmless repeats
        load(Pa + sp / nkp, (sp % nkp) * kBK16, nxt);
        if (active) {
        bf16x8 ah[IB], al[IB], bh[2], bl[2];
        const int rb0 = rb0w + fr;
        bh[0] = *reinterpret_cast<const bf16x8*>(&Xt[cur][2][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            const int r = ra0 + i * 16 + fr;
            al[i] = *reinterpret_cast<const bf16x8*>(&Xt[cur][1][r][swz16(r, fc)]);
        }
        bl[0] = *reinterpret_cast<const bf16x8*>(&Xt[cur][3][rb0][swz16(rb0, fc)]);
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            const int r = ra0 + i * 16 + fr;
            ah[i] = *reinterpret_cast<const bf16x8*>(&Xt[cur][0][r][swz16(r, fc)]);
        }
        static_for<0, JB>([&](auto J) {
            constexpr int j = decltype(J)::value;
            if constexpr (j + 1 < JB) {
                const int r = rb0w + (j + 1) * 16 + fr;
                bh[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Xt[cur][2][r][swz16(r, fc)]);
                bl[(j + 1) & 1] = *reinterpret_cast<const bf16x8*>(&Xt[cur][3][r][swz16(r, fc)]);
            }
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(al[I], bh[j & 1], acc[I][j]); });
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bl[j & 1], acc[I][j]); });
            static_for<0, IB>([&](auto I) { acc[I][j] = mfma_bf16(ah[I], bh[j & 1], acc[I][j]); });
            __builtin_amdgcn_sched_barrier(0);
        });
        }
        drain_and_barrier();
    }
    }
    if (!active) return;
    double* Ks = Kpart + (int64_t)s * N * N;
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int col = n0 + rb0w + j * 16 + (lane & 15);
            if (col >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + ra0 + i * 16 + 4 * (lane >> 4) + r;
                if (row >= N) continue;
                double* dst = Ks + (int64_t)row * N + col;
                const double v = (double)acc[i][j][r];
                *dst = accumulate ? (*dst + v) : v;
            }
        }
}
template <int TS, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC, (TS == 128 ? 2 : 1)) void ks_bf16x3_dma_kernel(
    const u16* __restrict__ Xh, const u16* __restrict__ Xl, int N, int OPAD, int ioff, int width,
    int Pc, int nsplit, int nlower, double* __restrict__ Kpart, int accumulate) {
    ks_bf16x3_dma_body<TS, WR, WC>(Xh, Xl, N, OPAD, ioff, width, Pc, nsplit, nlower, Kpart, accumulate,
                                   blockIdx.x, gridDim.x);
}

// K[m][n] = K[n][m] = sum_s Kpart[s][m][n] for m >= n (fixed order in s).  A
// block holds 4 rows x 16 columns; its four waves sum every fourth split each
// and are added in order (one thread per element took 30-60 us below nbf 400,
// a serial chain over the splits).
__device__ __forceinline__ void k_reduce_body(const double* __restrict__ Kpart, int nsplit, int N,
                                              double* __restrict__ K, int m4, int n16) {
    __shared__ double red[3][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m = m4 * 4 + (lane >> 4), n = n16 * 16 + (lane & 15);
    const bool on = m < N && n <= m;
    const int64_t NN = (int64_t)N * N;
    double s = 0.0;
    if (on) {
        const double* p = Kpart + (int64_t)m * N + n;
#pragma unroll 8
        for (int c = w; c < nsplit; c += 4) s += p[c * NN];
    }
    if (w > 0) red[w - 1][lane] = s;
    __syncthreads();
    if (w == 0 && on) {
        s = ((s + red[0][lane]) + red[1][lane]) + red[2][lane];
        K[(int64_t)m * N + n] = s;
        K[(int64_t)n * N + m] = s;
    }
    __syncthreads();
}
// blocks of the reduction of one N x N matrix (n16 past the diagonal: nothing to do)
__host__ __device__ inline int k_reduce_blocks(int N) { return ((N + 3) / 4) * ((N + 15) / 16); }
// the K (or D) of every density of a call
struct KPtrs {
    double* p[8];
};
// grid (16-column blocks, 4-row blocks, densities); the partials of one density are dstride doubles
__global__ __launch_bounds__(256) void k_reduce_kernel(const double* __restrict__ Kpart, int64_t dstride, int nsplit,
                                                       int N, KPtrs K) {
    const int m4 = blockIdx.y, n16 = blockIdx.x;
    if (n16 * 16 > m4 * 4 + 3) return;
    k_reduce_body(Kpart + blockIdx.z * dstride, nsplit, N, K.p[blockIdx.z], m4, n16);
}

}  // namespace f2jk
