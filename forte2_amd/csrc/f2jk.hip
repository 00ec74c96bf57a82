// C ABI of the MI355X density-fitted J/K builder.  Declarations and the
// reference functions each entry point replaces are in include/f2jk.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "f2jk.h"
#include "f2jk_kernels.h"
#include "f2jk_fp64.h"
#include "f2jk_group.h"

using namespace f2jk;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

#define F2JK_HIP(call)                                                                   \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess)                                                            \
            return fail(F2JK_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define F2JK_LAUNCHED(what)                                                             \
    do {                                                                                \
        hipError_t e_ = hipGetLastError();                                              \
        if (e_ != hipSuccess)                                                           \
            return fail(F2JK_EHIP, std::string("launch ") + what + ": " +               \
                                       hipGetErrorString(e_));                         \
    } while (0)

constexpr int kMaxDens = 8;
constexpr int kMaxEvents = 512;
constexpr int kEPT = 4;                 // vector elements per thread in the J kernels
constexpr int kJ1PerBlock = 32;         // P values per block in J pass 1
constexpr int kTargetBlocks = 2048;     // blocks wanted per launch to fill 256 CUs
constexpr size_t kDefaultXChunkBytes = size_t(4) << 30;
// The threads of a launch are counted in 32 bits per dimension, and one more
// wraps around without an error.  The FP64 half-transform has four threads per
// row (wider rows than one column tile's fit no card at this count), the sum of
// its row sums a wave per P.
constexpr int64_t kMaxLaunchRows = int64_t(1) << 29;
constexpr int64_t kMaxLaunchP = int64_t(1) << 25;

size_t align_up(size_t x, size_t a = 256) { return (x + a - 1) / a * a; }
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace

struct f2jk_ctx {
    int device = 0;
    const void* B[2] = {nullptr, nullptr};
    int64_t naux = 0, nbf = 0;
    int* rowoff[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};  // by VEC (1, 2, 4)
    int nvec[5] = {0, 0, 0, 0, 0};
    // J over the nonzero vector elements only ("j_sparse"): per B copy (dtype)
    // the list of lower-triangle vector elements (of that copy's J width)
    // where B is nonzero for some P
    bool j_sparse = false;
    uint32_t* jlist[2] = {nullptr, nullptr};
    int* jinv[2] = {nullptr, nullptr};   // lower-triangle element -> place in the list, or -1
    // the listed elements of the FP32 copy one after the other (P-major), when asked
    // for ("j_pack") and there is room: the J passes then read whole lines
    bool j_pack = false;
    void* jpacked = nullptr;
    int jlist_vec[2] = {0, 0};
    int jlist_n[2] = {0, 0};
    size_t xchunk_bytes = kDefaultXChunkBytes;
    bool j_nontemporal = true;
    int bf16_nbw_max = 10;          // widest BF16x3 half-transform tile: 32 * 10 columns
    // J (HBM-bound) runs on a side stream concurrently with K (MFMA-bound): 0, 1,
    // -1 = FP64 builds whose J pass is long enough
    int overlap_jk = -1;
    int kx_waves = 8;               // waves per BF16x3 half-transform workgroup (4 or 8)
    int ks_tile = 0;                // BF16x3 contraction tile edge: 128, 256, 0 = by nbf
    int kx_rows = 0;                // BF16x3 half-transform tile rows: 128, 256, 0 = by nbf
    int ks_dma = -1;                // BF16x3 contraction tiles by direct-to-LDS loads: 0, 1, -1 = with 256 tiles
    int kx_wide = -1;               // FP32 half-transform in 320-column tiles: 0, 1, -1 = above 128 columns
    hipStream_t side = nullptr;     // default priority, created with the context
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    std::mutex ev_mu;               // an event is recorded and waited on in one piece
    int target_blocks = kTargetBlocks;
    // timing
    hipEvent_t ev[kMaxEvents];      // (start, end) pairs of non-nested phases
    int ev_phase[kMaxEvents / 2];
    int nev = 0;
    hipEvent_t ev_total[2];         // the whole build
    bool total_recorded = false;
    bool timing = false;
};

namespace {

// ---------------------------------------------------------------------------
// Launch plan and workspace layout of one build.
// ---------------------------------------------------------------------------
struct Plan {
    int N = 0, Q = 0, nd = 0;
    bool want_j = false, want_k = false, need_c = false;
    int prec = 0;
    size_t tk = 8;             // bytes of a K-path element (8 fp64, 4 fp32)
    // C packing (K and the D of build_jk)
    int OPAD = 0;
    int width[kMaxDens] = {}, ioff[kMaxDens] = {};
    // J
    int jvec = 1, nvec = 0, neg = 0, npc1 = 0, ppw2 = 0, npc2 = 0;
    const uint32_t* jlist = nullptr;  // element list of the J passes (null: every element)
    const int* jinv = nullptr;        // element -> place in that list
    const void* jpacked = nullptr;    // the listed elements, packed
    int jdense = 0;                   // lower-triangle elements in all
    size_t jb = 8;             // bytes of a B element read by J
    // K
    int Pc = 0, nchunks = 0, ntile = 0, nlower = 0, nsplit = 0, ncolt = 0, kva = 1, nbw = 0, kx_waves = 4;
    int ks_tile = 128;  // edge of the contraction's lower tiles (256: BF16x3 8-wave tiles)
    int kx_rows = 128;  // rows of a BF16x3 half-transform tile (256: the tall kernel)
    bool kx_wide = false;  // FP32 half-transform in 320-column tiles (kx_wide_kernel)
    int dnb = 0, dncolt = 0, dnks = 0;  // FP64 half-transform: column blocks of a tile, tiles, 16-k steps
    size_t per_p = 0;      // bytes of X per P
    DTiles dt{};           // FP64 contraction: tiles and their P splits
    bool gamma_x = false;  // gamma of J from the half-transform's row sums (FP64 J and K from C)
    bool small = false;    // ... by the blocks of the second J pass, and both reductions in one launch
    int ctrows = 0;     // rows of the padded bf16 coefficient planes (>= ncolt * tile columns)
    // workspace offsets
    int KP = 0;                // nbf rounded up to the bf16 k step
    size_t off_cp32 = 0, off_cth = 0, off_ctl = 0, off_cq = 0;
    size_t off_grow = 0;
    size_t off_cp = 0, off_d = 0, off_gpart = 0, off_gamma = 0, off_jpart = 0,
           off_x = 0, off_kpart = 0, total = 0;
    // sizes of the regions that scale with the launch-shape knobs
    size_t jpart_bytes = 0, x_bytes = 0, kpart_bytes = 0;
    // the workspace is the library's scratch array: the build may not allocate
    bool no_alloc = false;
};

int j_vec_for(int dtype, int64_t N) {
    if (dtype == F2JK_F64) return (N % 2 == 0) ? 2 : 1;
    return (N % 4 == 0) ? 4 : ((N % 2 == 0) ? 2 : 1);
}

int ensure_rowoff(f2jk_ctx* ctx, int vec) {
    if (ctx->rowoff[vec]) return F2JK_OK;
    const int64_t N = ctx->nbf;
    std::vector<int> h(N + 1);
    int64_t acc = 0;
    for (int64_t m = 0; m < N; ++m) {
        h[m] = (int)acc;
        acc += (m + 1 + vec - 1) / vec;
    }
    h[N] = (int)acc;
    if (acc > (int64_t)INT32_MAX) return fail(F2JK_EUNSUPPORTED, "nbf too large for J element tables");
    F2JK_HIP(hipSetDevice(ctx->device));
    F2JK_HIP(hipMalloc(&ctx->rowoff[vec], sizeof(int) * (N + 1)));
    F2JK_HIP(hipMemcpy(ctx->rowoff[vec], h.data(), sizeof(int) * (N + 1), hipMemcpyHostToDevice));
    ctx->nvec[vec] = (int)acc;
    return F2JK_OK;
}

// The J element list of B copy `dtype` (see f2jk_ctx::jlist): the device
// flags the lower-triangle vector elements where B is nonzero for some P (one
// pass over the lower triangle), the host compacts them.  Set-up work: it
// synchronises the device.
template <typename TB, int VEC>
int scan_jlist(f2jk_ctx* ctx, const TB* B, unsigned char* flag) {
    const int nvec = ctx->nvec[VEC];
    hipLaunchKernelGGL(fill_bytes_kernel, dim3((unsigned)cdiv(nvec, 256)), dim3(256), 0, nullptr, flag, nvec);
    F2JK_LAUNCHED("fill_bytes");
    const unsigned ny = (unsigned)std::max<int64_t>(1, std::min<int64_t>(64, ctx->naux / 32));
    hipLaunchKernelGGL((j_scan_kernel<TB, VEC>), dim3((unsigned)cdiv(nvec, 256), ny), dim3(256), 0, nullptr, B,
                       (int)ctx->nbf, (int)ctx->naux, ctx->rowoff[VEC], nvec, flag);
    F2JK_LAUNCHED("j_scan");
    return F2JK_OK;
}

template <int VEC>
int pack_jlist(f2jk_ctx* ctx) {
    const int n = ctx->jlist_n[F2JK_F32];
    const unsigned ny = (unsigned)std::max<int64_t>(1, std::min<int64_t>(ctx->naux, 128));
    hipLaunchKernelGGL((j_pack_kernel<float, VEC>), dim3((unsigned)cdiv(n, 256), ny), dim3(256), 0, nullptr,
                       (const float*)ctx->B[F2JK_F32], (int)ctx->nbf, (int)ctx->naux, ctx->jlist[F2JK_F32], n,
                       (float*)ctx->jpacked);
    F2JK_LAUNCHED("j_pack");
    return F2JK_OK;
}

// the values of the FP32 copy into its packed elements
int pack_elements(f2jk_ctx* ctx) {
    const int vec = ctx->jlist_vec[F2JK_F32];
    const int rc = vec == 4 ? pack_jlist<4>(ctx) : vec == 2 ? pack_jlist<2>(ctx) : pack_jlist<1>(ctx);
    if (rc) return rc;
    F2JK_HIP(hipStreamSynchronize(nullptr));  // builds on any stream read it
    return F2JK_OK;
}

// The packed elements of the FP32 copy, where they save bytes and a sixteenth of
// the free memory holds them (a build that just fits the card keeps its room;
// the passes give the same J, bitwise, either way).
int build_jpacked(f2jk_ctx* ctx) {
    const int64_t N = ctx->nbf, elements = (int64_t)ctx->jlist_n[F2JK_F32] * ctx->jlist_vec[F2JK_F32];
    const double bytes = (double)elements * 4.0 * (double)ctx->naux;
    if ((double)elements > 0.85 * (double)N * (N + 1) / 2) return F2JK_OK;
    size_t free_b = 0, total_b = 0;
    F2JK_HIP(hipMemGetInfo(&free_b, &total_b));
    if (bytes > (double)free_b / 16) return F2JK_OK;
    if (hipMalloc(&ctx->jpacked, (size_t)bytes) != hipSuccess) {
        (void)hipGetLastError();
        ctx->jpacked = nullptr;
        return F2JK_OK;
    }
    return pack_elements(ctx);
}

void free_jpacked(f2jk_ctx* ctx) {
    if (ctx->jpacked) (void)hipFree(ctx->jpacked);
    ctx->jpacked = nullptr;
}

void free_jlist(f2jk_ctx* ctx, int dtype) {
    if (dtype == F2JK_F32) free_jpacked(ctx);
    if (ctx->jlist[dtype]) (void)hipFree(ctx->jlist[dtype]);
    if (ctx->jinv[dtype]) (void)hipFree(ctx->jinv[dtype]);
    ctx->jlist[dtype] = nullptr;
    ctx->jinv[dtype] = nullptr;
    ctx->jlist_vec[dtype] = ctx->jlist_n[dtype] = 0;
}

int build_jlist(f2jk_ctx* ctx, int dtype) {
    free_jlist(ctx, dtype);
    if (!ctx->B[dtype]) return F2JK_OK;
    const int vec = j_vec_for(dtype, ctx->nbf);
    int rc = ensure_rowoff(ctx, vec);
    if (rc) return rc;
    const int N = (int)ctx->nbf, nvec = ctx->nvec[vec];
    F2JK_HIP(hipSetDevice(ctx->device));
    F2JK_HIP(hipDeviceSynchronize());  // B may have been written on any stream
    unsigned char* flag = nullptr;
    F2JK_HIP(hipMalloc(&flag, nvec));
    if (dtype == F2JK_F64)
        rc = vec == 2 ? scan_jlist<double, 2>(ctx, (const double*)ctx->B[dtype], flag)
                      : scan_jlist<double, 1>(ctx, (const double*)ctx->B[dtype], flag);
    else
        rc = vec == 4 ? scan_jlist<float, 4>(ctx, (const float*)ctx->B[dtype], flag)
           : vec == 2 ? scan_jlist<float, 2>(ctx, (const float*)ctx->B[dtype], flag)
                      : scan_jlist<float, 1>(ctx, (const float*)ctx->B[dtype], flag);
    std::vector<unsigned char> h(nvec);
    hipError_t e = rc ? hipSuccess : hipMemcpy(h.data(), flag, nvec, hipMemcpyDeviceToHost);
    (void)hipFree(flag);
    if (rc) return rc;
    if (e != hipSuccess) return fail(F2JK_EHIP, std::string("j_scan flags: ") + hipGetErrorString(e));
    std::vector<uint32_t> list;
    std::vector<int> inv(nvec, -1);
    if (std::none_of(h.begin(), h.end(), [](unsigned char f) { return f != 0; }))
        h[0] = 1;  // an all-zero B: one element keeps the launches non-empty
    int el = 0;
    for (int m = 0; m < N; ++m)
        for (int c = 0; c <= m; c += vec, ++el)
            if (h[el]) {
                inv[el] = (int)list.size();
                list.push_back(((uint32_t)m << 16) | (uint32_t)c);
            }
    F2JK_HIP(hipMalloc(&ctx->jlist[dtype], list.size() * sizeof(uint32_t)));
    F2JK_HIP(hipMemcpy(ctx->jlist[dtype], list.data(), list.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    F2JK_HIP(hipMalloc(&ctx->jinv[dtype], inv.size() * sizeof(int)));
    F2JK_HIP(hipMemcpy(ctx->jinv[dtype], inv.data(), inv.size() * sizeof(int), hipMemcpyHostToDevice));
    ctx->jlist_vec[dtype] = vec;
    ctx->jlist_n[dtype] = (int)list.size();
    if (ctx->j_pack && dtype == F2JK_F32) return build_jpacked(ctx);
    return F2JK_OK;
}

constexpr int kDSlots = 512;  // workgroups of the FP64 K kernels that run at once: two per CU


// the row sums of the half-transform's epilogue (grow null: none)
struct KxdGamma {
    const double* cp = nullptr;
    double* grow = nullptr;
    int64_t stride = 0;
    DCols dc{};
};

// Limits of a plan that are otherwise the context's launch-shape knobs; the
// no-alloc entry point lowers them until the plan fits its scratch array.
struct PlanCaps {
    size_t xchunk_bytes;
    int target_blocks;
};

int make_plan(const f2jk_ctx* ctx, int ndens, const int64_t* nocc, int precision, int flags,
              bool j_from_c, Plan& p, int jvec_override = 0, bool grouped = false,
              const PlanCaps* caps = nullptr) {
    const size_t xchunk_bytes = caps ? caps->xchunk_bytes : ctx->xchunk_bytes;
    const int target_blocks = caps ? caps->target_blocks : ctx->target_blocks;
    if (ctx->nbf <= 0 || ctx->naux <= 0) return fail(F2JK_ESTATE, "B has not been set");
    if (ndens < 1 || ndens > kMaxDens)
        return fail(F2JK_EINVAL, "ndens must be in [1, " + std::to_string(kMaxDens) + "]");
    if (precision < F2JK_PREC_FP64 || precision > F2JK_PREC_BF16X3)
        return fail(F2JK_EINVAL, "unknown precision");
    p.N = (int)ctx->nbf;
    p.Q = (int)ctx->naux;
    p.nd = ndens;
    p.prec = precision;
    p.want_j = flags & F2JK_WANT_J;
    p.want_k = flags & F2JK_WANT_K;
    p.need_c = p.want_k || (p.want_j && j_from_c);
    p.gamma_x = precision == F2JK_PREC_FP64 && p.want_j && p.want_k && j_from_c;
    const int jdtype = (precision == F2JK_PREC_FP64) ? F2JK_F64 : F2JK_F32;
    const int kdtype = jdtype;
    if (p.want_j && !ctx->B[jdtype])
        return fail(F2JK_ESTATE, jdtype == F2JK_F64 ? "FP64 B not set" : "FP32 B not set");
    if (p.want_k && !ctx->B[kdtype])
        return fail(F2JK_ESTATE, kdtype == F2JK_F64 ? "FP64 B not set" : "FP32 B not set");
    p.tk = (kdtype == F2JK_F64) ? 8 : 4;
    const int N = p.N, Q = p.Q;

    size_t off = 0;
    if (p.need_c) {
        if (!nocc) return fail(F2JK_EINVAL, "nocc is required");
        int o = 0;
        // the FP64 contraction takes k steps of 8, the others whole LDS stages
        const int kalign = precision == F2JK_PREC_BF16X3 ? kBK16 : (precision == F2JK_PREC_FP64 && p.want_k) ? 8 : 16;
        for (int d = 0; d < ndens; ++d) {
            if (nocc[d] < 0 || nocc[d] > N) return fail(F2JK_EINVAL, "nocc out of range");
            p.width[d] = (int)(cdiv(std::max<int64_t>(nocc[d], 1), kalign) * kalign);
            p.ioff[d] = o;
            o += p.width[d];
        }
        p.OPAD = (int)cdiv(o, 16) * 16;
        // the C copy used for D (always fp64) and the K copy (fp64 or fp32)
        if (precision == F2JK_PREC_FP64 && p.want_k) {
            // column tiles of equal width, at most 20 blocks of 16
            const int nb = (int)cdiv(p.OPAD, 16);
            p.dncolt = (int)cdiv(nb, kDMaxNB);
            p.dnb = (int)cdiv(nb, p.dncolt);
            p.dnks = (int)cdiv(N, kDK);
        }
        // FP64 K alone reads neither of them, and with J no fp32 copy: K-only builds
        // that fitted the no-alloc scratch array before Cq came still do
        const bool dk = precision == F2JK_PREC_FP64 && p.want_k;
        p.off_cp = off;
        if (!dk || p.gamma_x) off += align_up((size_t)N * std::max(p.OPAD, p.dncolt * p.dnb * 16) * 8);
        p.off_cp32 = off;
        if (!dk) off += align_up((size_t)N * p.OPAD * 4);  // fp32 copy (FP32 K)
        if (precision == F2JK_PREC_FP64 && p.want_k) {
            p.off_cq = off;
            // where J and K come from C, D is not formed: Cq lies in the room of
            // D and its partials (of which there is still as much as before)
            const size_t cq = align_up((size_t)p.dncolt * p.dnks * p.dnb * 256 * 8);
            off += p.gamma_x ? std::max(cq, align_up((size_t)ndens * N * N * 8) + align_up((size_t)N * N * 8)) : cq;
        }
        p.KP = (int)(cdiv(N, kBK16) * kBK16);
        if (precision == F2JK_PREC_BF16X3) {
            // transposed hi/lo bf16 copies (BF16X3 K), with zero rows up to a
            // whole number of half-transform column tiles (at most 320 wide)
            p.ctrows = p.OPAD + 320;
            p.off_cth = off;
            off += align_up((size_t)p.ctrows * p.KP * 2);
            p.off_ctl = off;
            off += align_up((size_t)p.ctrows * p.KP * 2);
        }
    }
    if (p.want_j) {
        p.jb = (jdtype == F2JK_F64) ? 8 : 4;
        p.jvec = jvec_override ? jvec_override : j_vec_for(jdtype, N);
        int64_t nvec = 0;
        for (int64_t m = 0; m < N; ++m) nvec += (m + 1 + p.jvec - 1) / p.jvec;
        p.jdense = (int)nvec;
        if (!grouped && ctx->jlist[jdtype] && ctx->jlist_vec[jdtype] == p.jvec) {
            p.jlist = ctx->jlist[jdtype];
            p.jinv = ctx->jinv[jdtype];
            if (jdtype == F2JK_F32) p.jpacked = ctx->jpacked;
            nvec = ctx->jlist_n[jdtype];
        }
        p.nvec = (int)nvec;
        p.neg = (int)cdiv(nvec, (int64_t)kJThreads * kEPT);
        p.npc1 = (int)cdiv(Q, kJ1PerBlock);
        p.npc2 = (int)std::max<int64_t>(1, std::min<int64_t>(Q, cdiv(target_blocks, p.neg)));
        p.ppw2 = (int)cdiv(Q, p.npc2);
        // FP64 builds of up to 8 element groups (nbf ~180) are bound by their
        // launches: fewer of them, and (grouped too, for the same sums) no more
        // partials than two rounds of the reduction's loads (64 chunks), as long
        // as a block can form the gamma of its own P
        if (p.gamma_x && p.neg <= 8 && ndens <= 2) {
            p.ppw2 = std::max(p.ppw2, std::min<int>(kGBlock, (int)cdiv(Q, 64)));
            p.small = !grouped && p.ppw2 <= kGBlock;
        }
        p.npc2 = (int)cdiv(Q, p.ppw2);
        if (j_from_c && !p.gamma_x) {
            p.off_d = off;
            off += align_up((size_t)ndens * N * N * 8);
        }
        p.off_gpart = off;
        if (!p.gamma_x) off += align_up((size_t)p.neg * ndens * Q * 8);
        p.off_gamma = off;
        off += align_up((size_t)ndens * Q * 8);
        p.off_jpart = off;
        p.jpart_bytes = align_up((size_t)p.npc2 * ndens * (size_t)nvec * p.jvec * 8);
        off += p.jpart_bytes;
    }
    if (p.want_k) {
        // the row sums come beside X and not out of its cap: J does not change the
        // chunks of K, and a grouped job whose X fits stays one chunk
        const size_t per_p = (size_t)N * p.OPAD * p.tk;
        const size_t grow_p = p.gamma_x ? (size_t)p.dncolt * ndens * N * 8 : 0;
        int64_t pc = (int64_t)(xchunk_bytes / std::max<size_t>(per_p, 1));
        pc = std::max<int64_t>(1, std::min<int64_t>(pc, Q));
        // rows of a chunk are numbered in 32 bits; grouped launches walk their blocks
        pc = std::min<int64_t>(pc, grouped ? INT32_MAX / N : std::min(kMaxLaunchP, kMaxLaunchRows / N));
        p.per_p = per_p;
        // as many chunks as the cap needs, of balanced size: no short last
        // chunk whose launches would be all set-up and Kpart traffic
        pc = cdiv(Q, cdiv(Q, pc));
        p.Pc = (int)pc;
        p.nchunks = (int)cdiv(Q, pc);
        // BF16x3 single-job builds of large nbf contract in 256-wide tiles
        // (one 8-wave workgroup per CU); everything else in 128-wide tiles
        p.ks_tile = 128;
        if (precision == F2JK_PREC_BF16X3 && !grouped)
            p.ks_tile = ctx->ks_tile ? ctx->ks_tile : (N >= 768 ? 256 : 128);
        p.ntile = (int)cdiv(N, p.ks_tile);
        p.nlower = p.ntile * (p.ntile + 1) / 2;
        // splits of the P range: at most wg_target workgroups per launch
        // (rounded down, so that a launch fills whole rounds of the CUs
        // instead of starting a nearly empty last one)
        const int64_t wg_target = p.ks_tile == 256 ? target_blocks / 4 : target_blocks / 2;
        p.nsplit = (int)std::max<int64_t>(1, std::min<int64_t>(pc, wg_target / p.nlower));
        if (precision == F2JK_PREC_BF16X3) {
            // single-job builds run the tall (256-row) half-transform: build
            // times with 128 and 256 rows at nbf 192 175 / 171 us, 288 381 / 369,
            // 384 798 / 788, 576 2524 / 2437, 700 4379 / 4169, 960 12.5 / 11.1 ms
            p.kx_rows = 128;
            if (!grouped) p.kx_rows = ctx->kx_rows ? ctx->kx_rows : (N >= 192 ? 256 : 128);
            if (N % 4 || N < 32) p.kx_rows = 128;  // the tall kernel loads A rows 16 bytes at a time
            p.nbw = bf16_tile_units((int)cdiv(p.OPAD, 32), ctx->bf16_nbw_max, p.kx_rows);
            p.kx_waves = ctx->kx_waves;
            p.ncolt = (int)cdiv(p.OPAD, 32 * p.nbw);
        } else if (precision == F2JK_PREC_FP32) {
            // one 320-column tile reads each row block of B once (the
            // 128-column kernel once per column tile)
            p.kx_wide = !grouped && (ctx->kx_wide < 0 ? p.OPAD > kTile : ctx->kx_wide == 1);
            p.ncolt = (int)cdiv(p.OPAD, p.kx_wide ? kWideCols : kTile);
        }
        p.kva = (N % 4 == 0) ? 4 : ((N % 2 == 0) ? 2 : 1);
        p.off_x = off;
        p.x_bytes = align_up((size_t)p.Pc * per_p);
        off += p.x_bytes;
        p.off_grow = off;
        off += align_up((size_t)p.Pc * grow_p);
        if (p.nchunks > 1) p.small = false;  // the row sums of the last chunk only are there
        if (precision == F2JK_PREC_FP64) {
            p.dt = dtile_plan(N, pc, p.width[0], (int)std::min<int64_t>(kDSlots, target_blocks));
            p.nsplit = p.dt.G;  // partials held per density
        }
        p.off_kpart = off;
        p.kpart_bytes = align_up((size_t)p.nsplit * ndens * N * N * 8);
        off += p.kpart_bytes;
    }
    p.total = std::max<size_t>(off, 256);
    return F2JK_OK;
}

// --------------------------------------------------------------------------- timing
void tim_begin(f2jk_ctx* ctx, bool on) {
    ctx->timing = on;
    ctx->nev = 0;
    ctx->total_recorded = false;
}
int tim_mark(f2jk_ctx* ctx, int phase, hipStream_t st, bool start) {
    if (!ctx->timing) return F2JK_OK;
    if (phase == F2JK_PH_TOTAL) {
        F2JK_HIP(hipEventRecord(ctx->ev_total[start ? 0 : 1], st));
        if (!start) ctx->total_recorded = true;
        return F2JK_OK;
    }
    if (start && ctx->nev + 2 > kMaxEvents) return F2JK_OK;  // table full: phase not timed
    if (!start && (ctx->nev % 2) == 0) return F2JK_OK;       // end of an untimed phase
    if (start) ctx->ev_phase[ctx->nev / 2] = phase;
    F2JK_HIP(hipEventRecord(ctx->ev[ctx->nev], st));
    ctx->nev++;
    return F2JK_OK;
}
#define TIM(phase, start)                                        \
    do {                                                         \
        int rc_ = tim_mark(ctx, phase, st, start);               \
        if (rc_) return rc_;                                     \
    } while (0)

// --------------------------------------------------------------------------- J
dim3 j_reduce_grid(int nvec) {
    const int64_t nb = cdiv(nvec, kJRedElems), x = std::min<int64_t>(nb, 1 << 22);
    return dim3((unsigned)x, (unsigned)cdiv(nb, x));
}
dim3 k_reduce_grid(int N, int nd) { return dim3((unsigned)cdiv(N, 16), (unsigned)cdiv(N, 4), nd); }

// densities d0 .. d0 + ND - 1; without D, gamma is there already
template <typename TB, int VEC, int ND, bool NT>
int launch_j(f2jk_ctx* ctx, const Plan& p, const TB* B, int d0, const double* const* D, int64_t ldd,
             double* const* J, char* ws, hipStream_t st) {
    DPtrs<ND> dp;
    JPtrs<ND> jp;
    for (int d = 0; d < ND; ++d) {
        dp.p[d] = D ? D[d0 + d] : nullptr;
        jp.p[d] = J[d0 + d];
    }
    double* gpart = (double*)(ws + p.off_gpart);
    double* gamma = (double*)(ws + p.off_gamma) + (D ? 0 : (size_t)d0 * p.Q);
    double* jpart = (double*)(ws + p.off_jpart);
    const int* rowoff = ctx->rowoff[VEC];
    const uint32_t* elist = p.jlist;
    if (D) {
        TIM(F2JK_PH_JGAMMA, true);
        hipLaunchKernelGGL((j_gamma_kernel<TB, VEC, kEPT, ND, NT>), dim3(p.neg, p.npc1), dim3(kJThreads), 0,
                           st, B, p.N, p.Q, dp, ldd, rowoff, elist, (const TB*)p.jpacked, p.nvec, kJ1PerBlock,
                           gpart);
        F2JK_LAUNCHED("j_gamma");
        const int64_t ng = (int64_t)ND * p.Q;
        hipLaunchKernelGGL(j_gamma_reduce_kernel, dim3((unsigned)cdiv(ng, 256)), dim3(256), 0, st,
                           gpart, p.neg, ND, p.Q, gamma);
        F2JK_LAUNCHED("j_gamma_reduce");
        TIM(F2JK_PH_JGAMMA, false);
    }
    TIM(F2JK_PH_JACC, true);
    if constexpr (sizeof(TB) == 8 && VEC <= 2) {
        if (p.small) {
            hipLaunchKernelGGL((j_accum_rows_kernel<VEC, kEPT, ND>), dim3(p.neg, p.npc2), dim3(kJThreads), 0, st, B,
                               p.N, p.Q, (const double*)(ws + p.off_grow), (int64_t)p.Pc * p.N, p.dncolt, rowoff, elist,
                               p.nvec, p.ppw2, jpart);
            F2JK_LAUNCHED("j_accum_rows");
            TIM(F2JK_PH_JACC, false);
            return F2JK_OK;  // reduced together with K
        }
    }
    hipLaunchKernelGGL((j_accum_kernel<TB, VEC, kEPT, ND, NT>), dim3(p.neg, p.npc2), dim3(kJThreads), 0,
                       st, B, p.N, p.Q, gamma, rowoff, elist, (const TB*)p.jpacked, p.nvec, p.ppw2, jpart);
    F2JK_LAUNCHED("j_accum");
    hipLaunchKernelGGL((j_reduce_kernel<VEC, ND>), j_reduce_grid(p.jdense), dim3(kJThreads), 0, st, jpart, p.npc2,
                       p.N, rowoff, p.jinv, p.nvec, p.jdense, jp);
    F2JK_LAUNCHED("j_reduce");
    TIM(F2JK_PH_JACC, false);
    return F2JK_OK;
}

template <typename TB, int VEC>
int launch_j_nd(f2jk_ctx* ctx, const Plan& p, const TB* B, int nd, const double* const* D,
                int64_t ldd, double* const* J, char* ws, hipStream_t st) {
    // densities are processed two at a time: one read of B serves both
    int d = 0;
    while (d < nd) {
        int rc;
        const bool nt = ctx->j_nontemporal;
        if (nd - d >= 2) {
            rc = nt ? launch_j<TB, VEC, 2, true>(ctx, p, B, d, D, ldd, J, ws, st)
                    : launch_j<TB, VEC, 2, false>(ctx, p, B, d, D, ldd, J, ws, st);
            d += 2;
        } else {
            rc = nt ? launch_j<TB, VEC, 1, true>(ctx, p, B, d, D, ldd, J, ws, st)
                    : launch_j<TB, VEC, 1, false>(ctx, p, B, d, D, ldd, J, ws, st);
            d += 1;
        }
        if (rc) return rc;
    }
    return F2JK_OK;
}

int run_j(f2jk_ctx* ctx, const Plan& p, const double* const* D, int64_t ldd, double* const* J,
          char* ws, hipStream_t st) {
    if (p.no_alloc && !ctx->rowoff[p.jvec])
        return fail(F2JK_ESTATE, "J element table missing (set B of this precision first)");
    int rc = ensure_rowoff(ctx, p.jvec);
    if (rc) return rc;
    if (p.prec == F2JK_PREC_FP64) {
        const double* B = (const double*)ctx->B[F2JK_F64];
        if (p.jvec == 2) return launch_j_nd<double, 2>(ctx, p, B, p.nd, D, ldd, J, ws, st);
        return launch_j_nd<double, 1>(ctx, p, B, p.nd, D, ldd, J, ws, st);
    }
    const float* B = (const float*)ctx->B[F2JK_F32];
    if (p.jvec == 4) return launch_j_nd<float, 4>(ctx, p, B, p.nd, D, ldd, J, ws, st);
    if (p.jvec == 2) return launch_j_nd<float, 2>(ctx, p, B, p.nd, D, ldd, J, ws, st);
    return launch_j_nd<float, 1>(ctx, p, B, p.nd, D, ldd, J, ws, st);
}

// --------------------------------------------------------------------------- C packing, D
DCols dcols_of(const Plan& p, const int64_t* nocc) {
    DCols dc{};
    dc.nd = p.nd;
    for (int d = 0; d < p.nd; ++d) {
        dc.nocc[d] = (int)nocc[d];
        dc.width[d] = p.width[d];
        dc.ioff[d] = p.ioff[d];
    }
    return dc;
}

int pack_c(f2jk_ctx* ctx, const Plan& p, const double* const* C, const int64_t* nocc,
           const int64_t* ldc, char* ws, hipStream_t st) {
    double* cp = (double*)(ws + p.off_cp);
    DCoef cs{};
    for (int d = 0; d < p.nd; ++d) {
        if (nocc[d] > 0 && (!C[d] || !ldc || ldc[d] < nocc[d]))
            return fail(F2JK_EINVAL, "C pointer / ldc invalid");
        cs.C[d] = C[d];
        cs.ldc[d] = nocc[d] > 0 ? ldc[d] : 1;
    }
    if (p.want_k && p.prec == F2JK_PREC_FP64) {
        const int64_t n = (int64_t)p.dncolt * p.dnks * p.dnb * 256;
        hipLaunchKernelGGL(pack_cq_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, st, cs, dcols_of(p, nocc), p.N,
                           p.dncolt * p.dnb * 16, p.dnb, p.dnks, n, p.gamma_x ? cp : nullptr, (double*)(ws + p.off_cq));
        F2JK_LAUNCHED("pack_cq");
        return F2JK_OK;
    }
    PackOut out{};
    if (p.want_j) out.Cp = cp;
    if (p.want_k && p.prec == F2JK_PREC_FP32) out.Cp32 = (float*)(ws + p.off_cp32);
    int64_t n = (int64_t)p.N * p.OPAD;
    if (p.want_k && p.prec == F2JK_PREC_BF16X3) {
        // with zero rows past the occupied columns: the tall half-transform loads
        // whole column tiles without clamping
        out.Th = (u16*)(ws + p.off_cth);
        out.Tl = (u16*)(ws + p.off_ctl);
        out.rows = p.ctrows;
        out.KP = p.KP;
        n = (int64_t)p.ctrows * p.KP;
    }
    hipLaunchKernelGGL(pack_c_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, st, cs, dcols_of(p, nocc), p.N, p.OPAD,
                       out);
    F2JK_LAUNCHED("pack_c");
    return F2JK_OK;
}

// D_d = Cp_d Cp_d^T
int build_d(const Plan& p, const int64_t* nocc, char* ws, hipStream_t st) {
    hipLaunchKernelGGL(d_kernel, dim3(d_blocks(p.N), p.nd), dim3(256), 0, st, (const double*)(ws + p.off_cp), p.N, p.OPAD,
                       dcols_of(p, nocc), (double*)(ws + p.off_d));
    F2JK_LAUNCHED("d");
    return F2JK_OK;
}

// --------------------------------------------------------------------------- K
// X = A Cp (FP32) over `grid` tiles: 128 x 320 tiles (kx_wide_kernel) or 128 x 128
// (kx_kernel), as the plan's column tiling says
void launch_kx_fp32(const Plan& p, unsigned grid, const float* A, int64_t R, const float* cp, float* X,
                    hipStream_t st) {
    if (p.kx_wide) {
        if (p.kva == 4)
            hipLaunchKernelGGL((kx_wide_kernel<4>), dim3(grid), dim3(kWideThreads), 0, st, A, R, p.N, cp,
                               p.OPAD, X, p.ncolt);
        else if (p.kva == 2)
            hipLaunchKernelGGL((kx_wide_kernel<2>), dim3(grid), dim3(kWideThreads), 0, st, A, R, p.N, cp,
                               p.OPAD, X, p.ncolt);
        else
            hipLaunchKernelGGL((kx_wide_kernel<1>), dim3(grid), dim3(kWideThreads), 0, st, A, R, p.N, cp,
                               p.OPAD, X, p.ncolt);
    } else if (p.kva == 4) {
        hipLaunchKernelGGL((kx_kernel<4>), dim3(grid), dim3(kGThreads), 0, st, A, R, p.N, cp, p.OPAD, X,
                           p.ncolt);
    } else if (p.kva == 2) {
        hipLaunchKernelGGL((kx_kernel<2>), dim3(grid), dim3(kGThreads), 0, st, A, R, p.N, cp, p.OPAD, X,
                           p.ncolt);
    } else {
        hipLaunchKernelGGL((kx_kernel<1>), dim3(grid), dim3(kGThreads), 0, st, A, R, p.N, cp, p.OPAD, X,
                           p.ncolt);
    }
}

// FP64 half-transform of R rows: kxd_ib row blocks per wave when that still
// gives two workgroups to every CU, one otherwise (the products of an element
// of X and their order do not depend on it).
template <int NB, int IB>
void launch_kxd_ib(const Plan& p, const double* A, int64_t R, const double* cq, double* X, int64_t ldx, int ncol,
                   const KxdGamma& g, hipStream_t st) {
    const unsigned grid = (unsigned)(cdiv(R, 64 * IB) * p.dncolt);
    hipLaunchKernelGGL((kxd_kernel<NB, IB>), dim3(grid), dim3(256), 0, st, A, R, p.N, cq, p.dnks, X, ldx, ncol,
                       p.dncolt, g.cp, g.dc, g.grow, g.stride);
}
template <int NB>
void launch_kxd_nb(const Plan& p, const double* A, int64_t R, const double* cq, double* X, int64_t ldx, int ncol,
                   const KxdGamma& g, hipStream_t st) {
    constexpr int IB = kxd_ib(NB);
    if constexpr (IB >= 2) {
        if (cdiv(R, 64 * IB) * p.dncolt >= kDSlots)
            return launch_kxd_ib<NB, IB>(p, A, R, cq, X, ldx, ncol, g, st);
    }
    launch_kxd_ib<NB, 1>(p, A, R, cq, X, ldx, ncol, g, st);
}
template <int NB = 1>
void launch_kxd(const Plan& p, const double* A, int64_t R, const double* cq, double* X, int64_t ldx, int ncol,
                const KxdGamma& g, hipStream_t st) {
    if constexpr (NB <= kDMaxNB) {
        if (p.dnb == NB) return launch_kxd_nb<NB>(p, A, R, cq, X, ldx, ncol, g, st);
        launch_kxd<NB + 1>(p, A, R, cq, X, ldx, ncol, g, st);
    }
}

template <int NB = 1>
void launch_kxt(int nb, const double* M, int64_t pstride, int ld, int K, int ncol, int64_t nP, const double* cq, int nks,
                double* Y, int ni, int ncolt, hipStream_t st) {
    if constexpr (NB <= kDMaxNB) {
        if (nb != NB) return launch_kxt<NB + 1>(nb, M, pstride, ld, K, ncol, nP, cq, nks, Y, ni, ncolt, st);
        constexpr int IB = kxd_ib(NB);
        const int64_t nblocks = nP * cdiv(ncol, 16);
        hipLaunchKernelGGL((kxt_kernel<NB, IB>), dim3((unsigned)(cdiv(nblocks, 4 * IB) * ncolt)), dim3(256), 0, st, M,
                           pstride, ld, K, ncol, nblocks, cq, nks, Y, ni, ncolt);
    }
}

template <int VEC, int ND>
void launch_jkred(const f2jk_ctx* ctx, const Plan& p, const double* jpart, double* const* J, const double* kpart,
                  int64_t dstride, const KPtrs& kp, hipStream_t st) {
    JPtrs<ND> jp;
    for (int d = 0; d < ND; ++d) jp.p[d] = J[d];
    const int nbj = (int)cdiv(p.jdense, kJRedElems);
    hipLaunchKernelGGL((jkred_kernel<VEC, ND>), dim3(nbj + k_reduce_blocks(p.N) * ND), dim3(256), 0, st, jpart, p.npc2,
                       p.N, ctx->rowoff[VEC], p.jinv, p.nvec, p.jdense, jp, nbj, kpart, dstride, p.dt, kp);
}

// `after_kx` runs once the last chunk's half-transform (and gamma) is queued
template <typename T, typename F>
int run_k_typed(f2jk_ctx* ctx, const Plan& p, const int64_t* nocc, double* const* J, double* const* K, char* ws,
                hipStream_t st, F&& after_kx) {
    const T* B = (const T*)ctx->B[sizeof(T) == 8 ? F2JK_F64 : F2JK_F32];
    const T* cp = (sizeof(T) == 8) ? (const T*)(ws + p.off_cp) : (const T*)(ws + p.off_cp32);
    T* X = (T*)(ws + p.off_x);
    double* kpart = (double*)(ws + p.off_kpart);
    const int64_t NN = (int64_t)p.N * p.N;
    for (int c = 0; c < p.nchunks; ++c) {
        const int P0 = c * p.Pc;
        const int pc = std::min(p.Pc, p.Q - P0);
        const int64_t R = (int64_t)pc * p.N;
        const int64_t nrowt = cdiv(R, kTile);
        TIM(F2JK_PH_KX, true);
        const T* A = B + (int64_t)P0 * NN;
        if constexpr (sizeof(T) == 8) {
            KxdGamma g;
            if (p.gamma_x) {
                g.cp = cp;
                g.grow = (double*)(ws + p.off_grow);
                g.stride = (int64_t)p.Pc * p.N;
                g.dc = dcols_of(p, nocc);
            }
            launch_kxd(p, A, R, (const double*)(ws + p.off_cq), X, p.OPAD, p.OPAD, g, st);
        } else
            launch_kx_fp32(p, (unsigned)(nrowt * p.ncolt), A, R, cp, X, st);
        F2JK_LAUNCHED("kx");
        TIM(F2JK_PH_KX, false);
        if (p.gamma_x && !p.small) {
            TIM(F2JK_PH_JGAMMA, true);
            hipLaunchKernelGGL(gamma_rows_kernel, dim3((unsigned)cdiv(pc, 4), p.nd), dim3(256), 0, st,
                               (const double*)(ws + p.off_grow), (int64_t)p.Pc * p.N, p.nd, p.dncolt, p.N, pc,
                               (double*)(ws + p.off_gamma) + P0, p.Q);
            F2JK_LAUNCHED("gamma_rows");
            TIM(F2JK_PH_JGAMMA, false);
        }
        if (c + 1 == p.nchunks) {
            const int rc = after_kx();
            if (rc) return rc;
        }
        TIM(F2JK_PH_KS, true);
        const int nsplit = std::min(p.nsplit, pc);
        if constexpr (sizeof(T) == 8) {
            hipLaunchKernelGGL(ksd_kernel, dim3(p.dt.total * p.nd), dim3(256), 0, st, X, p.N, p.OPAD, dcols_of(p, nocc),
                               pc, p.dt, kpart, (int64_t)p.nsplit * NN, c > 0 ? 1 : 0);
            F2JK_LAUNCHED("ks");
        } else {
            for (int d = 0; d < p.nd; ++d) {
                hipLaunchKernelGGL(ks_kernel, dim3(p.nlower * nsplit), dim3(kGThreads), 0, st, X, p.N,
                                   p.OPAD, p.ioff[d], p.width[d], pc, nsplit, p.nlower,
                                   kpart + (size_t)d * p.nsplit * NN, c > 0 ? 1 : 0);
                F2JK_LAUNCHED("ks");
            }
        }
        TIM(F2JK_PH_KS, false);
    }
    TIM(F2JK_PH_KRED, true);
    const int nsplit_used = std::min(p.nsplit, std::min(p.Pc, p.Q));
    KPtrs kp{};
    for (int d = 0; d < p.nd; ++d) kp.p[d] = K[d];
    if constexpr (sizeof(T) == 8) {
        if (p.small) {
            const bool v2 = p.jvec == 2;
            const auto red = p.nd == 2 ? (v2 ? launch_jkred<2, 2> : launch_jkred<1, 2>)
                                       : (v2 ? launch_jkred<2, 1> : launch_jkred<1, 1>);
            red(ctx, p, (const double*)(ws + p.off_jpart), J, kpart, (int64_t)p.nsplit * NN, kp, st);
        } else {
            hipLaunchKernelGGL(kred_kernel, k_reduce_grid(p.N, p.nd), dim3(256), 0, st, kpart,
                               (int64_t)p.nsplit * NN, p.dt, p.N, kp);
        }
    } else
        hipLaunchKernelGGL(k_reduce_kernel, k_reduce_grid(p.N, p.nd), dim3(256), 0, st, kpart,
                           (int64_t)p.nsplit * NN, nsplit_used, p.N, kp);
    F2JK_LAUNCHED("k_reduce");
    TIM(F2JK_PH_KRED, false);
    return F2JK_OK;
}

template <int NBW, int WAVES>
void launch_kx_bf16_w(const Plan& p, unsigned grid, const float* A, int64_t R, const u16* th,
                      const u16* tl, u16* xh, u16* xl, hipStream_t st) {
    if (p.kva == 4)
        hipLaunchKernelGGL((kx_bf16x3_kernel<NBW, 4, WAVES>), dim3(grid), dim3(64 * WAVES), 0, st, A, R, p.N,
                           p.KP, th, tl, p.OPAD, xh, xl, p.ncolt);
    else if (p.kva == 2)
        hipLaunchKernelGGL((kx_bf16x3_kernel<NBW, 2, WAVES>), dim3(grid), dim3(64 * WAVES), 0, st, A, R, p.N,
                           p.KP, th, tl, p.OPAD, xh, xl, p.ncolt);
    else
        hipLaunchKernelGGL((kx_bf16x3_kernel<NBW, 1, WAVES>), dim3(grid), dim3(64 * WAVES), 0, st, A, R, p.N,
                           p.KP, th, tl, p.OPAD, xh, xl, p.ncolt);
}

// 8 waves for tiles of an even number of 32-column units (each wave then
// holds NBW/2 blocks of 16 columns); 4 waves otherwise
template <int NBW>
void launch_kx_bf16(const Plan& p, unsigned grid, const float* A, int64_t R, const u16* th,
                    const u16* tl, u16* xh, u16* xl, hipStream_t st) {
    if constexpr (NBW % 2 == 0 && NBW >= 4) {
        if (p.kx_waves == 8) return launch_kx_bf16_w<NBW, 8>(p, grid, A, R, th, tl, xh, xl, st);
    }
    launch_kx_bf16_w<NBW, 4>(p, grid, A, R, th, tl, xh, xl, st);
}

// The tall (256-row) half-transform: 2 x 4 waves at even widths (in 32-column
// units), 4 x 2 at odd ones, which 2 x 4 cannot split.  Widths that fit the
// job: at 224 columns (nbf 960) 7 units take 3.31 ms per chunk where 8 took
// 3.44; 4 x 2 waves at 6 units took 5.12 ms where 2 x 4 take 5.02 (nbf 1188).
// 9 units would spill.
template <int NBW = 1>
void launch_kx_bf16_tall(const Plan& p, unsigned grid, const float* A, int64_t R, const u16* th,
                         const u16* tl, u16* xh, u16* xl, hipStream_t st) {
    if constexpr (NBW <= 10) {
        if (p.nbw != NBW) return launch_kx_bf16_tall<NBW == 8 ? 10 : NBW + 1>(p, grid, A, R, th, tl, xh, xl, st);
        constexpr int WR = NBW % 2 ? 4 : 2;
        hipLaunchKernelGGL((kx_bf16x3_tall_kernel<NBW, WR, 8 / WR>), dim3(grid), dim3(512), 0, st, A, R, p.N, p.KP, th,
                           tl, p.OPAD, xh, xl, p.ncolt);
    }
}

template <typename F>
int run_k_bf16x3(f2jk_ctx* ctx, const Plan& p, double* const* K, char* ws, hipStream_t st, F&& after_kx) {
    const float* B = (const float*)ctx->B[F2JK_F32];
    const u16* th = (const u16*)(ws + p.off_cth);
    const u16* tl = (const u16*)(ws + p.off_ctl);
    // X chunk: hi half then lo half
    u16* xh = (u16*)(ws + p.off_x);
    u16* xl = xh + (size_t)p.Pc * p.N * p.OPAD;
    double* kpart = (double*)(ws + p.off_kpart);
    const int64_t NN = (int64_t)p.N * p.N;
    for (int c = 0; c < p.nchunks; ++c) {
        const int P0 = c * p.Pc;
        const int pc = std::min(p.Pc, p.Q - P0);
        const int64_t R = (int64_t)pc * p.N;
        const float* A = B + (int64_t)P0 * NN;
        TIM(F2JK_PH_KX, true);
        if (p.kx_rows == 256) {
            const unsigned grid = (unsigned)(cdiv(R, kTallRows) * p.ncolt);
            launch_kx_bf16_tall(p, grid, A, R, th, tl, xh, xl, st);
        } else {
        const unsigned grid = (unsigned)(cdiv(R, kTile) * p.ncolt);
        switch (p.nbw) {
            case 2: launch_kx_bf16<2>(p, grid, A, R, th, tl, xh, xl, st); break;
            case 4: launch_kx_bf16<4>(p, grid, A, R, th, tl, xh, xl, st); break;
            case 5: launch_kx_bf16<5>(p, grid, A, R, th, tl, xh, xl, st); break;
            case 6: launch_kx_bf16<6>(p, grid, A, R, th, tl, xh, xl, st); break;
            case 8: launch_kx_bf16<8>(p, grid, A, R, th, tl, xh, xl, st); break;
            default: launch_kx_bf16<10>(p, grid, A, R, th, tl, xh, xl, st); break;
        }
        }
        F2JK_LAUNCHED("kx_bf16x3");
        TIM(F2JK_PH_KX, false);
        if (c + 1 == p.nchunks) {
            const int rc = after_kx();
            if (rc) return rc;
        }
        TIM(F2JK_PH_KS, true);
        const int nsplit = std::min(p.nsplit, pc);
        const bool ks_dma = ctx->ks_dma < 0 ? p.ks_tile == 256 : ctx->ks_dma == 1;
        for (int d = 0; d < p.nd; ++d) {
            if (ks_dma && p.ks_tile == 256)
                hipLaunchKernelGGL((ks_bf16x3_dma_kernel<256, 4, 2>), dim3(p.nlower * nsplit), dim3(512), 0, st,
                                   xh, xl, p.N, p.OPAD, p.ioff[d], p.width[d], pc, nsplit, p.nlower,
                                   kpart + (size_t)d * p.nsplit * NN, c > 0 ? 1 : 0);
            else if (ks_dma)
                hipLaunchKernelGGL((ks_bf16x3_dma_kernel<kTile, 2, 2>), dim3(p.nlower * nsplit), dim3(kGThreads), 0,
                                   st, xh, xl, p.N, p.OPAD, p.ioff[d], p.width[d], pc, nsplit, p.nlower,
                                   kpart + (size_t)d * p.nsplit * NN, c > 0 ? 1 : 0);
            else if (p.ks_tile == 256)
                hipLaunchKernelGGL((ks_bf16x3_kernel<256, 4, 2>), dim3(p.nlower * nsplit), dim3(512), 0, st,
                                   xh, xl, p.N, p.OPAD, p.ioff[d], p.width[d], pc, nsplit, p.nlower,
                                   kpart + (size_t)d * p.nsplit * NN, c > 0 ? 1 : 0);
            else
                hipLaunchKernelGGL((ks_bf16x3_kernel<kTile, 2, 2>), dim3(p.nlower * nsplit), dim3(kGThreads), 0,
                                   st, xh, xl, p.N, p.OPAD, p.ioff[d], p.width[d], pc, nsplit, p.nlower,
                                   kpart + (size_t)d * p.nsplit * NN, c > 0 ? 1 : 0);
            F2JK_LAUNCHED("ks_bf16x3");
        }
        TIM(F2JK_PH_KS, false);
    }
    TIM(F2JK_PH_KRED, true);
    const int nsplit_used = std::min(p.nsplit, std::min(p.Pc, p.Q));
    KPtrs kp{};
    for (int d = 0; d < p.nd; ++d) kp.p[d] = K[d];
    hipLaunchKernelGGL(k_reduce_kernel, k_reduce_grid(p.N, p.nd), dim3(256), 0, st, kpart,
                       (int64_t)p.nsplit * NN, nsplit_used, p.N, kp);
    F2JK_LAUNCHED("k_reduce");
    TIM(F2JK_PH_KRED, false);
    return F2JK_OK;
}

// FP64 J beside K pays from a J pass of this many bytes on: the second pass then
// reads B while the contraction (two waves of 182 registers and 64 KB of LDS
// per workgroup, so J's waves fit beside it) keeps the matrix cores busy.
// nbf 384 (B 1.3 GB in the pass) 1608 -> 1435 us per build, nbf 318 (0.3 GB)
// 408 -> 376, nbf 1152 99.1 -> 97.5 ms; at nbf 115 (28 MB) the events cost more
// than the 8 us pass (61 -> 73 us).  In the BF16x3 form both passes run beside
// the last chunk's contraction (nbf 960: 11.84 -> 11.38 ms); beside the
// half-transform, which fills the register file, they gained 1%, and beside the
// contraction in 128-wide tiles, itself bound by reading X, nothing (nbf 384:
// 769 and 775 us).
constexpr double kOverlapBytes = 128e6;
double j_pass_bytes(const Plan& p) { return (double)p.nvec * p.jvec * p.jb * p.Q; }

// A stream that joins a capture stays in it until the capture ends, and another
// stream's build on the same context meanwhile would be drawn in: a build being
// captured keeps to its own stream unless "overlap_jk" asks for the side stream.
bool capturing(hipStream_t st) {
    if (!st) return false;  // the default stream cannot be captured
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &status) != hipSuccess) (void)hipGetLastError();
    return status != hipStreamCaptureStatusNone;
}

int check_ws(size_t need, void* ws, size_t ws_bytes) {
    if (!ws) return fail(F2JK_EINVAL, "workspace pointer is NULL");
    if (ws_bytes < need)
        return fail(F2JK_ENOMEM, "workspace too small: need " + std::to_string(need) + " bytes, got " +
                                     std::to_string(ws_bytes));
    if (((uintptr_t)ws) % 256) return fail(F2JK_EINVAL, "workspace must be 256-byte aligned");
    return F2JK_OK;
}

int build_common(f2jk_ctx* ctx, int ndens, const double* const* C, const int64_t* nocc,
                 const int64_t* ldc, const double* const* Din, int64_t ldd, double* const* J,
                 double* const* K, int precision, int flags, void* ws, size_t ws_bytes, void* stream,
                 bool j_from_c, const PlanCaps* caps = nullptr, bool no_alloc = false) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    Plan p;
    int rc = make_plan(ctx, ndens, nocc, precision, flags, j_from_c, p, 0, false, caps);
    if (rc) return rc;
    p.no_alloc = no_alloc;
    if ((rc = check_ws(p.total, ws, ws_bytes))) return rc;
    for (int d = 0; d < ndens; ++d) {
        if (p.want_j && !J[d]) return fail(F2JK_EINVAL, "J output pointer is NULL");
        if (p.want_k && !K[d]) return fail(F2JK_EINVAL, "K output pointer is NULL");
        if (p.want_j && !j_from_c && !Din[d]) return fail(F2JK_EINVAL, "D pointer is NULL");
    }
    F2JK_HIP(hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    // a captured build reads B itself: its replays see values written later, and
    // do not depend on memory that "j_pack" may have given back by then
    if (p.jpacked && capturing(st)) p.jpacked = nullptr;
    char* w = (char*)ws;
    tim_begin(ctx, flags & F2JK_TIMING);
    TIM(F2JK_PH_TOTAL, true);
    if (p.need_c) {
        TIM(F2JK_PH_PREP, true);
        if ((rc = pack_c(ctx, p, C, nocc, ldc, w, st))) return rc;
        if (p.want_j && j_from_c && !p.gamma_x)
            if ((rc = build_d(p, nocc, w, st))) return rc;
        TIM(F2JK_PH_PREP, false);
    }
    // the J passes: on the side stream (forked once their inputs exist) when they
    // run beside K
    const bool overlap = p.want_j && p.want_k && !p.small &&
                         (ctx->overlap_jk < 0 ? (p.gamma_x || (p.prec == F2JK_PREC_BF16X3 && p.ks_tile == 256)) &&
                                                    !ctx->timing && j_pass_bytes(p) >= kOverlapBytes && !capturing(st)
                                              : ctx->overlap_jk == 1);
    hipStream_t sj = overlap ? ctx->side : st;
    bool forked = false;
    auto do_j = [&]() -> int {
        if (!p.want_j) return F2JK_OK;
        if (overlap) {
            std::lock_guard<std::mutex> lock(ctx->ev_mu);
            F2JK_HIP(hipEventRecord(ctx->ev_fork, st));
            F2JK_HIP(hipStreamWaitEvent(ctx->side, ctx->ev_fork, 0));
            forked = true;
        }
        if (p.gamma_x) return run_j(ctx, p, nullptr, 0, J, w, sj);
        std::vector<const double*> dptr(ndens);
        for (int d = 0; d < ndens; ++d)
            dptr[d] = j_from_c ? (const double*)(w + p.off_d) + (size_t)d * p.N * p.N : Din[d];
        return run_j(ctx, p, dptr.data(), j_from_c ? p.N : ldd, J, w, sj);
    };
    // J once the last half-transform is queued (FP64: its gamma comes with it)
    const bool j_late = p.gamma_x || (overlap && p.prec == F2JK_PREC_BF16X3);
    if (!j_late) rc = do_j();
    if (!rc && p.want_k) {
        if (p.prec == F2JK_PREC_BF16X3)
            rc = run_k_bf16x3(ctx, p, K, w, st, [&] { return j_late ? do_j() : F2JK_OK; });
        else if (p.tk == 8)
            rc = run_k_typed<double>(ctx, p, nocc, J, K, w, st, [&] { return p.gamma_x ? do_j() : F2JK_OK; });
        else
            rc = run_k_typed<float>(ctx, p, nocc, J, K, w, st, [] { return F2JK_OK; });
    }
    // join, also after a failed launch: later work on the caller's stream comes
    // after the side stream's
    if (forked) {
        std::lock_guard<std::mutex> lock(ctx->ev_mu);
        F2JK_HIP(hipEventRecord(ctx->ev_join, sj));
        F2JK_HIP(hipStreamWaitEvent(st, ctx->ev_join, 0));
    }
    if (rc) return rc;
    TIM(F2JK_PH_TOTAL, false);
    g_last_error.clear();
    return F2JK_OK;
}

// --------------------------------------------------------------------------- no-alloc builds
// Scratch of f2jk_build_jk_noalloc: one array per device, held until the
// process ends.  In host code `scratch` names a host-side stand-in, never the
// device memory; the device address comes from hipGetSymbolAddress, once per
// device (f2jk_ctx_create), and only that address is handed to kernels.
static __device__ __align__(256) unsigned char scratch[F2JK_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// with `device` current
int scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return fail(F2JK_EUNSUPPORTED, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return F2JK_OK;
    void* ptr = nullptr;
    F2JK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr || ((uintptr_t)ptr) % 256) return fail(F2JK_EHIP, "scratch array has no aligned device address");
    g_scratch_ptr[device] = ptr;
    return F2JK_OK;
}

// The widest launch shapes whose build_jk plan fits `budget` bytes: starting
// from the context's knobs, the X chunk or the split count (the larger of the
// two regions first) is halved until the plan fits; ENOMEM when even one P
// per chunk and one split do not.
int fit_plan(const f2jk_ctx* ctx, int ndens, const int64_t* nocc, int precision, int flags, size_t budget,
             PlanCaps& caps) {
    caps = PlanCaps{ctx->xchunk_bytes, ctx->target_blocks};
    for (int it = 0; it < 256; ++it) {
        Plan p;
        int rc = make_plan(ctx, ndens, nocc, precision, flags, true, p, 0, false, &caps);
        if (rc) return rc;
        const size_t per_p = p.per_p;
        if (p.total <= budget) {
            // a chunk that was halved may have missed the array by little (nbf 384,
            // 76 columns: 139 P at 67.3 of 67.1 MB, then 68 P at 46): three more tries
            for (int q = 7; it > 0 && p.want_k && p.nchunks > 1 && q > 4; --q) {
                const PlanCaps more{std::min(ctx->xchunk_bytes, per_p * ((size_t)p.Pc * q / 4)), caps.target_blocks};
                Plan r;
                if (make_plan(ctx, ndens, nocc, precision, flags, true, r, 0, false, &more) || r.total > budget) continue;
                caps = more;
                break;
            }
            return F2JK_OK;
        }
        if (p.want_k && p.Pc > 1 && p.x_bytes >= p.jpart_bytes + p.kpart_bytes)
            caps.xchunk_bytes = per_p * (size_t)(p.Pc / 2);
        else if (caps.target_blocks > 1)
            caps.target_blocks /= 2;
        else if (p.want_k && p.Pc > 1)
            caps.xchunk_bytes = per_p * (size_t)(p.Pc / 2);
        else
            return fail(F2JK_ENOMEM, "build needs " + std::to_string(p.total) +
                                         " bytes of scratch at its smallest launch shapes; the no-alloc scratch "
                                         "array holds " + std::to_string(budget) + " (use f2jk_build_jk with a "
                                         "caller workspace)");
    }
    return fail(F2JK_ENOMEM, "no launch shape fits the no-alloc scratch array");
}

// --------------------------------------------------------------------------- grouped builds
int group_plan(f2jk_ctx* const* ctxs, int njobs, const int* ndens, const int64_t* nocc, int precision,
               int flags, std::vector<Plan>& plans) {
    if (njobs < 1) return fail(F2JK_EINVAL, "njobs must be >= 1");
    if (!ctxs || !ndens || !nocc) return fail(F2JK_EINVAL, "null argument");
    if (precision < F2JK_PREC_FP64 || precision > F2JK_PREC_BF16X3) return fail(F2JK_EINVAL, "unknown precision");
    const int jk = flags & (F2JK_WANT_J | F2JK_WANT_K);
    if (jk != (F2JK_WANT_J | F2JK_WANT_K) && jk != F2JK_WANT_K)
        return fail(F2JK_EUNSUPPORTED, "grouped builds compute J and K, or K only");
    plans.resize(njobs);
    int64_t k = 0;
    for (int j = 0; j < njobs; ++j) {
        if (!ctxs[j]) return fail(F2JK_EINVAL, "null context in group");
        if (ndens[j] < 1 || ndens[j] > 2) return fail(F2JK_EUNSUPPORTED, "grouped jobs have 1 or 2 densities");
        // one J vector width (2) for the whole group, so one kernel serves every job
        int rc = make_plan(ctxs[j], ndens[j], nocc + k, precision, flags, true, plans[j], 2, true);
        if (rc) return rc;
        const Plan& p = plans[j];
        if (p.N % 2) return fail(F2JK_EUNSUPPORTED, "grouped builds need an even nbf");
        if (p.nchunks != 1) return fail(F2JK_EUNSUPPORTED, "grouped builds need X in one chunk");
        if (ctxs[j]->device != ctxs[0]->device) return fail(F2JK_EINVAL, "group spans devices");
        k += ndens[j];
    }
    return F2JK_OK;
}

template <int PH, int PREC, int NBW = 2, int VA = 2>
int launch_group_phase(const GArgs& a, hipStream_t st) {
    GArgs b = a;
    int total = 0;
    for (int j = 0; j < a.njobs; ++j) {
        b.first[j] = total;
        total += phase_blocks<PREC>(a.job[j], PH);
    }
    for (int j = a.njobs; j <= kMaxGroup; ++j) b.first[j] = total;
    if (total == 0) return F2JK_OK;
    const unsigned grid = (unsigned)std::min(total, 4096);
    hipLaunchKernelGGL((grouped_kernel<PH, PREC, NBW, VA>), dim3(grid), dim3(256), 0, st, b);
    F2JK_LAUNCHED("grouped phase " + std::to_string(PH));
    return F2JK_OK;
}

// the half-transform of a BF16x3 group: tile width NBW (the widest job's) and load width VA
template <int VA>
int launch_group_kx_bf16(const GArgs& a, int nbw, hipStream_t st) {
    switch (nbw) {
        case 2: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 2, VA>(a, st);
        case 4: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 4, VA>(a, st);
        case 5: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 5, VA>(a, st);
        case 6: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 6, VA>(a, st);
        case 8: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 8, VA>(a, st);
        default: return launch_group_phase<GP_KX, F2JK_PREC_BF16X3, 10, VA>(a, st);
    }
}

// `beside`: the second J pass of an FP64 group runs on the side stream, beside
// the contraction (see kOverlapBytes); the caller joins it
template <int PREC>
int run_group(f2jk_ctx* ctx, const GArgs& a, int nbw, int va, hipStream_t st, bool beside) {
    int rc;
    constexpr bool gamma_x = PREC == F2JK_PREC_FP64;  // gamma comes with the half-transform
    TIM(F2JK_PH_PREP, true);
    if ((rc = launch_group_phase<GP_PAD, PREC>(a, st))) return rc;
    if constexpr (!gamma_x)
        if ((rc = launch_group_phase<GP_D, PREC>(a, st))) return rc;
    TIM(F2JK_PH_PREP, false);
    TIM(F2JK_PH_KX, true);
    if constexpr (PREC == F2JK_PREC_BF16X3) {
        rc = (va == 4) ? launch_group_kx_bf16<4>(a, nbw, st) : launch_group_kx_bf16<2>(a, nbw, st);
        if (rc) return rc;
    } else if constexpr (PREC == F2JK_PREC_FP64) {
        rc = nbw <= kGroupNarrowNB ? launch_group_phase<GP_KX, PREC, kGroupNarrowNB>(a, st)
                                   : launch_group_phase<GP_KX, PREC, kDMaxNB>(a, st);
        if (rc) return rc;
    } else {
        if ((rc = launch_group_phase<GP_KX, PREC>(a, st))) return rc;
    }
    TIM(F2JK_PH_KX, false);
    TIM(F2JK_PH_JGAMMA, true);
    if constexpr (!gamma_x)
        if ((rc = launch_group_phase<GP_GAMMA, PREC>(a, st))) return rc;
    if ((rc = launch_group_phase<GP_GRED, PREC>(a, st))) return rc;
    TIM(F2JK_PH_JGAMMA, false);
    hipStream_t sj = st;
    if (beside) {
        std::lock_guard<std::mutex> lock(ctx->ev_mu);
        F2JK_HIP(hipEventRecord(ctx->ev_fork, st));
        F2JK_HIP(hipStreamWaitEvent(ctx->side, ctx->ev_fork, 0));
        sj = ctx->side;
    }
    TIM(F2JK_PH_JACC, true);
    if ((rc = launch_group_phase<GP_JACC, PREC>(a, sj))) return rc;
    if ((rc = launch_group_phase<GP_JRED, PREC>(a, sj))) return rc;
    TIM(F2JK_PH_JACC, false);
    TIM(F2JK_PH_KS, true);
    if ((rc = launch_group_phase<GP_KS, PREC>(a, st))) return rc;
    TIM(F2JK_PH_KS, false);
    TIM(F2JK_PH_KRED, true);
    if ((rc = launch_group_phase<GP_KRED, PREC>(a, st))) return rc;
    TIM(F2JK_PH_KRED, false);
    return F2JK_OK;
}

}  // namespace

// =========================================================================== C ABI
extern "C" {

int f2jk_ctx_create(int device, f2jk_ctx** out) {
    if (!out) return fail(F2JK_EINVAL, "out is NULL");
    int ndev = 0;
    F2JK_HIP(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return fail(F2JK_EINVAL, "device index out of range");
    F2JK_HIP(hipSetDevice(device));
    int rc = scratch_init(device);
    if (rc) return rc;
    f2jk_ctx* ctx = new f2jk_ctx();
    ctx->device = device;
    for (int i = 0; i < kMaxEvents + 2; ++i) {
        hipEvent_t* slot = (i < kMaxEvents) ? &ctx->ev[i] : &ctx->ev_total[i - kMaxEvents];
        hipError_t e = hipEventCreate(slot);
        if (e != hipSuccess) {
            for (int j = 0; j < i; ++j)
                (void)hipEventDestroy(j < kMaxEvents ? ctx->ev[j] : ctx->ev_total[j - kMaxEvents]);
            delete ctx;
            return fail(F2JK_EHIP, std::string("hipEventCreate: ") + hipGetErrorString(e));
        }
    }
    hipError_t e1 = hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking);
    hipError_t e2 = (e1 == hipSuccess) ? hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) : e1;
    hipError_t e3 = (e2 == hipSuccess) ? hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming) : e2;
    if (e3 != hipSuccess) {
        f2jk_ctx_destroy(ctx);
        return fail(F2JK_EHIP, std::string("side stream: ") + hipGetErrorString(e3));
    }
    *out = ctx;
    return F2JK_OK;
}

int f2jk_ctx_destroy(f2jk_ctx* ctx) {
    if (!ctx) return F2JK_OK;
    (void)hipSetDevice(ctx->device);
    for (int i = 0; i < kMaxEvents; ++i) (void)hipEventDestroy(ctx->ev[i]);
    for (int i = 0; i < 2; ++i) (void)hipEventDestroy(ctx->ev_total[i]);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->side) {
        (void)hipStreamSynchronize(ctx->side);
        (void)hipStreamDestroy(ctx->side);
    }
    for (int v = 0; v < 5; ++v)
        if (ctx->rowoff[v]) (void)hipFree(ctx->rowoff[v]);
    free_jlist(ctx, F2JK_F64);
    free_jlist(ctx, F2JK_F32);
    delete ctx;
    return F2JK_OK;
}

int f2jk_set_B(f2jk_ctx* ctx, int dtype, const void* B, int64_t naux, int64_t nbf) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    if (dtype != F2JK_F64 && dtype != F2JK_F32) return fail(F2JK_EINVAL, "unknown dtype");
    if (!B) return fail(F2JK_EINVAL, "B is NULL");
    if (naux <= 0 || nbf <= 0 || naux > INT32_MAX || nbf > 65535)
        return fail(F2JK_EINVAL, "naux/nbf out of range");
    if (((uintptr_t)B) % 16) return fail(F2JK_EINVAL, "B must be 16-byte aligned");
    const void* other = ctx->B[1 - dtype];
    if (other && (ctx->naux != naux || ctx->nbf != nbf))
        return fail(F2JK_EINVAL, "B copies must share naux and nbf");
    if (ctx->nbf != nbf) {
        (void)hipSetDevice(ctx->device);
        for (int v = 0; v < 5; ++v)
            if (ctx->rowoff[v]) {
                (void)hipFree(ctx->rowoff[v]);
                ctx->rowoff[v] = nullptr;
                ctx->nvec[v] = 0;
            }
    }
    ctx->B[dtype] = B;
    ctx->naux = naux;
    ctx->nbf = nbf;
    // build the J element tables now so that builds allocate nothing
    int rc = ensure_rowoff(ctx, j_vec_for(dtype, nbf));
    if (rc) return rc;
    if (ctx->j_sparse && (rc = build_jlist(ctx, dtype))) return rc;
    g_last_error.clear();
    return F2JK_OK;
}

int f2jk_get_shape(const f2jk_ctx* ctx, int64_t* naux, int64_t* nbf) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    if (naux) *naux = ctx->naux;
    if (nbf) *nbf = ctx->nbf;
    return F2JK_OK;
}

int f2jk_set_tuning(f2jk_ctx* ctx, const char* key, int64_t value) {
    if (!ctx || !key) return fail(F2JK_EINVAL, "null argument");
    if (!strcmp(key, "xchunk_bytes")) {
        if (value < (1 << 20)) return fail(F2JK_EINVAL, "xchunk_bytes must be >= 1 MiB");
        ctx->xchunk_bytes = (size_t)value;
    } else if (!strcmp(key, "j_nontemporal")) {
        ctx->j_nontemporal = value != 0;
    } else if (!strcmp(key, "j_sparse")) {
        ctx->j_sparse = value != 0;
        for (int dt = 0; dt < 2; ++dt) {
            if (ctx->j_sparse) {
                int rc = build_jlist(ctx, dt);
                if (rc) return rc;
            } else {
                free_jlist(ctx, dt);
            }
        }
    } else if (!strcmp(key, "j_pack")) {
        ctx->j_pack = value != 0;
        F2JK_HIP(hipSetDevice(ctx->device));
        if (ctx->j_pack && ctx->jlist[F2JK_F32]) {
            F2JK_HIP(hipDeviceSynchronize());  // builds that read them, writes to B on any stream
            int rc = ctx->jpacked ? pack_elements(ctx) : build_jpacked(ctx);
            if (rc) return rc;
        } else if (!ctx->j_pack && ctx->jpacked) {
            F2JK_HIP(hipDeviceSynchronize());
            free_jpacked(ctx);
        }
    } else if (!strcmp(key, "ks_dma")) {
        if (value < -1 || value > 1) return fail(F2JK_EINVAL, "ks_dma must be -1, 0 or 1");
        ctx->ks_dma = (int)value;
    } else if (!strcmp(key, "kx_wide")) {
        if (value < -1 || value > 1) return fail(F2JK_EINVAL, "kx_wide must be -1, 0 or 1");
        ctx->kx_wide = (int)value;
    } else if (!strcmp(key, "kx_rows")) {
        if (value != 0 && value != 128 && value != 256) return fail(F2JK_EINVAL, "kx_rows must be 0, 128 or 256");
        ctx->kx_rows = (int)value;
    } else if (!strcmp(key, "bf16_nbw_max")) {
        if (value != 2 && value != 4 && value != 5 && value != 6 && value != 8 && value != 10)
            return fail(F2JK_EINVAL, "bf16_nbw_max must be 2, 4, 5, 6, 8 or 10");
        ctx->bf16_nbw_max = (int)value;
    } else if (!strcmp(key, "overlap_jk")) {
        ctx->overlap_jk = value < 0 ? -1 : value != 0;
    } else if (!strcmp(key, "ks_tile")) {
        if (value != 0 && value != 128 && value != 256) return fail(F2JK_EINVAL, "ks_tile must be 0, 128 or 256");
        ctx->ks_tile = (int)value;
    } else if (!strcmp(key, "kx_waves")) {
        if (value != 4 && value != 8) return fail(F2JK_EINVAL, "kx_waves must be 4 or 8");
        ctx->kx_waves = (int)value;

    } else if (!strcmp(key, "target_blocks")) {
        if (value < 1 || value > (1 << 20)) return fail(F2JK_EINVAL, "target_blocks out of range");
        ctx->target_blocks = (int)value;
    } else {
        return fail(F2JK_EINVAL, std::string("unknown tuning key ") + key);
    }
    return F2JK_OK;
}

int f2jk_workspace_size(const f2jk_ctx* ctx, int ndens, const int64_t* nocc, int precision, int flags,
                        size_t* bytes) {
    if (!ctx || !bytes) return fail(F2JK_EINVAL, "null argument");
    Plan p, j;
    int rc = make_plan(ctx, ndens, nocc, precision, flags, nocc != nullptr, p);
    if (rc) return rc;
    // J and K in FP64 keep neither D nor the partial gamma, which J alone has:
    // the size is enough for that too (K alone needs less as it is)
    if (p.gamma_x) {
        rc = make_plan(ctx, ndens, nocc, precision, flags & ~F2JK_WANT_K, true, j);
        if (rc) return rc;
    }
    p.total = std::max(p.total, j.total);
    *bytes = p.total;
    return F2JK_OK;
}

int f2jk_build_jk(f2jk_ctx* ctx, int ndens, const double* const* C, const int64_t* nocc,
                  const int64_t* ldc, double* const* J, double* const* K, int precision, int flags,
                  void* ws, size_t ws_bytes, void* stream) {
    if (!C || !nocc) return fail(F2JK_EINVAL, "C and nocc are required");
    return build_common(ctx, ndens, C, nocc, ldc, nullptr, 0, J, K, precision, flags, ws, ws_bytes,
                        stream, true);
}

int f2jk_build_jk_noalloc(f2jk_ctx* ctx, int ndens, const double* const* C, const int64_t* nocc,
                          const int64_t* ldc, double* const* J, double* const* K, int precision, int flags,
                          void* stream) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    if (!C || !nocc) return fail(F2JK_EINVAL, "C and nocc are required");
    void* ws = (ctx->device >= 0 && ctx->device < kMaxDevices) ? g_scratch_ptr[ctx->device] : nullptr;
    if (!ws) return fail(F2JK_ESTATE, "no scratch address for this device");
    PlanCaps caps;
    int rc = fit_plan(ctx, ndens, nocc, precision, flags, F2JK_NOALLOC_SCRATCH_BYTES, caps);
    if (rc) return rc;
    return build_common(ctx, ndens, C, nocc, ldc, nullptr, 0, J, K, precision, flags, ws,
                        F2JK_NOALLOC_SCRATCH_BYTES, stream, true, &caps, true);
}

int f2jk_build_j(f2jk_ctx* ctx, int ndens, const double* const* D, int64_t ldd, double* const* J,
                 int precision, int flags, void* ws, size_t ws_bytes, void* stream) {
    if (!D || !J) return fail(F2JK_EINVAL, "D and J are required");
    if (ctx && ldd < ctx->nbf) return fail(F2JK_EINVAL, "ldd < nbf");
    const int fl = (flags & F2JK_TIMING) | F2JK_WANT_J;
    return build_common(ctx, ndens, nullptr, nullptr, nullptr, D, ldd, J, nullptr, precision, fl, ws,
                        ws_bytes, stream, false);
}

int f2jk_build_k(f2jk_ctx* ctx, int ndens, const double* const* C, const int64_t* nocc,
                 const int64_t* ldc, double* const* K, int precision, int flags, void* ws,
                 size_t ws_bytes, void* stream) {
    if (!C || !nocc || !K) return fail(F2JK_EINVAL, "C, nocc and K are required");
    const int fl = (flags & F2JK_TIMING) | F2JK_WANT_K;
    return build_common(ctx, ndens, C, nocc, ldc, nullptr, 0, nullptr, K, precision, fl, ws, ws_bytes,
                        stream, false);
}

int f2jk_last_timings(f2jk_ctx* ctx, double* ms, int n) {
    if (!ctx || !ms) return fail(F2JK_EINVAL, "null argument");
    double acc[F2JK_NPHASE] = {0};
    for (int i = 0; i + 1 < ctx->nev; i += 2) {
        F2JK_HIP(hipEventSynchronize(ctx->ev[i + 1]));
        float t = 0.f;
        F2JK_HIP(hipEventElapsedTime(&t, ctx->ev[i], ctx->ev[i + 1]));
        acc[ctx->ev_phase[i / 2]] += t;
    }
    if (ctx->total_recorded) {
        F2JK_HIP(hipEventSynchronize(ctx->ev_total[1]));
        float t = 0.f;
        F2JK_HIP(hipEventElapsedTime(&t, ctx->ev_total[0], ctx->ev_total[1]));
        acc[F2JK_PH_TOTAL] = t;
    }
    for (int i = 0; i < n && i < F2JK_NPHASE; ++i) ms[i] = acc[i];
    return F2JK_OK;
}

int f2jk_last_launches(const f2jk_ctx* ctx, int* counts, int n) {
    if (!ctx || !counts) return fail(F2JK_EINVAL, "null argument");
    int c[F2JK_NPHASE] = {0};
    for (int i = 0; i + 1 < ctx->nev; i += 2) c[ctx->ev_phase[i / 2]]++;
    c[F2JK_PH_TOTAL] = ctx->total_recorded ? 1 : 0;
    for (int i = 0; i < n && i < F2JK_NPHASE; ++i) counts[i] = c[i];
    return F2JK_OK;
}

int f2jk_work(const f2jk_ctx* ctx, int ndens, const int64_t* nocc, int precision, int flags,
              double* j_bytes, double* k_flops) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    const double N = (double)ctx->nbf, Q = (double)ctx->naux;
    const double sb = (precision == F2JK_PREC_FP64) ? 8.0 : 4.0;
    if (j_bytes) {
        // two passes over the lower triangle of every B_P, plus D/J and gamma traffic
        *j_bytes = (flags & F2JK_WANT_J)
                       ? 2.0 * Q * (N * (N + 1) / 2) * sb + 8.0 * ndens * (2.0 * Q + 2.0 * N * N)
                       : 0.0;
    }
    if (k_flops) {
        double f = 0.0;
        if ((flags & F2JK_WANT_K) && nocc)
            for (int d = 0; d < ndens; ++d) {
                const double o = (double)nocc[d];
                f += 2.0 * Q * N * N * o + N * (N + 1) * Q * o;
            }
        *k_flops = f;
    }
    return F2JK_OK;
}

int f2jk_group_workspace_size(f2jk_ctx* const* ctxs, int njobs, const int* ndens, const int64_t* nocc,
                              int precision, int flags, size_t* job_bytes) {
    if (!job_bytes) return fail(F2JK_EINVAL, "null argument");
    std::vector<Plan> plans;
    int rc = group_plan(ctxs, njobs, ndens, nocc, precision, flags, plans);
    if (rc) return rc;
    for (int j = 0; j < njobs; ++j) job_bytes[j] = plans[j].total;
    return F2JK_OK;
}

int f2jk_group_build_jk(f2jk_ctx* const* ctxs, int njobs, const int* ndens, const double* const* C,
                        const int64_t* nocc, const int64_t* ldc, double* const* J, double* const* K,
                        int precision, int flags, void* const* ws, const size_t* ws_bytes, void* stream) {
    if (!C || !ldc || !K || !ws || !ws_bytes) return fail(F2JK_EINVAL, "null argument");
    std::vector<Plan> plans;
    int rc = group_plan(ctxs, njobs, ndens, nocc, precision, flags, plans);
    if (rc) return rc;
    const bool want_j = flags & F2JK_WANT_J;
    if (want_j && !J) return fail(F2JK_EINVAL, "null argument");
    F2JK_HIP(hipSetDevice(ctxs[0]->device));
    hipStream_t st = (hipStream_t)stream;
    // the group's tile width (widest job; FP64: column blocks) and the BF16x3 load
    // width (4 when every nbf allows it)
    int nbw = precision == F2JK_PREC_FP64 ? 1 : 2, va = 4;
    for (int j = 0; j < njobs; ++j) {
        nbw = std::max(nbw, precision == F2JK_PREC_FP64 ? plans[j].dnb : plans[j].nbw);
        if (plans[j].N % 4) va = 2;
    }
    std::vector<GJob> jobs(njobs);
    int64_t k = 0;
    for (int j = 0; j < njobs; ++j) {
        const Plan& p = plans[j];
        if ((rc = check_ws(p.total, ws[j], ws_bytes[j]))) return rc;
        if (want_j && (rc = ensure_rowoff(ctxs[j], p.jvec))) return rc;
        char* w = (char*)ws[j];
        GJob& g = jobs[j];
        std::memset(&g, 0, sizeof(g));
        g.B = ctxs[j]->B[precision == F2JK_PREC_FP64 ? F2JK_F64 : F2JK_F32];
        g.rowoff = want_j ? ctxs[j]->rowoff[p.jvec] : nullptr;
        g.Cp = precision != F2JK_PREC_FP64 || p.gamma_x ? (double*)(w + p.off_cp) : nullptr;
        g.Cp32 = (float*)(w + p.off_cp32);
        g.Cq = (double*)(w + p.off_cq);
        g.dnb = p.dnb;
        g.dncolt = p.dncolt;
        g.dnks = p.dnks;
        g.dt = p.dt;
        g.drows = 64 * (nbw <= kGroupNarrowNB ? 1 : kxd_ib(std::max(1, p.dnb)));
        if (precision == F2JK_PREC_BF16X3) {
            g.Cth = (u16*)(w + p.off_cth);
            g.Ctl = (u16*)(w + p.off_ctl);
        }
        g.X = (void*)(w + p.off_x);
        g.Kpart = (double*)(w + p.off_kpart);
        if (want_j) {
            g.grow = (double*)(w + p.off_grow);
            g.D = (double*)(w + p.off_d);
            g.gpart = (double*)(w + p.off_gpart);
            g.gamma = (double*)(w + p.off_gamma);
            g.jpart = (double*)(w + p.off_jpart);
        }
        g.want_j = want_j ? 1 : 0;
        g.N = p.N;
        g.Q = p.Q;
        g.nd = p.nd;
        g.OPAD = p.OPAD;
        g.KP = p.KP;
        for (int d = 0; d < p.nd; ++d, ++k) {
            if (!C[k] || !K[k] || (want_j && !J[k])) return fail(F2JK_EINVAL, "null C/J/K pointer in group");
            if (nocc[k] > 0 && ldc[k] < nocc[k]) return fail(F2JK_EINVAL, "ldc < nocc");
            g.C[d] = C[k];
            g.ldc[d] = nocc[k] > 0 ? ldc[k] : 1;
            g.nocc[d] = (int)nocc[k];
            g.width[d] = p.width[d];
            g.ioff[d] = p.ioff[d];
            g.J[d] = want_j ? J[k] : nullptr;
            g.K[d] = K[k];
        }
        g.nvec = p.nvec;
        g.neg = p.neg;
        g.npc1 = p.npc1;
        g.npc2 = p.npc2;
        g.ppw2 = p.ppw2;
        g.nlower = p.nlower;
        g.nsplit = std::min(p.nsplit, std::min(p.Pc, p.Q));
        g.ncolt = (precision == F2JK_PREC_BF16X3) ? (int)cdiv(p.OPAD, 32 * nbw) : p.ncolt;
    }
    // the longest jobs first: a launch starts its blocks in this order and ends
    // with short ones
    std::stable_sort(jobs.begin(), jobs.end(), [](const GJob& x, const GJob& y) {
        return (double)x.Q * x.N * x.N * x.OPAD > (double)y.Q * y.N * y.N * y.OPAD;
    });
    f2jk_ctx* ctx = ctxs[0];  // timing events of the group
    tim_begin(ctx, flags & F2JK_TIMING);
    TIM(F2JK_PH_TOTAL, true);
    double jbytes = 0.0;
    for (const Plan& p : plans) jbytes += j_pass_bytes(p);
    const bool beside = want_j && precision == F2JK_PREC_FP64 && !ctx->timing &&
                        (ctx->overlap_jk < 0 ? jbytes >= kOverlapBytes && !capturing(st) : ctx->overlap_jk == 1);
    for (int j0 = 0; j0 < njobs; j0 += kMaxGroup) {
        GArgs a;
        std::memset(&a, 0, sizeof(a));
        a.njobs = std::min(kMaxGroup, njobs - j0);
        for (int j = 0; j < a.njobs; ++j) a.job[j] = jobs[j0 + j];
        if (precision == F2JK_PREC_FP64)
            rc = run_group<F2JK_PREC_FP64>(ctx, a, nbw, va, st, beside);
        else if (precision == F2JK_PREC_FP32)
            rc = run_group<F2JK_PREC_FP32>(ctx, a, nbw, va, st, false);
        else
            rc = run_group<F2JK_PREC_BF16X3>(ctx, a, nbw, va, st, false);
        if (rc) break;
    }
    if (beside) {  // also after a failed launch: later work comes after the side stream's
        std::lock_guard<std::mutex> lock(ctx->ev_mu);
        F2JK_HIP(hipEventRecord(ctx->ev_join, ctx->side));
        F2JK_HIP(hipStreamWaitEvent(st, ctx->ev_join, 0));
    }
    if (rc) return rc;
    TIM(F2JK_PH_TOTAL, false);
    g_last_error.clear();
    return F2JK_OK;
}

// The packed coefficients of a plan are all that the half-transform keeps in its
// workspace (they come first): X goes to the caller's array.
int f2jk_half_transform_workspace_size(const f2jk_ctx* ctx, int64_t ncol, size_t* bytes) {
    if (!ctx || !bytes) return fail(F2JK_EINVAL, "null argument");
    if (ncol < 1) return fail(F2JK_EINVAL, "ncol must be >= 1");
    Plan p;
    int rc = make_plan(ctx, 1, &ncol, F2JK_PREC_FP64, F2JK_WANT_K, false, p);
    if (rc) return rc;
    *bytes = p.off_x;
    return F2JK_OK;
}

int f2jk_half_transform(f2jk_ctx* ctx, const double* C, int64_t ncol, int64_t ldc, int64_t p0, int64_t p1,
                        double* X, int64_t ldx, int precision, void* ws, size_t ws_bytes, void* stream) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    if (!C || !X) return fail(F2JK_EINVAL, "C and X are required");
    if (precision != F2JK_PREC_FP64) return fail(F2JK_EUNSUPPORTED, "the half-transform is FP64");
    if (ncol < 1 || ldc < ncol || ldx < ncol) return fail(F2JK_EINVAL, "ncol, ldc or ldx invalid");
    Plan p;
    int rc = make_plan(ctx, 1, &ncol, precision, F2JK_WANT_K, false, p);
    if (rc) return rc;
    if (p0 < 0 || p1 > p.Q || p0 >= p1) return fail(F2JK_EINVAL, "aux range [p0, p1) invalid");
    if ((rc = check_ws(p.off_x, ws, ws_bytes))) return rc;
    F2JK_HIP(hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    char* w = (char*)ws;
    const double* Cs[1] = {C};
    const int64_t lds[1] = {ldc};
    if ((rc = pack_c(ctx, p, Cs, &ncol, lds, w, st))) return rc;
    const double* B = (const double*)ctx->B[F2JK_F64];
    const double* cq = (const double*)(w + p.off_cq);
    const int64_t NN = (int64_t)p.N * p.N;
    const int64_t step = kMaxLaunchRows / p.N;
    for (int64_t P0 = p0; P0 < p1; P0 += step) {
        const int64_t R = std::min<int64_t>(step, p1 - P0) * p.N;
        launch_kxd(p, B + P0 * NN, R, cq, X + (P0 - p0) * p.N * ldx, ldx, (int)ncol, KxdGamma{}, st);
        F2JK_LAUNCHED("kx");
    }
    g_last_error.clear();
    return F2JK_OK;
}

// Scratch of f2jk_mo_block: both coefficient sets, and the intermediate of one
// block of P.  64 MB of it: what the first product writes the second one then
// reads from the last-level cache.  More where 64 MB give either launch less
// than one round of workgroups (100 to 200 of the 512 for wide sets at nbf 500
// and above), up to 512 MB: nbf 640 with 128 + 128 columns 4.52 ms with 64 MB,
// 3.57 with this (4.02 with at most 256 MB), 320 + 320 13.96 and 10.7, 640 + 640
// 35.8 and 28.9, nbf 499 with 99 + 99 2.46 and 1.77.
namespace {
struct MoPlan {
    Plan c[2];           // coefficient packing of C1 and C2
    bool rows_first;     // C1 first (Y = C1^T B_P, then Y C2), or C2 first (X = B_P C2, then C1^T X)
    int64_t step;        // P per block
    size_t off_c[2], off_t, total;
};
constexpr size_t kMoBlockBytes = size_t(64) << 20, kMoBlockMaxBytes = size_t(512) << 20;
int mo_plan(const f2jk_ctx* ctx, int64_t n1, int64_t n2, MoPlan& m) {
    const int64_t n[2] = {n1, n2};
    size_t off = 0;
    for (int i = 0; i < 2; ++i) {
        Plan& p = m.c[i];
        int rc = make_plan(ctx, 1, &n[i], F2JK_PREC_FP64, F2JK_WANT_K, false, p);
        if (rc) return rc;
        // only the packed coefficients of the plan are used
        m.off_c[i] = off;
        off += p.off_x;
    }
    const int64_t N = m.c[0].N, Q = m.c[0].Q;
    m.rows_first = n1 < n2;  // the narrow set first: fewer products
    const int64_t per_p = 8 * N * std::min(n1, n2);
    // workgroups per P of the transform of the row index and of the other one
    const Plan &p1 = m.c[0], &p2 = m.c[1];
    const int64_t cols = m.rows_first ? N : n2, rows = m.rows_first ? n1 : N;
    const double wg = std::min((double)cdiv(cols, 16) / (4 * kxd_ib(p1.dnb)) * p1.dncolt,
                               (double)rows / (64 * kxd_ib(p2.dnb)) * p2.dncolt);
    const int64_t step = std::max((int64_t)kMoBlockBytes / per_p,
                                  std::min((int64_t)(kDSlots / wg), (int64_t)kMoBlockMaxBytes / per_p));
    m.step = std::max<int64_t>(1, std::min<int64_t>({Q, step, INT32_MAX / std::max(N, std::max(n1, n2))}));
    m.off_t = off;
    off += align_up((size_t)(m.step * per_p));
    m.total = off;
    return F2JK_OK;
}
}  // namespace

int f2jk_mo_block_workspace_size(const f2jk_ctx* ctx, int64_t n1, int64_t n2, size_t* bytes) {
    if (!ctx || !bytes) return fail(F2JK_EINVAL, "null argument");
    if (n1 < 1 || n2 < 1) return fail(F2JK_EINVAL, "n1 and n2 must be >= 1");
    MoPlan m;
    int rc = mo_plan(ctx, n1, n2, m);
    if (rc) return rc;
    *bytes = m.total;
    return F2JK_OK;
}

int f2jk_mo_block(f2jk_ctx* ctx, const double* C1, int64_t n1, int64_t ld1, const double* C2, int64_t n2, int64_t ld2,
                  double* out, void* ws, size_t ws_bytes, void* stream) {
    if (!ctx) return fail(F2JK_EINVAL, "null context");
    if (!C1 || !C2 || !out) return fail(F2JK_EINVAL, "C1, C2 and out are required");
    if (n1 < 1 || n2 < 1 || ld1 < n1 || ld2 < n2) return fail(F2JK_EINVAL, "n1, n2, ld1 or ld2 invalid");
    MoPlan m;
    int rc = mo_plan(ctx, n1, n2, m);
    if (rc) return rc;
    if ((rc = check_ws(m.total, ws, ws_bytes))) return rc;
    F2JK_HIP(hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    const double* C[2] = {C1, C2};
    const int64_t n[2] = {n1, n2}, ld[2] = {ld1, ld2};
    const double* cq[2];
    for (int i = 0; i < 2; ++i) {
        char* w = (char*)ws + m.off_c[i];
        if ((rc = pack_c(ctx, m.c[i], &C[i], &n[i], &ld[i], w, st))) return rc;
        cq[i] = (const double*)(w + m.c[i].off_cq);
    }
    const Plan &p1 = m.c[0], &p2 = m.c[1];
    const double* B = (const double*)ctx->B[F2JK_F64];
    double* T = (double*)((char*)ws + m.off_t);
    const int N = p1.N;
    const int64_t NN = (int64_t)N * N;
    for (int64_t P0 = 0; P0 < p1.Q; P0 += m.step) {
        const int64_t nP = std::min<int64_t>(m.step, p1.Q - P0);
        double* o = out + P0 * n1 * n2;
        if (m.rows_first) {
            launch_kxt(p1.dnb, B + P0 * NN, NN, N, N, N, nP, cq[0], p1.dnks, T, (int)n1, p1.dncolt, st);
            F2JK_LAUNCHED("kxt");
            launch_kxd(p2, T, nP * n1, cq[1], o, n2, (int)n2, KxdGamma{}, st);
            F2JK_LAUNCHED("kx");
        } else {
            launch_kxd(p2, B + P0 * NN, nP * N, cq[1], T, n2, (int)n2, KxdGamma{}, st);
            F2JK_LAUNCHED("kx");
            launch_kxt(p1.dnb, T, N * n2, (int)n2, N, (int)n2, nP, cq[0], p1.dnks, o, (int)n1, p1.dncolt, st);
            F2JK_LAUNCHED("kxt");
        }
    }
    g_last_error.clear();
    return F2JK_OK;
}

const char* f2jk_last_error(void) { return g_last_error.c_str(); }

}  // extern "C"
