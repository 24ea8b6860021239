// C ABI of the language-model cross-entropy (declared in include/mft/lm_loss.h).
//
// Validation mirrors the reference's checks (core/lm_loss.cpp:273-286 for the
// dense variant, :389-414 for the selected-token / streaming variant).  The
// streaming variant cuts the vocabulary into chunks of `chunk` rows of the
// LM-head weight; per chunk, with fp32 GEMMs on the bf16 matrix units
// (gemm_f32.h) or, for bf16 operands, rocBLAS:
//   forward   Z = hidden . W_c^T          (fp32 [N, chunk], workspace)
//             row statistics of Z merged into the running (max, sum)
//   backward  Z recomputed, G = (exp(Z - lse) - onehot) * coeff  (input dtype)
//             grad_hidden += G . W_c,  grad_weight[c] = G^T . hidden
// so the [N, V] logits never exist at once.  With bf16 operands and H a
// multiple of 64 the fused kernels of lm_loss_fused.hip replace the logits
// GEMM and the passes over it: the forward computes the row statistics in
// one pass with no logits at all, and the backward writes each chunk's G
// straight from the recomputed logits (no fp32 chunk).
#include "mft/lm_loss.h"

#include <algorithm>
#include <string>

#include "blas_util.h"
#include "capi_util.h"
#include "gemm_f32.h"
#include "lm_loss_kernels.h"

namespace {

using namespace mft::capi;

constexpr int64_t kDefaultChunk = 16384;
// fp32: the default chunk grows, so that few positions do not run GEMMs too
// short to fill the GPU (forward and backward at 512 positions, a vocabulary of
// 50257 and H 768 take 966 us as one chunk and 1060 as four), while its logits
// stay within kDefaultLogits values (half of the last-level cache) and within
// the two buffers of the default chunk and kMoreLogits values: G then takes the
// logits' place, and the workspace stays about that of the default chunk with
// the library's 64 MB.
constexpr int64_t kDefaultLogits = int64_t(1) << 25, kMoreLogits = int64_t(10) << 20;
constexpr size_t kBlasWorkspace = size_t(64) << 20;

size_t up(size_t x) { return (x + 255) & ~size_t(255); }

struct Layout {
    size_t m, s, tgt, nll, count, z, g, blas, part, total;
};

int64_t chunk_of(const mft_lm_loss_desc* d) {
    int64_t c = d->chunk > 0 ? d->chunk : kDefaultChunk;
    if (d->chunk == 0 && d->dtype == MFT_F32) {
        const int64_t N = d->B * d->S, most = std::min(kDefaultLogits / N, 2 * kDefaultChunk + kMoreLogits / N);
        if (most > c) {  // in chunks of one size (multiples of 64)
            const int64_t n = (d->V + most - 1) / most;
            c = std::max(c, ((d->V + n - 1) / n + 63) / 64 * 64);
        }
    }
    return c < d->V ? c : d->V;
}

// Whether a chunk's G is written over its logits (value by value, by the
// thread that read it).
bool g_over_logits(const mft_lm_loss_desc* d) { return d->dtype == MFT_F32 && chunk_of(d) > kDefaultChunk; }

// Row stride of a chunk's logits and G: a multiple of 8 elements, so that
// every row takes vector loads and stores (at a vocabulary of 50257 in one
// chunk the fp32 G . W took 431 us on unaligned rows, 248 on aligned ones).
int64_t chunk_ld(int64_t chunk) { return (chunk + 7) / 8 * 8; }

// The three products of a chunk of nc vocabulary rows in fp32:
// Z[N, nc] = hidden . W_c^T (row stride ldg), grad_hidden (+)= G . W_c, grad_W_c = G^T . hidden.
struct ChunkGemms {
    mft::GemmF32 z, dh, dw;
};
ChunkGemms chunk_gemms(const mft_lm_loss_desc* d, int64_t nc, int64_t ldg) {
    const int64_t N = d->B * d->S, H = d->H;
    ChunkGemms c{};
    c.z.M = N, c.z.N = nc, c.z.ldc = ldg;
    c.z.terms[0] = {nullptr, nullptr, H, H, H, 0, 1, 1.f};
    c.dh.M = N, c.dh.N = H, c.dh.ldc = H, c.dh.add = 1;
    c.dh.terms[0] = {nullptr, nullptr, ldg, H, nc, 0, 0, 1.f};
    c.dw.M = nc, c.dw.N = H, c.dw.ldc = H;
    c.dw.terms[0] = {nullptr, nullptr, ldg, H, N, 1, 0, 1.f};
    return c;
}
// Their workspace, for whole chunks and the last one.
size_t chunk_gemms_workspace(const mft_lm_loss_desc* d, int64_t chunk) {
    size_t w = 0;
    for (const int64_t nc : {chunk, d->V % chunk ? d->V % chunk : chunk}) {
        const ChunkGemms c = chunk_gemms(d, nc, chunk_ld(chunk));
        for (const mft::GemmF32* g : {&c.z, &c.dh, &c.dw}) w = std::max(w, mft::gemm_f32_workspace(*g));
    }
    return w;
}

Layout layout(const mft_lm_loss_desc* d, bool streaming) {
    const size_t N = (size_t)(d->B * d->S);
    Layout l{};
    size_t o = 0;
    l.m = o, o += up(N * 4);
    l.s = o, o += up(N * 8);
    l.tgt = o, o += up(N * 4);
    l.nll = o, o += up(N * 8);
    l.count = o, o += up(8);
    if (streaming) {
        const size_t c = (size_t)chunk_of(d);
        const size_t esz = d->dtype == MFT_BF16 ? 2 : 4;
        // the fused kernels need no fp32 logits chunk
        const bool fused = mft::ce_fused_supported(d->H, d->dtype == MFT_BF16);
        l.z = o, o += fused ? 0 : up(N * chunk_ld((int64_t)c) * 4);
        if (g_over_logits(d))
            l.g = l.z;
        else
            l.g = o, o += up(N * chunk_ld((int64_t)c) * esz);
        l.blas = o, o += d->dtype == MFT_F32 ? up(chunk_gemms_workspace(d, (int64_t)c)) : kBlasWorkspace;
        // fused forward: (max, sum) pairs per position and vocabulary part
        l.part = o, o += up(N * 2 * mft::kCeFusedMaxRanges * sizeof(float2));
    }
    l.total = o;
    return l;
}

mft_status check(const mft_lm_loss_desc* d, const char* who, bool streaming) {
    if (!d) return fail(MFT_ERR_INVALID_ARG, std::string(who) + ": desc is NULL");
    if (d->B <= 0 || d->S <= 0 || d->V <= 0)
        return fail(MFT_ERR_INVALID_ARG, "lm_cross_entropy: logits must be [B,S,V] and labels [B,S] (positive sizes)");
    if (d->dtype != MFT_F32 && d->dtype != MFT_BF16)
        return fail(MFT_ERR_INVALID_ARG, std::string(who) + ": dtype must be MFT_F32 or MFT_BF16");
    if (d->reduction != MFT_REDUCE_MEAN && d->reduction != MFT_REDUCE_SUM && d->reduction != MFT_REDUCE_NONE)
        return fail(MFT_ERR_INVALID_ARG, std::string(who) + ": reduction must be MEAN, SUM or NONE");
    if (d->chunk < 0) return fail(MFT_ERR_INVALID_ARG, std::string(who) + ": chunk must be >= 0");
    if (d->B * d->S > (int64_t(1) << 31) - 1 || d->V > (int64_t(1) << 31) - 1)
        return fail(MFT_ERR_UNSUPPORTED, std::string(who) + ": B*S and V must be below 2^31");
    if (streaming) {
        if (d->H <= 0) return fail(MFT_ERR_INVALID_ARG, "selected_token_lm_cross_entropy: hidden must be [B,S,H]");
        if (d->H > (int64_t(1) << 31) - 1) return fail(MFT_ERR_UNSUPPORTED, std::string(who) + ": H >= 2^31");
        if (d->reduction == MFT_REDUCE_NONE)
            return fail(MFT_ERR_INVALID_ARG,
                        "selected_token_lm_cross_entropy: only mean and sum reductions are supported");
    }
    return MFT_OK;
}

mft::CeArgs args(const mft_lm_loss_desc* d, const Layout& l, void* ws, const int32_t* labels) {
    mft::CeArgs a{};
    char* w = static_cast<char*>(ws);
    a.B = d->B;
    a.S = d->S;
    a.V = d->V;
    a.N = d->B * d->S;
    a.ignore = d->ignore_index;
    a.reduction = d->reduction;
    a.labels = labels;
    a.run_m = reinterpret_cast<float*>(w + l.m);
    a.run_s = reinterpret_cast<double*>(w + l.s);
    a.tgt = reinterpret_cast<float*>(w + l.tgt);
    a.nll = reinterpret_cast<double*>(w + l.nll);
    a.count = reinterpret_cast<long long*>(w + l.count);
    return a;
}

// The streaming variant's GEMMs of one call: gemm_f32 for fp32 operands, one
// rocBLAS handle (locked for the call) for bf16.
class Gemms {
public:
    Gemms(const mft_lm_loss_desc* d, const void* hidden, char* ws, hipStream_t st)
        : d_(d), hidden_(hidden), ws_(ws), st_(st), bf_(d->dtype == MFT_BF16), N_(d->B * d->S), H_(d->H) {}
    mft_status begin(const char* who) {
        who_ = who;
        if (!bf_) return MFT_OK;
        lock_ = mft::blas::lock();
        return mft::blas::bind(who, st_, ws_, kBlasWorkspace, &h_);
    }
    // Z[N, nc] (row stride ldz, fp32) = hidden[N, H] . W[v0 : v0 + nc, :]^T
    mft_status logits(const void* weight, int64_t v0, int64_t nc, float* Z, int64_t ldz) {
        const char* W = static_cast<const char*>(weight) + v0 * H_ * (bf_ ? 2 : 4);
        if (bf_)
            return mft::blas::gemm_rm(who_, h_, N_, nc, H_, 1.f, hidden_, H_, false, W, H_, true, 0.f, Z, ldz, true);
        return run(chunk_gemms(d_, nc, ldz).z, hidden_, W, Z);
    }
    // gh[N, H] (+)= G[N, nc] . W_c[nc, H]
    mft_status grad_hidden(const void* G, int64_t ldg, const void* Wc, int64_t nc, bool add, float* gh) {
        if (bf_)
            return mft::blas::gemm_rm(who_, h_, N_, H_, nc, 1.f, G, ldg, false, Wc, H_, false, add ? 1.f : 0.f, gh, H_,
                                      true);
        mft::GemmF32 g = chunk_gemms(d_, nc, ldg).dh;
        g.add = add;
        return run(g, G, Wc, gh);
    }
    // gw[nc, H] = G^T . hidden
    mft_status grad_weight(const void* G, int64_t ldg, int64_t nc, float* gw) {
        if (bf_)
            return mft::blas::gemm_rm(who_, h_, nc, H_, N_, 1.f, G, ldg, true, hidden_, H_, false, 0.f, gw, H_, true);
        return run(chunk_gemms(d_, nc, ldg).dw, G, hidden_, gw);
    }

private:
    mft_status run(mft::GemmF32 g, const void* A, const void* B, float* C) {
        g.terms[0].A = static_cast<const float*>(A);
        g.terms[0].B = static_cast<const float*>(B);
        g.C = C;
        g.partial = reinterpret_cast<float*>(ws_);
        return hip_status(mft::launch_gemm_f32(g, st_), who_);
    }
    const mft_lm_loss_desc* d_;
    const void* hidden_;
    char* ws_;
    hipStream_t st_;
    bool bf_;
    int64_t N_, H_;
    const char* who_ = "";
    std::unique_lock<std::mutex> lock_;
    rocblas_handle h_ = nullptr;
};

}  // namespace

extern "C" {

mft_status mft_lm_ce_workspace_size(const mft_lm_loss_desc* desc, size_t* fwd_bytes, size_t* bwd_bytes) {
    const bool streaming = desc && desc->H > 0;
    mft_status r = check(desc, "mft_lm_ce_workspace_size", streaming);
    if (r != MFT_OK) return r;
    const size_t t = layout(desc, streaming).total;
    if (fwd_bytes) *fwd_bytes = t;
    if (bwd_bytes) *bwd_bytes = t;
    return MFT_OK;
}

mft_status mft_lm_ce_fwd(const mft_lm_loss_desc* desc, const void* logits, const int32_t* labels, float* loss,
                         float* lse, int32_t* status, void* workspace, hipStream_t stream) {
    mft_status r = check(desc, "mft_lm_ce_fwd", false);
    if (r != MFT_OK) return r;
    if (!logits || !labels || !loss || !workspace)
        return fail(MFT_ERR_INVALID_ARG, "mft_lm_ce_fwd: logits, labels, loss and workspace must be non-NULL");
    const Layout l = layout(desc, false);
    mft::CeArgs a = args(desc, l, workspace, labels);
    a.lse = lse;
    a.loss = loss;
    a.status = status;
    hipError_t e = mft::launch_ce_stats(a, logits, desc->dtype == MFT_BF16, desc->V, desc->V, 0, true, stream);
    if (e == hipSuccess) e = mft::launch_ce_finalize(a, stream);
    return hip_status(e, "mft_lm_ce_fwd launch");
}

mft_status mft_lm_ce_bwd(const mft_lm_loss_desc* desc, const void* logits, const int32_t* labels, const float* lse,
                         const float* grad_loss, float* grad_logits, void* workspace, hipStream_t stream) {
    mft_status r = check(desc, "mft_lm_ce_bwd", false);
    if (r != MFT_OK) return r;
    if (!logits || !labels || !lse || !grad_logits || !workspace)
        return fail(MFT_ERR_INVALID_ARG,
                    "mft_lm_ce_bwd: logits, labels, lse, grad_logits and workspace must be non-NULL");
    const Layout l = layout(desc, false);
    mft::CeArgs a = args(desc, l, workspace, labels);
    a.lse_in = lse;
    a.grad_loss = grad_loss;
    hipError_t e = mft::launch_ce_count(a, stream);
    if (e == hipSuccess)
        e = mft::launch_ce_grad(a, logits, desc->dtype == MFT_BF16, desc->V, desc->V, 0, grad_logits, false, desc->V,
                                stream);
    return hip_status(e, "mft_lm_ce_bwd launch");
}

mft_status mft_lm_ce_streaming_fwd(const mft_lm_loss_desc* desc, const void* hidden, const void* weight,
                                   const int32_t* labels, float* loss, float* lse, int32_t* status, void* workspace,
                                   hipStream_t stream) {
    mft_status r = check(desc, "mft_lm_ce_streaming_fwd", true);
    if (r != MFT_OK) return r;
    if (!hidden || !weight || !labels || !loss || !workspace)
        return fail(MFT_ERR_INVALID_ARG,
                    "mft_lm_ce_streaming_fwd: hidden, weight, labels, loss and workspace must be non-NULL");
    const Layout l = layout(desc, true);
    mft::CeArgs a = args(desc, l, workspace, labels);
    a.lse = lse;
    a.loss = loss;
    a.status = status;
    char* w = static_cast<char*>(workspace);
    if (mft::ce_fused_supported(desc->H, desc->dtype == MFT_BF16)) {
        const mft::CeFusedArgs plan = mft::ce_fused_plan(a.N, desc->V, desc->H);
        hipError_t e = mft::launch_ce_fused_fwd(a, plan, hidden, weight, reinterpret_cast<float2*>(w + l.part), stream);
        if (e == hipSuccess) e = mft::launch_ce_finalize(a, stream);
        return hip_status(e, "mft_lm_ce_streaming_fwd launch");
    }
    float* Z = reinterpret_cast<float*>(w + l.z);
    const int64_t chunk = chunk_of(desc), ldz = chunk_ld(chunk);
    Gemms gemms(desc, hidden, w + l.blas, stream);
    if ((r = gemms.begin("mft_lm_ce_streaming_fwd")) != MFT_OK) return r;
    for (int64_t v0 = 0; v0 < desc->V; v0 += chunk) {
        const int64_t nc = desc->V - v0 < chunk ? desc->V - v0 : chunk;
        if ((r = gemms.logits(weight, v0, nc, Z, ldz)) != MFT_OK) return r;
        const hipError_t e = mft::launch_ce_stats(a, Z, false, ldz, nc, v0, v0 == 0, stream);
        if (e != hipSuccess) return hip_status(e, "mft_lm_ce_streaming_fwd launch");
    }
    return hip_status(mft::launch_ce_finalize(a, stream), "mft_lm_ce_streaming_fwd launch");
}

mft_status mft_lm_ce_streaming_bwd(const mft_lm_loss_desc* desc, const void* hidden, const void* weight,
                                   const int32_t* labels, const float* lse, const float* grad_loss, float* grad_hidden,
                                   float* grad_weight, void* workspace, hipStream_t stream) {
    mft_status r = check(desc, "mft_lm_ce_streaming_bwd", true);
    if (r != MFT_OK) return r;
    if (!hidden || !weight || !labels || !lse || !workspace)
        return fail(MFT_ERR_INVALID_ARG,
                    "mft_lm_ce_streaming_bwd: hidden, weight, labels, lse and workspace must be non-NULL");
    if (!grad_hidden && !grad_weight) return MFT_OK;
    const Layout l = layout(desc, true);
    mft::CeArgs a = args(desc, l, workspace, labels);
    a.lse_in = lse;
    a.grad_loss = grad_loss;
    char* w = static_cast<char*>(workspace);
    float* Z = reinterpret_cast<float*>(w + l.z);
    void* G = w + l.g;
    const bool bf = desc->dtype == MFT_BF16;
    const int64_t chunk = chunk_of(desc), N = desc->B * desc->S, H = desc->H;
    hipError_t e = mft::launch_ce_count(a, stream);
    if (e != hipSuccess) return hip_status(e, "mft_lm_ce_streaming_bwd launch");
    Gemms gemms(desc, hidden, w + l.blas, stream);
    if ((r = gemms.begin("mft_lm_ce_streaming_bwd")) != MFT_OK) return r;
    const bool fused = mft::ce_fused_supported(H, bf);
    const int64_t ldg = chunk_ld(chunk);
    mft::CeFusedArgs plan{};
    for (int64_t v0 = 0; v0 < desc->V; v0 += chunk) {
        const int64_t nc = desc->V - v0 < chunk ? desc->V - v0 : chunk;
        const char* Wc = static_cast<const char*>(weight) + v0 * H * (bf ? 2 : 4);
        if (fused) {  // G straight from the recomputed logits, no fp32 chunk
            if (v0 == 0 || nc != chunk) plan = mft::ce_fused_plan(N, nc, H);
            e = mft::launch_ce_fused_grad(a, plan, hidden, Wc, v0, G, ldg, stream);
        } else {
            if ((r = gemms.logits(weight, v0, nc, Z, ldg)) != MFT_OK) return r;
            e = mft::launch_ce_grad(a, Z, false, ldg, nc, v0, G, bf, ldg, stream);
        }
        if (e != hipSuccess) return hip_status(e, "mft_lm_ce_streaming_bwd launch");
        if (grad_hidden && (r = gemms.grad_hidden(G, ldg, Wc, nc, v0 > 0, grad_hidden)) != MFT_OK) return r;
        if (grad_weight && (r = gemms.grad_weight(G, ldg, nc, grad_weight + v0 * H)) != MFT_OK) return r;
    }
    return MFT_OK;
}

}  // extern "C"
