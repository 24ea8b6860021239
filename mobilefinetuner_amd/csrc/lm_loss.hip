// Language-model cross-entropy kernels (C ABI in include/mft/lm_loss.h).
//
// Rows are the B*S positions; position (b, s) is scored against
// labels[b, s + 1] (core/lm_loss.cpp:28-47, 292-296), not at s = S - 1 nor
// when that label is ignore_index.  The dense path runs each pass over whole
// rows of V logits; the streaming path runs the same passes over one chunk
// of vocabulary columns at a time (the GEMM output), merging the row
// statistics across chunks.
//
//   ce_row_stats  one workgroup per row: the chunk's online (max, sum of
//                 exp(z - max)) merged into the row's running pair, and the
//                 target logit when the label falls in the chunk
//   ce_finalize   lse = max + log(sum) and nll = lse - z[label] per row, as
//                 core/lm_loss.cpp:305-312 (double logsumexp)
//   ce_reduce     scored-row count and the sum of nll in a fixed order
//                 (double), with the work of ce_finalize where rows are few;
//                 MEAN divides by the count (NaN if zero), as :345-352
//   ce_grad       (exp(z - lse) - onehot(label)) * coeff, coeff = grad_loss *
//                 (1 / count for MEAN), as LMCrossEntropyBackward
//                 (:85-158): zero rows for unscored positions.
#include <hip/hip_runtime.h>

#include <cmath>

#include "attn_common.h"
#include "lm_loss_kernels.h"

namespace mft {
namespace {

constexpr int kCeThreads = 256;

__device__ __forceinline__ bool scored(const CeArgs& a, int64_t n, int* label) {
    const unsigned s = (unsigned)n % (unsigned)a.S;  // N < 2^31 (checked by the C ABI): a 32-bit division
    if (s + 1 >= (unsigned)a.S) return false;
    const int y = a.labels[n + 1];
    *label = y;
    return y != a.ignore;
}

template <typename T> __device__ __forceinline__ float to_f(T x) { return (float)x; }

// Block-wide (max, sum) merge of per-thread online pairs.
__device__ __forceinline__ void merge_pair(float& m, float& s, float m2, float s2) {
    const float mn = fmaxf(m, m2);
    if (mn == -INFINITY) {
        s += s2;  // 0, or the NaN of a value
        return;
    }
    s = s * __expf(m - mn) + s2 * __expf(m2 - mn);
    m = mn;
}

// VEC consecutive elements of a row as floats (VEC * sizeof(T) <= 16 bytes).
template <typename T, int VEC> struct RowVec {
    typedef T raw __attribute__((ext_vector_type(VEC)));
    __device__ static void load(const T* p, float* x) {
        const raw r = *reinterpret_cast<const raw*>(p);
#pragma unroll
        for (int e = 0; e < VEC; ++e) x[e] = (float)r[e];
    }
};

// Online (max, sum) update with VEC new values: one rescale per vector.
template <int VEC>
__device__ __forceinline__ void online_add(float& m, float& s, const float* x) {
    float vm = x[0];
#pragma unroll
    for (int e = 1; e < VEC; ++e) vm = fmaxf(vm, x[e]);
    if (vm > m) {
        s *= __expf(m - vm);
        m = vm;
    }
    // While all are -inf the exponentials are 0, but a NaN, which the maximum passes over, counts.
    const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int e = 0; e < VEC; ++e) s += __expf(x[e] - base);
}

// Elements from p to the next VEC-element boundary.
template <int VEC, typename T> __device__ __forceinline__ int to_boundary(const T* p) {
    return (int)(-(reinterpret_cast<uintptr_t>(p) / sizeof(T)) & (VEC - 1));
}

// HBM-bound: one pass over the logits.  A row of an odd number of values
// starts anywhere, so the vectors begin at the row's first 16-byte boundary
// and the elements around them are read singly.  NT threads to a row, four
// vectors in flight each: 1024 where the row fills that once, so that few rows
// are open at a time (long_rows), else 256.  fp32, 2048 rows of 50257, after
// their backward: 140 us (2.9 TB/s) when such rows were read element by
// element, 108 in vectors, 100 with 1024 threads, 56 (7.4 TB/s) since the
// backward leaves rows in the last-level cache (see ce_grad).
constexpr int kCeUnroll = 4;
template <typename T, int VEC, int NT>
__global__ __launch_bounds__(NT) void ce_row_stats(CeArgs a, const T* z, int64_t ld, int64_t ncols,
                                                           int64_t v0, int first) {
    __shared__ float sm[NT / 64], ss[NT / 64];
    const int64_t n = blockIdx.x;
    int y = 0;
    if (!scored(a, n, &y) || y < 0 || y >= a.V) return;
    const T* row = z + n * ld;
    float m = -INFINITY, s = 0.f;
    const int64_t head = min<int64_t>(to_boundary<VEC>(row), ncols), nvec = (ncols - head) / VEC;
    int64_t j = threadIdx.x;
    for (; j + (kCeUnroll - 1) * NT < nvec; j += kCeUnroll * NT) {
        float x[kCeUnroll * VEC];
#pragma unroll
        for (int u = 0; u < kCeUnroll; ++u) RowVec<T, VEC>::load(row + head + (j + u * NT) * VEC, x + u * VEC);
        online_add<kCeUnroll * VEC>(m, s, x);
    }
    for (; j < nvec; j += NT) {
        float x[VEC];
        RowVec<T, VEC>::load(row + head + j * VEC, x);
        online_add<VEC>(m, s, x);
    }
    // the fewer than 2 VEC elements around the vectors
    const int64_t rest = ncols - nvec * VEC;
    if (threadIdx.x < rest) {
        float x[1] = {(float)row[threadIdx.x < head ? threadIdx.x : nvec * VEC + threadIdx.x]};
        online_add<1>(m, s, x);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) merge_pair(m, s, __shfl_xor(m, o, 64), __shfl_xor(s, o, 64));
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sm[w] = m;
        ss[w] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float bm = sm[0], bs = ss[0];
        for (int k = 1; k < NT / 64; ++k) merge_pair(bm, bs, sm[k], ss[k]);
        // merge into the row's running pair (sum kept in double)
        if (first) {
            a.run_m[n] = bm;
            a.run_s[n] = (double)bs;
        } else if (a.run_m[n] == -INFINITY || bm == -INFINITY) {  // one of the sums is 0 (or NaN)
            a.run_m[n] = fmaxf(a.run_m[n], bm);
            a.run_s[n] += (double)bs;
        } else {
            const float om = a.run_m[n];
            const float mn = fmaxf(om, bm);
            a.run_s[n] = a.run_s[n] * exp((double)om - (double)mn) + (double)bs * exp((double)bm - (double)mn);
            a.run_m[n] = mn;
        }
        if (y >= v0 && y < v0 + ncols) a.tgt[n] = to_f(row[y - v0]);
    }
}

// lse and nll of row n.
__device__ __forceinline__ double finalize_row(const CeArgs& a, int64_t n, bool* is_scored) {
    int y = 0;
    double nll = 0.0;
    float lse = 0.f;
    *is_scored = scored(a, n, &y);
    if (*is_scored) {
        if (y < 0 || y >= a.V) {
            if (a.status) *a.status = 1;  // the reference throws "label out of range"
            nll = NAN;
        } else {
            const double l = (double)a.run_m[n] + log(a.run_s[n]);
            nll = l - (double)a.tgt[n];
            lse = (float)l;
        }
    }
    a.nll[n] = nll;
    if (a.lse) a.lse[n] = lse;
    if (a.reduction == CE_NONE && a.loss) a.loss[n] = (float)nll;
    return nll;
}

__global__ __launch_bounds__(kCeThreads) void ce_finalize(CeArgs a) {
    const int64_t n = (int64_t)blockIdx.x * kCeThreads + threadIdx.x;
    bool on;
    if (n < a.N) finalize_row(a, n, &on);
}

enum { kReduceCount = 0, kReduceLoss = 1, kReduceRows = 2 };

// One workgroup: count of scored rows and, but for kReduceCount, the loss.
// Each thread sums rows t, t + 1024, ... in order (coalesced), then the
// threads' sums combine in a fixed tree, in double.  kReduceRows finalizes
// the rows in the same pass (see launch_ce_finalize).
constexpr int kReduceThreads = 1024;
template <int MODE> __global__ __launch_bounds__(kReduceThreads) void ce_reduce(CeArgs a) {
    __shared__ double ps[kReduceThreads / 64];
    __shared__ int pc[kReduceThreads / 64];
    double sum = 0.0;
    int cnt = 0;
#pragma unroll 4
    for (int64_t n = threadIdx.x; n < a.N; n += kReduceThreads) {
        bool on;
        double nll = 0.0;
        if constexpr (MODE == kReduceRows) {
            nll = finalize_row(a, n, &on);
        } else {
            int y;
            on = scored(a, n, &y);
            if (MODE == kReduceLoss) nll = a.nll[n];
        }
        if (on) {
            ++cnt;
            sum += nll;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o, 64);
        cnt += __shfl_xor(cnt, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        ps[threadIdx.x >> 6] = sum;
        pc[threadIdx.x >> 6] = cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        long long c = 0;
        for (int k = 0; k < kReduceThreads / 64; ++k) {
            t += ps[k];
            c += pc[k];
        }
        *a.count = c;
        if (MODE != kReduceCount && a.reduction != CE_NONE && a.loss) {
            if (a.reduction == CE_SUM)
                a.loss[0] = (float)t;
            else
                a.loss[0] = c > 0 ? (float)(t / (double)c) : NAN;
        }
    }
}

template <typename OutT, int VEC, bool STREAM> struct OutVec {
    typedef OutT raw __attribute__((ext_vector_type(VEC)));
    __device__ static void store(OutT* p, const float* x) {
        raw r;
#pragma unroll
        for (int e = 0; e < VEC; ++e) r[e] = (OutT)x[e];
        if constexpr (STREAM)
            __builtin_nontemporal_store(r, reinterpret_cast<raw*>(p));
        else
            *reinterpret_cast<raw*>(p) = r;
    }
};

// HBM-bound: one read of the logits, one write of the gradient.  Vectors
// begin at the row's first boundary, as in ce_row_stats; a row whose z and g
// reach it at different elements (bases of different alignment, or row
// strides that differ) goes element by element.  Rows go last to first: the
// forward has just read them first to last, so the last ones are still in the
// last-level cache.  STREAM: a gradient too large to stay cached is stored
// past the caches, which leaves them to the logits.  fp32, 2048 rows of 50257,
// forward and backward passes in turn: 183 us element by element, 153 in
// vectors, 136 with 1024 threads to a row, the rows reversed and streaming
// stores (the passes' sum: 324, 261, 192; without streaming stores 220,
// without the reversal 223).
template <typename T, typename OutT, int VEC, int NT, bool STREAM>
__global__ __launch_bounds__(NT) void ce_grad(CeArgs a, const T* z, int64_t ld, int64_t ncols, int64_t v0,
                                                      OutT* g, int64_t ldg) {
    const int64_t n = a.N - 1 - (int64_t)blockIdx.x;
    OutT* grow = g + n * ldg;
    const T* row = z + n * ld;
    int y = 0;
    const bool on = scored(a, n, &y) && y >= 0 && y < a.V;
    float coeff = 0.f;
    if (on) {
        const float outer = a.grad_loss ? (a.reduction == CE_NONE ? a.grad_loss[n] : a.grad_loss[0]) : 1.f;
        const long long c = *a.count;
        const float base = a.reduction == CE_MEAN ? (c > 0 ? 1.0f / (float)c : 0.f) : 1.f;
        coeff = outer * base;
    }
    const int to = to_boundary<VEC>(grow);
    const int64_t head = to == to_boundary<VEC>(row) ? min<int64_t>(to, ncols) : ncols, nvec = (ncols - head) / VEC;
    const int64_t tail = head + nvec * VEC;  // first element after the vectors
    if (!on || coeff == 0.f) {
        float zero[VEC] = {};
        for (int64_t j = threadIdx.x; j < nvec; j += NT) OutVec<OutT, VEC, STREAM>::store(grow + head + j * VEC, zero);
        for (int64_t v = threadIdx.x; v < head; v += NT) grow[v] = (OutT)0.f;
        for (int64_t v = tail + threadIdx.x; v < ncols; v += NT) grow[v] = (OutT)0.f;
        return;
    }
    const float l = a.lse_in[n];
    for (int64_t j = threadIdx.x; j < nvec; j += NT) {
        float x[VEC];
        RowVec<T, VEC>::load(row + head + j * VEC, x);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            float p = __expf(x[e] - l);
            if (v0 + head + j * VEC + e == y) p -= 1.0f;
            x[e] = p * coeff;
        }
        OutVec<OutT, VEC, STREAM>::store(grow + head + j * VEC, x);
    }
    auto single = [&](int64_t v) {
        float p = __expf(to_f(row[v]) - l);
        if (v0 + v == y) p -= 1.0f;
        grow[v] = (OutT)(p * coeff);
    };
    for (int64_t v = threadIdx.x; v < head; v += NT) single(v);
    for (int64_t v = tail + threadIdx.x; v < ncols; v += NT) single(v);
}

// Whether rows of n elements keep 1024 threads with kCeUnroll vectors each.
bool long_rows(int64_t n, int vec) { return n >= (int64_t)kCeUnroll * 1024 * vec; }

// Bytes of gradient past which it is stored around the caches: half of the
// 256 MiB last-level cache, as much as can stay beside the logits.
constexpr int64_t kStreamBytes = int64_t(128) << 20;

}  // namespace

hipError_t launch_ce_stats(const CeArgs& a, const void* z, bool z_bf16, int64_t ld, int64_t ncols, int64_t v0,
                           bool first, hipStream_t st) {
    const dim3 grid((unsigned)a.N);
#define MFT_CE_STATS(T, VEC, NT) \
    hipLaunchKernelGGL((ce_row_stats<T, VEC, NT>), grid, dim3(NT), 0, st, a, (const T*)z, ld, ncols, v0, (int)first)
    if (z_bf16) {
        if (long_rows(ncols, 8)) MFT_CE_STATS(bf16, 8, 1024);
        else MFT_CE_STATS(bf16, 8, 256);
    } else {
        if (long_rows(ncols, 4)) MFT_CE_STATS(float, 4, 1024);
        else MFT_CE_STATS(float, 4, 256);
    }
#undef MFT_CE_STATS
    return hipGetLastError();
}

hipError_t launch_ce_finalize(const CeArgs& a, hipStream_t st) {
    // A few rows to each thread of one workgroup: one launch.  More rows go
    // to a launch of their own (the double logarithms would serialise).
    if (a.N <= 8 * kReduceThreads) {
        hipLaunchKernelGGL(ce_reduce<kReduceRows>, dim3(1), dim3(kReduceThreads), 0, st, a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(ce_finalize, dim3((unsigned)((a.N + kCeThreads - 1) / kCeThreads)), dim3(kCeThreads), 0, st,
                       a);
    hipLaunchKernelGGL(ce_reduce<kReduceLoss>, dim3(1), dim3(kReduceThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ce_count(const CeArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(ce_reduce<kReduceCount>, dim3(1), dim3(kReduceThreads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ce_grad(const CeArgs& a, const void* z, bool z_bf16, int64_t ld, int64_t ncols, int64_t v0, void* g,
                          bool g_bf16, int64_t ldg, hipStream_t st) {
    const dim3 grid((unsigned)a.N);
    // 4 elements per access: fp32 16 B, bf16 8 B
    const bool wide = long_rows(ncols, 4), stream = a.N * ncols * (g_bf16 ? 2 : 4) > kStreamBytes;
#define MFT_CE_GRAD(T, OutT, NT, STREAM)                                                                   \
    hipLaunchKernelGGL((ce_grad<T, OutT, 4, NT, STREAM>), grid, dim3(NT), 0, st, a, (const T*)z, ld, ncols, \
                       v0, (OutT*)g, ldg)
#define MFT_CE_GRAD_T(T, OutT)                            \
    do {                                                  \
        if (!wide) MFT_CE_GRAD(T, OutT, 256, false);      \
        else if (stream) MFT_CE_GRAD(T, OutT, 1024, true); \
        else MFT_CE_GRAD(T, OutT, 1024, false);           \
    } while (0)
    if (z_bf16 && !g_bf16) {
        MFT_CE_GRAD_T(bf16, float);
    } else if (!z_bf16 && !g_bf16) {
        MFT_CE_GRAD_T(float, float);
    } else if (!z_bf16 && g_bf16) {
        MFT_CE_GRAD_T(float, bf16);
    } else {
        return hipErrorInvalidValue;
    }
#undef MFT_CE_GRAD_T
#undef MFT_CE_GRAD
    return hipGetLastError();
}

}  // namespace mft
