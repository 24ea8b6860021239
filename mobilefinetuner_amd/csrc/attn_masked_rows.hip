// Query rows that see no key at all (key padding).
//
// With key padding (valid keys j < len of each batch) a query row can be left
// without a visible key: every row when len = 0, and with a causal sliding
// window of W keys every row i >= len + W - 1.  The reference still gives
// such a row a defined result: its scores are scale q.k plus the -1e10
// entries of the masks (graph/gemma_model.cpp:481-505: add(base mask), then
// add(pad mask)), so a key hidden by exactly one of the two masks scores
// -1e10 and a key hidden by both -2e10; the softmax (core/ops.cpp softmax,
// max-subtracted) is then exactly uniform over the keys hidden once,
//   T_i = [tlo(i), thi(i)] u [0, len),  |T_i| = thi - tlo + 1 + len,
// the keys the base mask lets through (all padded) plus the unpadded keys the
// base mask hides (scale q.k is far below the 1e10 spacing of 1024, so it
// vanishes from the sum).  Its output is the mean of V over T_i, independent
// of q, and its backward is that of P_ij = 1 / |T_i| on T_i:
//   dS_ij = (dO_i . v_j - delta_i) / |T_i|,  delta_i = dO_i . O_i
//   dq_i = scale sum_j dS_ij k_j,  dk_j += scale dS_ij q_i,  dv_j += dO_i / |T_i|.
// The main kernels leave these rows at O = 0, LSE = +inf, P = 0 (no visible
// key); the kernels below write the reference's values afterwards.  They run
// only when the caller passes key lengths, do O(rows x |T_i| x D) work, and
// skip rows whose dO is all zero (training with the padded positions' loss
// masked out: their gradients are exactly zero).
#include "attn_common.h"
#include "attn_kernels.h"

namespace mft {
namespace {

struct MaskedArgs {
    const void* q;
    const void* k;
    const void* v;
    void* o;          // forward output (overwritten on masked rows)
    const void* dO;
    float* dq;
    float* dk;
    float* dv;
    float* row_delta;  // [B*Hq*S] delta of masked rows (backward scratch)
    int* row_active;   // [B*Hq*S] masked row with non-zero dO (backward scratch)
    const int* kv_len;
    int B, Hq, Hkv, S, D, group, window, causal;
    float scale;
    Strides sq, sk, sv, so, sdo, sdq, sdk, sdv;  // operand layouts
};

// Rows [first, S) of a batch see no key; T_i as above.
struct MaskedRows {
    int S, W, len;
    bool causal;
    __device__ int first() const { return len <= 0 ? 0 : (W > 0 ? min(S, len + W - 1) : S); }
    __device__ int tlo(int i) const { return W > 0 ? max(i - W + 1, 0) : 0; }
    __device__ int thi(int i) const { return causal ? i : S - 1; }
    __device__ int count(int i) const { return thi(i) - tlo(i) + 1 + len; }
};

__device__ __forceinline__ MaskedRows masked_rows(const MaskedArgs& a, int b) {
    return MaskedRows{a.S, a.window, min(max(a.kv_len[b], 0), a.S), a.causal != 0};
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
}

template <typename T> __device__ __forceinline__ float ld(const T* p) { return (float)*p; }

// VEC consecutive elements of a row (one 16-byte access, or a single one).
template <typename T, int VEC> struct alignas(VEC * sizeof(T)) Pack {
    T x[VEC];
};

// Lanes that span a row of D elements, VEC to a lane: a power of two, so that
// the rows a workgroup holds at once divide its threads.
__host__ __device__ constexpr int row_lanes(int D, int VEC) {
    int n = 1;
    while (n * VEC < D) n *= 2;
    return n;
}

// The forward's share of a row: one 128-byte line per workgroup where rows
// are read in vectors, so that many groups of lanes share the rows.
__host__ __device__ constexpr int fwd_lanes(int D, int VEC) {
    const int n = row_lanes(D, VEC), most = VEC > 1 ? 8 : 64;
    return n < most ? n : most;
}

// Forward: O_i = mean of V over T_i for every masked row, all query heads of
// the kv head.  Bound by the latency of reading [0, len) and the window.
// Workgroup = (G rows, batch x kv head, a line's columns), G = NT /
// fwd_lanes (128 rows of 64 bf16 columns with 1024 threads): group g of fwd_lanes threads sums
// every G-th row of T_r0 (r0 the workgroup's first masked row), eight rows'
// loads in flight, the groups' sums are added through LDS, and group g then
// owns row r0 + g, whose T differs from T_r0 by one entering and one leaving
// row per step: a prefix sum over the groups.  All sums in double.  One thread
// per column walking the rows alone took 245 us at B 3, Hkv 1, S 1000, D 256,
// window 512 with lengths down to 390; whole rows to a workgroup 16; this 10.
template <typename T, int VEC, int NT>
__global__ __launch_bounds__(NT) void attn_fwd_masked_rows(MaskedArgs a) {
    typedef Pack<T, VEC> P;
    __shared__ double part[VEC][NT], seg[NT];
    const int S = a.S, D = a.D, tid = threadIdx.x;
    const int lanes = fwd_lanes(D, VEC), G = NT / lanes, g = tid / lanes;
    const int d = ((int)blockIdx.z * lanes + tid % lanes) * VEC;
    const int bk = blockIdx.y, b = bk / a.Hkv, hk = bk % a.Hkv;
    const MaskedRows mr = masked_rows(a, b);
    const int r0 = max((int)blockIdx.x * G, mr.first()), r1 = min((int)blockIdx.x * G + G, S);
    if (r0 >= r1) return;
    const bool live = d < D;  // D is a multiple of VEC
    const T* V = (const T*)a.v + a.sv.at(b, hk) + (live ? d : 0);
    const int64_t lv = a.sv.s;
    double acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.0;
    // T_r0 as one list: [0, len), then [lo, hi].
    const int lo = mr.tlo(r0), total = mr.count(r0);
    constexpr int U = 8;
    for (int n0 = g; n0 < total; n0 += U * G) {
        P x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = min(n0 + u * G, total - 1);
            x[u] = *reinterpret_cast<const P*>(V + (int64_t)(n < mr.len ? n : lo + n - mr.len) * lv);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (n0 + u * G < total)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[e] += (double)(float)x[u].x[e];
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) part[e][tid] = acc[e];
    __syncthreads();
    // A column's G values are handled by Q = G / VEC threads, VEC values each:
    // thread (q, element ce, lane cl).
    const int cols = lanes * VEC, q = tid / cols, ce = (tid % cols) / lanes, cl = tid % lanes;
    const int Q = NT / cols;
    double* mine = &part[ce][q * VEC * lanes + cl];  // values s * lanes apart
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < VEC; ++s) sum += mine[s * lanes];
    seg[tid] = sum;
    __syncthreads();
    sum = 0.0;  // over T_r0
    for (int s = 0; s < Q; ++s) sum += seg[s * cols + tid % cols];
    // Row i = r0 + g: what entered T since row i - 1 less what left it.
    const int i = r0 + g;
    const bool in = i < r1;
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.0;
    if (in && g > 0) {
        const P add = *reinterpret_cast<const P*>(V + (int64_t)mr.thi(i) * lv);
        const P sub = *reinterpret_cast<const P*>(V + (int64_t)mr.tlo(i - 1) * lv);
        const bool enters = mr.thi(i) > mr.thi(i - 1), leaves = mr.tlo(i) > mr.tlo(i - 1);
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            acc[e] = (enters ? (double)(float)add.x[e] : 0.0) - (leaves ? (double)(float)sub.x[e] : 0.0);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) part[e][tid] = acc[e];
    __syncthreads();
    double d_seg = 0.0;
#pragma unroll
    for (int s = 0; s < VEC; ++s) d_seg += mine[s * lanes];
    seg[tid] = d_seg;
    __syncthreads();
    for (int s = 0; s < q; ++s) sum += seg[s * cols + tid % cols];
#pragma unroll
    for (int s = 0; s < VEC; ++s) {
        sum += mine[s * lanes];
        mine[s * lanes] = sum;
    }
    __syncthreads();
    if (!in || !live) return;
    const double n = (double)mr.count(i);
    P o;
#pragma unroll
    for (int e = 0; e < VEC; ++e) o.x[e] = (T)(float)(part[e][tid] / n);
    for (int h = hk * a.group; h < (hk + 1) * a.group; ++h)
        *reinterpret_cast<P*>((T*)a.o + a.so.at(b, h) + (int64_t)i * a.so.s + d) = o;
}

// This lane's columns lane + 64 c (c < 4, D <= 256) of a row.
template <typename T>
__device__ __forceinline__ void load_row4(const T* row, int D, float (&x)[4]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = lane + 64 * c < D ? (float)row[lane + 64 * c] : 0.f;
}
__device__ __forceinline__ float dot4(const float (&x)[4], const float (&y)[4]) {
    return x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
}

// Backward, dQ of masked rows (and the row terms the dK/dV pass reads): a
// workgroup per (64 rows, batch x query head), each wave 16 rows in turn.
// Workgroups without masked rows return at once (the common case).
template <typename T>
__device__ void masked_dq_row(const MaskedArgs& a, const MaskedRows& mr, int b, int h, int i);

// Bit i of the result: row r0 + i of dO (n <= 16 rows) holds a non-zero.  The
// rows' loads are in flight together (one row after the other, 16 memory
// round trips per wave, took 40 us at the shape above; now 5).
template <typename T, int VEC>
__device__ __forceinline__ unsigned nonzero_rows(const T* dO, int64_t ld, int D, int n) {
    typedef Pack<T, VEC> P;
    const int lane = threadIdx.x & 63;
    unsigned m = 0;
    if constexpr (VEC > 1) {
        const int lanes = row_lanes(D, VEC), rpw = 64 / lanes, q = lane / lanes, d = (lane % lanes) * VEC;
        const unsigned long long row = lanes == 64 ? ~0ull : (1ull << lanes) - 1;
        const T* p = dO + (d < D ? d : 0);
        for (int r0 = 0; r0 < n; r0 += 8 * rpw) {
            P x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = *reinterpret_cast<const P*>(p + (int64_t)min(r0 + u * rpw + q, n - 1) * ld);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                bool nz = false;
#pragma unroll
                for (int e = 0; e < VEC; ++e) nz |= (float)x[u].x[e] != 0.f;
                const unsigned long long hit = __ballot(nz && d < D);
                if (!hit) continue;
                for (int r = 0; r < rpw && r0 + u * rpw + r < n; ++r)
                    if (hit >> (r * lanes) & row) m |= 1u << (r0 + u * rpw + r);
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            bool nz = false;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                nz |= u < n && lane + 64 * c < D && (float)dO[(int64_t)min(u, n - 1) * ld + min(lane + 64 * c, D - 1)] != 0.f;
            if (__any(nz)) m |= 1u << u;
        }
    }
    return m;
}

template <typename T, int VEC>
__global__ __launch_bounds__(256) void attn_bwd_masked_dq(MaskedArgs a) {
    const int bh = blockIdx.y, b = bh / a.Hq, h = bh % a.Hq;
    const MaskedRows mr = masked_rows(a, b);
    const int r0 = max((int)blockIdx.x * 64 + 16 * (int)(threadIdx.x >> 6), mr.first());
    const int r1 = min((int)blockIdx.x * 64 + 16 * (int)(threadIdx.x >> 6) + 16, a.S);
    if (r0 >= r1) return;
    const unsigned active =
        nonzero_rows<T, VEC>((const T*)a.dO + a.sdo.at(b, h) + (int64_t)r0 * a.sdo.s, a.sdo.s, a.D, r1 - r0);
    const int lane = threadIdx.x & 63;
    if (lane < r1 - r0) a.row_active[((int64_t)b * a.Hq + h) * a.S + r0 + lane] = active >> lane & 1;
    // a row whose dO is zero has dq_i = 0, as the main pass left it
    for (int i = r0; i < r1; ++i)
        if (active >> (i - r0) & 1) masked_dq_row<T>(a, mr, b, h, i);
}

template <typename T>
__device__ void masked_dq_row(const MaskedArgs& a, const MaskedRows& mr, int b, int h, int i) {
    const int S = a.S, D = a.D, lane = threadIdx.x & 63, hk = h / a.group;
    const int64_t ri = ((int64_t)b * a.Hq + h) * S + i;  // row-term index (contiguous scratch)
    float g[4], o[4];
    load_row4((const T*)a.dO + a.sdo.at(b, h) + (int64_t)i * a.sdo.s, D, g);
    load_row4((const T*)a.o + a.so.at(b, h) + (int64_t)i * a.so.s, D, o);
    const float dl = wave_sum(dot4(g, o));
    if (lane == 0) a.row_delta[ri] = dl;
    const T* K = (const T*)a.k + a.sk.at(b, hk);
    const T* V = (const T*)a.v + a.sv.at(b, hk);
    const float inv_c = 1.f / (float)mr.count(i);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    auto key = [&](int j) {
        float vj[4], kj[4];
        load_row4(V + (int64_t)j * a.sv.s, D, vj);
        load_row4(K + (int64_t)j * a.sk.s, D, kj);
        const float ds = (wave_sum(dot4(g, vj)) - dl) * inv_c;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] += ds * kj[c];
    };
    for (int j = 0; j < mr.len; ++j) key(j);
    for (int j = mr.tlo(i); j <= mr.thi(i); ++j) key(j);
    float* dq = a.dq + a.sdq.at(b, h) + (int64_t)i * a.sdq.s;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < D) dq[lane + 64 * c] = acc[c] * a.scale;
}

// Backward, dK/dV contributions of masked rows, added to what the main pass
// wrote: a workgroup per (64 keys, batch x kv head), each wave 16 keys in
// turn.  The rows that hold key j in T_i: all masked rows for j < len, else
// rows j .. j + W - 1 (causal window) among the masked ones; active rows are
// found 64 at a time by ballot.  Batches without masked rows return at once.
template <typename T>
__device__ void masked_dkdv_key(const MaskedArgs& a, const MaskedRows& mr, int b, int hk, int j);

template <typename T>
__global__ __launch_bounds__(256) void attn_bwd_masked_dkdv(MaskedArgs a) {
    const int bk = blockIdx.y, b = bk / a.Hkv, hk = bk % a.Hkv;
    const MaskedRows mr = masked_rows(a, b);
    if (mr.first() >= a.S) return;
    // No active row among the group's heads (their padded positions carry no
    // loss): nothing to add.  Found by all threads together; each wave looking
    // through the rows for each of its keys took 48 us at the shape above.
    bool any = false;
    for (int h = hk * a.group; h < (hk + 1) * a.group; ++h) {
        const int* act = a.row_active + ((int64_t)b * a.Hq + h) * a.S;
#pragma unroll 4
        for (int i = mr.first() + (int)threadIdx.x; i < a.S; i += 256) any |= act[i] != 0;
    }
    if (!__syncthreads_or(any)) return;
    const int j0 = (int)blockIdx.x * 64 + 16 * (int)(threadIdx.x >> 6);
    for (int j = j0; j < min(j0 + 16, a.S); ++j) masked_dkdv_key<T>(a, mr, b, hk, j);
}

template <typename T>
__device__ void masked_dkdv_key(const MaskedArgs& a, const MaskedRows& mr, int b, int hk, int j) {
    const int S = a.S, D = a.D, lane = threadIdx.x & 63;
    int i_lo = mr.first(), i_hi = S - 1;
    if (j >= mr.len) {
        if (mr.causal) i_lo = max(i_lo, j);
        if (mr.W > 0) i_hi = min(i_hi, j + mr.W - 1);
    }
    if (i_lo > i_hi) return;
    float vj[4];
    load_row4((const T*)a.v + a.sv.at(b, hk) + (int64_t)j * a.sv.s, D, vj);
    float ak[4] = {0.f, 0.f, 0.f, 0.f}, av[4] = {0.f, 0.f, 0.f, 0.f};
    bool any = false;
    for (int h = hk * a.group; h < (hk + 1) * a.group; ++h) {
        const int64_t bh = (int64_t)b * a.Hq + h;
        for (int c0 = i_lo; c0 <= i_hi; c0 += 64) {
            const int ic = c0 + lane;
            unsigned long long m = __ballot(ic <= i_hi && a.row_active[bh * S + ic] != 0);
            while (m) {
                const int i = c0 + __builtin_ctzll(m);
                m &= m - 1;
                any = true;
                const int64_t ri = bh * S + i;
                float g[4], q[4];
                load_row4((const T*)a.dO + a.sdo.at(b, h) + (int64_t)i * a.sdo.s, D, g);
                load_row4((const T*)a.q + a.sq.at(b, h) + (int64_t)i * a.sq.s, D, q);
                const float inv_c = 1.f / (float)mr.count(i);
                const float ds = (wave_sum(dot4(g, vj)) - a.row_delta[ri]) * inv_c;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    av[c] += g[c] * inv_c;
                    ak[c] += ds * q[c];
                }
            }
        }
    }
    if (!any) return;
    float* dk = a.dk + a.sdk.at(b, hk) + (int64_t)j * a.sdk.s;
    float* dv = a.dv + a.sdv.at(b, hk) + (int64_t)j * a.sdv.s;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < D) {
            dk[lane + 64 * c] += ak[c] * a.scale;
            dv[lane + 64 * c] += av[c];
        }
}

MaskedArgs masked_args(const AttnShape& s) {
    MaskedArgs a{};
    a.kv_len = s.kv_len;
    a.B = (int)s.B;
    a.Hq = (int)s.Hq;
    a.Hkv = (int)s.Hkv;
    a.S = (int)s.S;
    a.D = (int)s.D;
    a.group = (int)(s.Hq / s.Hkv);
    a.window = s.window;
    a.causal = s.causal ? 1 : 0;
    a.scale = s.scale;
    a.sq = s.q;
    a.sk = s.k;
    a.sv = s.v;
    a.so = s.o;
    a.sdo = s.dO;
    a.sdq = s.dq;
    a.sdk = s.dk;
    a.sdv = s.dv;
    return a;
}

// Elements per access of a row: 16 bytes where every row starts on 16 bytes.
// Strides the caller gives are multiples of 16 bytes (checked by the C ABI);
// contiguous rows are when D is.
int row_vec(const AttnShape& s) {
    const int w = s.bf16 ? 8 : 4;
    return s.D % w == 0 ? w : 1;
}

}  // namespace

size_t masked_rows_workspace_bytes(const AttnShape& s) {
    if (!s.kv_len) return 0;
    const size_t rows = static_cast<size_t>(s.B * s.Hq * s.S);
    return ((rows * 4 + 255) & ~static_cast<size_t>(255)) * 2;
}

hipError_t launch_fwd_masked_rows(const AttnShape& s, const void* v, void* o, hipStream_t st) {
    if (!s.kv_len) return hipSuccess;
    MaskedArgs a = masked_args(s);
    a.v = v;
    a.o = o;
    // Short sequences take 256 threads: in a call without such rows every
    // workgroup returns at once, and 1024 threads and 72 KB of LDS for each cost
    // 0.1 to 0.2 us more (B 4, Hq 12, S 128, bf16 forward 8.52 -> 8.36); with
    // such rows fewer of them share T_r0 (14.0 -> 11.7, at S 500, D 256 34.9 ->
    // 31.4).  Past 512 rows the sum over T_r0 outweighs that.
    const int vec = row_vec(s), lanes = fwd_lanes(a.D, vec), nt = s.S <= 512 ? 256 : 1024, rows = nt / lanes;
    const dim3 grid((unsigned)((s.S + rows - 1) / rows), (unsigned)(s.B * s.Hkv),
                    (unsigned)((a.D + lanes * vec - 1) / (lanes * vec)));
#define MFT_MASKED_FWD(T, VEC)                                                                          \
    do {                                                                                                \
        if (nt == 256)                                                                                  \
            hipLaunchKernelGGL((attn_fwd_masked_rows<T, VEC, 256>), grid, dim3(256), 0, st, a);         \
        else                                                                                            \
            hipLaunchKernelGGL((attn_fwd_masked_rows<T, VEC, 1024>), grid, dim3(1024), 0, st, a);       \
    } while (0)
    if (s.bf16) {
        if (vec > 1) MFT_MASKED_FWD(bf16, 8);
        else MFT_MASKED_FWD(bf16, 1);
    } else {
        if (vec > 1) MFT_MASKED_FWD(float, 4);
        else MFT_MASKED_FWD(float, 1);
    }
#undef MFT_MASKED_FWD
    return hipGetLastError();
}

hipError_t launch_bwd_masked_rows(const AttnShape& s, const void* q, const void* k, const void* v, const void* o,
                                  const void* dO, float* dq, float* dk, float* dv, void* scratch, hipStream_t st) {
    if (!s.kv_len) return hipSuccess;
    MaskedArgs a = masked_args(s);
    a.q = q;
    a.k = k;
    a.v = v;
    a.o = const_cast<void*>(o);
    a.dO = dO;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    const size_t half = masked_rows_workspace_bytes(s) / 2;
    a.row_delta = static_cast<float*>(scratch);
    a.row_active = reinterpret_cast<int*>(static_cast<char*>(scratch) + half);
    const dim3 gq((unsigned)((s.S + 63) / 64), (unsigned)(s.B * s.Hq));
    const dim3 gk((unsigned)((s.S + 63) / 64), (unsigned)(s.B * s.Hkv));
    const bool vec = row_vec(s) > 1;
    if (s.bf16) {
        if (vec)
            hipLaunchKernelGGL((attn_bwd_masked_dq<bf16, 8>), gq, dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((attn_bwd_masked_dq<bf16, 1>), gq, dim3(256), 0, st, a);
        hipLaunchKernelGGL(attn_bwd_masked_dkdv<bf16>, gk, dim3(256), 0, st, a);
    } else {
        if (vec)
            hipLaunchKernelGGL((attn_bwd_masked_dq<float, 4>), gq, dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((attn_bwd_masked_dq<float, 1>), gq, dim3(256), 0, st, a);
        hipLaunchKernelGGL(attn_bwd_masked_dkdv<float>, gk, dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace mft
