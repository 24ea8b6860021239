// Element-wise and rank-r kernels of the LoRA linear layer (C ABI in include/mft/lora.h,
// GEMMs in lora_capi.cpp).
//
//   lora_round_bf16   fp32 -> bf16 operand staging for the bf16 MFMA GEMMs;
//                     HBM-bound, 6 bytes per element, 16-byte vectors.
//   lora_fill_bias    y = broadcast(bias) ahead of a beta = 1 GEMM (the
//                     reference's add(y, b), nn/lora_linear.cpp:349-351).
//   lora_merge        apply_lora_delta_to_base (nn/lora_linear.cpp:108-138):
//                     per element a rank-long double dot product, then one
//                     fp32 multiply and add, element for element as the
//                     reference rounds them (fp contract off).
//   lora_rowdot, lora_coldot   u, g and the adapters' gradients; each below.
//   lora_update       a slice's low-rank update of y or dx by itself.
#include <hip/hip_runtime.h>

#include "lora_kernels.h"

namespace mft {
namespace {

__device__ __forceinline__ uint16_t bf16_bits_rne(float x) {
    uint32_t bits = __float_as_uint(x);
    bits += 0x7FFFu + ((bits >> 16) & 1u);
    return (uint16_t)(bits >> 16);
}

__device__ __forceinline__ float bf16_bits_to_float(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__global__ __launch_bounds__(256) void lora_round_bf16_vec(const float4* __restrict__ src, uint2* __restrict__ dst,
                                                           int64_t n4) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        const float4 v = src[i];
        dst[i] = make_uint2((uint32_t)bf16_bits_rne(v.x) | ((uint32_t)bf16_bits_rne(v.y) << 16),
                            (uint32_t)bf16_bits_rne(v.z) | ((uint32_t)bf16_bits_rne(v.w) << 16));
    }
}

__global__ __launch_bounds__(256) void lora_round_bf16_tail(const float* __restrict__ src,
                                                            uint16_t* __restrict__ dst, int64_t i0, int64_t n) {
    const int64_t i = i0 + (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = bf16_bits_rne(src[i]);
}

__global__ __launch_bounds__(256) void lora_fill_bias_kernel(float* __restrict__ y, const float* __restrict__ bias,
                                                             int64_t N, int64_t out) {
    const int64_t total = N * out;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256)
        y[i] = bias[i % out];
}

// One thread per (i, o) element of the slice's [in, cols] block; o runs
// fastest so that B's row and W's row (untransposed layouts) are read in
// consecutive addresses.  Every multiply and add is rounded on its own, as
// the reference's are (fp contract off in this kernel only).
__global__ __launch_bounds__(256) void lora_merge_kernel(LoraMergeArgs a) {
#pragma clang fp contract(off)
    const int64_t total = a.in * a.cols;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e / a.cols, o = e % a.cols;
        double delta = 0.0;
        for (int64_t r = 0; r < a.rank; ++r) {
            const float av = a.a_transposed ? a.A[r * a.in + i] : a.A[i * a.rank + r];
            const float bv = a.b_transposed ? a.B[o * a.rank + r] : a.B[r * a.cols + o];
            delta += (double)av * (double)bv;
        }
        const int64_t c = a.col0 + o;
        const int64_t w = a.w_transposed ? c * a.in + i : i * a.out + c;
        if (a.w_bf16) {
            uint16_t* W = static_cast<uint16_t*>(a.W);
            W[w] = bf16_bits_rne(bf16_bits_to_float(W[w]) + a.sign_scale * (float)delta);
        } else {
            float* W = static_cast<float*>(a.W);
            W[w] = W[w] + a.sign_scale * (float)delta;
        }
    }
}

// ---- rank-r products (r is small, the inner dimension long) ----
//
// lora_rowdot: out[n, j] = alpha sum_k M[n, k] P(k, j).  A workgroup owns
// kRowsPerWg rows; its 256 threads stride jointly over k (thread t: columns
// VEC t + 256 VEC i) and each keeps kRowsPerWg x 8 partial sums (one 8-wide
// block of j at a time), so each P(k, j) it loads serves kRowsPerWg rows.  The
// 256 partials of each (row, j) are summed through LDS in a fixed order
// (deterministic).  M is read once per 8-wide block of j: HBM-bound for r <= 8.
// PV: P is k-contiguous and aligned, so its loads are 16 bytes wide like M's
// (four times as many 4-byte ones kept the load path busier than M did: [4096
// x 6912], r 8, with the bf16 copy 52 -> 37 us, 4.6 TB/s).
constexpr int kRowsPerWg = 8, kJB = 8;

template <int VEC, bool PV>
__global__ __launch_bounds__(256) void lora_rowdot_kernel(LoraRowDot a) {
    constexpr int NV = kRowsPerWg * kJB;  // partial sums per thread
    __shared__ float red[NV][257];
    __shared__ float red2[4][NV];
    const int t = threadIdx.x;
    const int64_t n0 = (int64_t)blockIdx.x * kRowsPerWg;
    for (int jb = 0; jb < a.r; jb += kJB) {
        float acc[kRowsPerWg][kJB];
#pragma unroll
        for (int i = 0; i < kRowsPerWg; ++i)
#pragma unroll
            for (int j = 0; j < kJB; ++j) acc[i][j] = 0.f;
        for (int64_t k = (int64_t)VEC * t; k < a.K; k += 256 * VEC) {
            float p[VEC][kJB];
#pragma unroll
            for (int j = 0; j < kJB; ++j) {
                // clamped index, so the load needs no branch; the select zeroes j >= r
                const int jj = jb + j < a.r ? jb + j : a.r - 1;
                float pv[VEC];
                if constexpr (PV) {
                    const float4 q = *reinterpret_cast<const float4*>(a.P + k + (int64_t)jj * a.pj);
                    pv[0] = q.x, pv[1 % VEC] = q.y, pv[2 % VEC] = q.z, pv[3 % VEC] = q.w;
                } else {
#pragma unroll
                    for (int v = 0; v < VEC; ++v) pv[v] = a.P[(k + v) * a.pk + (int64_t)jj * a.pj];
                }
#pragma unroll
                for (int v = 0; v < VEC; ++v) p[v][j] = jb + j < a.r ? pv[v] : 0.f;
            }
            float mv[kRowsPerWg][VEC];
#pragma unroll
            for (int i = 0; i < kRowsPerWg; ++i) {
                const int64_t n = n0 + i < a.rows ? n0 + i : a.rows - 1;
                const float* m = a.M + n * a.ldm + k;
                if (VEC == 4) {
                    const float4 q = *reinterpret_cast<const float4*>(m);
                    mv[i][0] = q.x, mv[i][1 % VEC] = q.y, mv[i][2 % VEC] = q.z, mv[i][3 % VEC] = q.w;
                } else {
                    mv[i][0] = m[0];
                }
            }
            if (a.mb && jb == 0) {  // the bf16 copy of M, from the first j-block's loads
#pragma unroll
                for (int i = 0; i < kRowsPerWg; ++i) {
                    if (n0 + i >= a.rows) continue;
                    uint16_t* d = a.mb + (n0 + i) * a.ldb + k;
                    if (VEC == 4)
                        *reinterpret_cast<uint2*>(d) =
                            make_uint2((uint32_t)bf16_bits_rne(mv[i][0]) | ((uint32_t)bf16_bits_rne(mv[i][1 % VEC]) << 16),
                                       (uint32_t)bf16_bits_rne(mv[i][2 % VEC]) |
                                           ((uint32_t)bf16_bits_rne(mv[i][3 % VEC]) << 16));
                    else
                        d[0] = bf16_bits_rne(mv[i][0]);
                }
            }
#pragma unroll
            for (int i = 0; i < kRowsPerWg; ++i)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
#pragma unroll
                    for (int j = 0; j < kJB; ++j) acc[i][j] += mv[i][v] * p[v][j];
        }
#pragma unroll
        for (int i = 0; i < kRowsPerWg; ++i)
#pragma unroll
            for (int j = 0; j < kJB; ++j) red[i * kJB + j][t] = acc[i][j];
        __syncthreads();
        {
            // quarter q of the 256 partials of value e, then the 4 quarters
            const int e = t % NV, q = t / NV;
            float s = 0.f;
            for (int l = 0; l < 64; ++l) s += red[e][64 * q + l];
            red2[q][e] = s;
        }
        __syncthreads();
        if (t < NV) {
            const int i = t / kJB, j = t % kJB;
            const float s = (red2[0][t] + red2[1][t]) + (red2[2][t] + red2[3][t]);
            const int64_t n = n0 + i;
            if (n < a.rows && jb + j < a.r) a.out[n * a.ldo + jb + j] = a.alpha * s;
        }
        __syncthreads();
    }
}

// lora_coldot: per chunk c of rows and column k, partial[c][j][k] = sum over
// the chunk's rows of M[n, k] V[n, j]; one wave per (64 VEC columns, chunk),
// the row of V is the same for the whole wave.  The chunk height is chosen so
// that about 2048 waves run (lora_coldot_chunk, lora_kernels.h).  Then
// lora_coldot_reduce sums the chunks in a fixed order.  The partials are
// contiguous in k, a lane's next to its neighbour's (with k outside j each of
// a wave's 32 stores touched 64 lines), and V comes through scalar loads, a
// row at a time (M, V and the partials do not overlap; unless the compiler is
// told, it loads every value of V as a vector).  4096 rows, r 8: K 1152 19.5 ->
// 10.1 us, K 6912 34.5 -> 20.5, 5.5 TB/s of M.

// acc += M[n, k ..]^T V[n, j0 ..] over rows r0 .. r1 - 1, j < nj (NJ: nj where
// it is known, so that a row of V is one scalar load; 0 otherwise).
template <int VEC, int NJ>
__device__ __forceinline__ void coldot_rows(const float* __restrict__ m, int64_t ldm, const float* __restrict__ V,
                                            int64_t ldv, int64_t r0, int64_t r1, int nj, float (&acc)[VEC][kJB]) {
    constexpr int J = NJ ? NJ : kJB;
#pragma unroll 8
    for (int64_t n = r0; n < r1; ++n) {
        const float* row = V + n * ldv;
        float vv[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const float x = row[NJ || j < nj ? j : nj - 1];
            vv[j] = NJ || j < nj ? x : 0.f;
        }
        float mv[VEC];
        if (VEC == 4) {
            const float4 q = *reinterpret_cast<const float4*>(m + n * ldm);
            mv[0] = q.x, mv[1 % VEC] = q.y, mv[2 % VEC] = q.z, mv[3 % VEC] = q.w;
        } else {
            mv[0] = m[n * ldm];
        }
#pragma unroll
        for (int v = 0; v < VEC; ++v)
#pragma unroll
            for (int j = 0; j < J; ++j) acc[v][j] += mv[v] * vv[j];
    }
}

template <int VEC>
__global__ __launch_bounds__(64) void lora_coldot_kernel(LoraColDot a, const float* __restrict__ M,
                                                         const float* __restrict__ V, float* __restrict__ partial,
                                                         int64_t chunk) {
    const int64_t k = ((int64_t)blockIdx.x * 64 + threadIdx.x) * VEC;
    const int64_t c = blockIdx.y;
    const int64_t r0 = c * chunk, r1 = r0 + chunk < a.rows ? r0 + chunk : a.rows;
    const bool live = k < a.K;
    const float* m = M + (live ? k : 0);  // lanes past K sum a column that they do not store
    for (int jb = 0; jb < a.r; jb += kJB) {
        float acc[VEC][kJB];
#pragma unroll
        for (int v = 0; v < VEC; ++v)
#pragma unroll
            for (int j = 0; j < kJB; ++j) acc[v][j] = 0.f;
        if (a.r - jb >= kJB)
            coldot_rows<VEC, kJB>(m, a.ldm, V + jb, a.ldv, r0, r1, kJB, acc);
        else if (a.r - jb == 4)
            coldot_rows<VEC, 4>(m, a.ldm, V + jb, a.ldv, r0, r1, 4, acc);
        else
            coldot_rows<VEC, 0>(m, a.ldm, V + jb, a.ldv, r0, r1, a.r - jb, acc);
        if (live) {
            float* part = partial + (c * a.r + jb) * a.K + k;
#pragma unroll
            for (int j = 0; j < kJB; ++j) {
                if (jb + j >= a.r) break;
                if (VEC == 4)
                    *reinterpret_cast<float4*>(part + j * a.K) =
                        make_float4(acc[0][j], acc[1 % VEC][j], acc[2 % VEC][j], acc[3 % VEC][j]);
                else
                    part[j * a.K] = acc[0][j];
            }
        }
    }
}

// A workgroup owns 64 consecutive output values; its wave l sums chunks l,
// l + 8, ... in order, then the eight sums combine in a fixed tree
// (deterministic).  Eight chunks' loads are in flight together: one after the
// other they cost a memory round trip each (256 chunks of 1152 x 8 8.0 ->
// 5.3 us, 64 of 6912 x 8 9.1 -> 5.0).
constexpr int kColRed = 8;
__global__ __launch_bounds__(64 * kColRed) void lora_coldot_reduce(LoraColDot a, int64_t chunks) {
    constexpr int B = 8;
    __shared__ float sums[kColRed][64];
    const int le = threadIdx.x % 64, l = threadIdx.x / 64;
    const int64_t total = a.K * a.r, e = (int64_t)blockIdx.x * 64 + le;
    const float* src = a.partial + (e < total ? e : total - 1);
    float s = 0.f;
    for (int64_t c = l; c < chunks; c += kColRed * B) {
        float x[B];
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int64_t cq = c + kColRed * q;
            x[q] = src[(cq < chunks ? cq : chunks - 1) * total];
        }
#pragma unroll
        for (int q = 0; q < B; ++q) s += c + kColRed * q < chunks ? x[q] : 0.f;
    }
    sums[l][le] = s;
    __syncthreads();
    if (l != 0 || e >= total) return;
    float v[kColRed];
#pragma unroll
    for (int i = 0; i < kColRed; ++i) v[i] = sums[i][le];
#pragma unroll
    for (int o = kColRed / 2; o >= 1; o >>= 1)
#pragma unroll
        for (int i = 0; i < o; ++i) v[i] += v[i + o];
    const int64_t j = e / a.K, k = e % a.K;
    a.out[k * a.ok + j * a.oj] = a.alpha * v[0];
}

// lora_update: a thread holds one column of kUpdRows rows, loads its column of
// B once for them, and takes the rows of U as scalars (U, B and C do not
// overlap).  Bound by the latency of its loads: 3 us for 64 rows of 768 columns
// at rank 8, where a tile of the general product takes 5.5.
constexpr int kUpdRows = 8;
__global__ __launch_bounds__(256) void lora_update_kernel(LoraUpdate a, const float* __restrict__ U,
                                                          const float* __restrict__ B, float* __restrict__ C,
                                                          unsigned col_blocks) {
    const int64_t o = (int64_t)(blockIdx.x % col_blocks) * 256 + threadIdx.x, oc = min(o, a.cols - 1);
    const int64_t n0 = (int64_t)(blockIdx.x / col_blocks) * kUpdRows;
    const int rows = (int)min<int64_t>(kUpdRows, a.rows - n0);
    const float* u[kUpdRows];  // rows past the end repeat the last one
    float c[kUpdRows], acc[kUpdRows];
#pragma unroll
    for (int i = 0; i < kUpdRows; ++i) {
        const int64_t n = n0 + min(i, rows - 1);
        u[i] = U + n * a.ldu;
        c[i] = C[n * a.ldc + oc];
        acc[i] = 0.f;
    }
    const float* b = B + (a.bt ? oc * a.r : oc);
    const int64_t step = a.bt ? 1 : a.cols;
    int k = 0;
    for (; k + 4 <= a.r; k += 4) {
        float bv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = b[(k + e) * step];
#pragma unroll
        for (int i = 0; i < kUpdRows; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i] = fmaf(u[i][k + e], bv[e], acc[i]);
    }
    for (; k < a.r; ++k) {
        const float bv = b[k * step];
#pragma unroll
        for (int i = 0; i < kUpdRows; ++i) acc[i] = fmaf(u[i][k], bv, acc[i]);
    }
    if (o >= a.cols) return;
#pragma unroll
    for (int i = 0; i < kUpdRows; ++i)
        if (i < rows) C[(n0 + i) * a.ldc + o] = fmaf(a.alpha, acc[i], c[i]);
}

__global__ __launch_bounds__(256) void lora_pack_kmajor_kernel(const float* __restrict__ P, int64_t pk, int64_t pj,
                                                               int64_t K, int r, float* __restrict__ dst) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= K * r) return;
    const int64_t j = e / K, k = e % K;
    dst[e] = P[k * pk + j * pj];
}

unsigned grid_for(int64_t work) {
    const int64_t g = (work + 255) / 256;
    return (unsigned)(g < 1 ? 1 : g > 8192 ? 8192 : g);
}

}  // namespace

hipError_t launch_lora_round_bf16(const float* src, uint16_t* dst, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const bool vec = ((uintptr_t)src % 16 == 0) && ((uintptr_t)dst % 8 == 0);
    const int64_t n4 = vec ? n / 4 : 0;
    if (n4 > 0)
        hipLaunchKernelGGL(lora_round_bf16_vec, dim3(grid_for(n4)), dim3(256), 0, st,
                           reinterpret_cast<const float4*>(src), reinterpret_cast<uint2*>(dst), n4);
    const int64_t rest = n - 4 * n4;
    if (rest > 0)
        hipLaunchKernelGGL(lora_round_bf16_tail, dim3((unsigned)((rest + 255) / 256)), dim3(256), 0, st, src, dst,
                           4 * n4, n);
    return hipGetLastError();
}

hipError_t launch_lora_fill_bias(float* y, const float* bias, int64_t N, int64_t out, hipStream_t st) {
    if (N <= 0 || out <= 0) return hipSuccess;
    hipLaunchKernelGGL(lora_fill_bias_kernel, dim3(grid_for(N * out)), dim3(256), 0, st, y, bias, N, out);
    return hipGetLastError();
}

hipError_t launch_lora_rowdot(const LoraRowDot& a, hipStream_t st) {
    if (a.rows <= 0 || a.r <= 0) return hipSuccess;
    const dim3 grid((unsigned)((a.rows + kRowsPerWg - 1) / kRowsPerWg));
    const bool vec = a.K % 4 == 0 && a.ldm % 4 == 0 && (uintptr_t)a.M % 16 == 0 &&
                     (!a.mb || (a.ldb % 4 == 0 && (uintptr_t)a.mb % 8 == 0));
    const bool pvec = a.pk == 1 && a.pj % 4 == 0 && (uintptr_t)a.P % 16 == 0;
    if (vec && pvec)
        hipLaunchKernelGGL((lora_rowdot_kernel<4, true>), grid, dim3(256), 0, st, a);
    else if (vec)
        hipLaunchKernelGGL((lora_rowdot_kernel<4, false>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((lora_rowdot_kernel<1, false>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_lora_pack_kmajor(const float* P, int64_t pk, int64_t pj, int64_t K, int r, float* dst,
                                   hipStream_t st) {
    if (K <= 0 || r <= 0) return hipSuccess;
    hipLaunchKernelGGL(lora_pack_kmajor_kernel, dim3((unsigned)((K * r + 255) / 256)), dim3(256), 0, st, P, pk, pj,
                       K, r, dst);
    return hipGetLastError();
}

int64_t lora_coldot_partial_floats(int64_t rows, int64_t K, int r) {
    const int64_t chunk = lora_coldot_chunk(rows, K);
    return (rows + chunk - 1) / chunk * K * r;
}

hipError_t launch_lora_update(const LoraUpdate& a, hipStream_t st) {
    if (a.rows <= 0 || a.cols <= 0 || a.r <= 0) return hipSuccess;
    const unsigned col_blocks = (unsigned)((a.cols + 255) / 256);
    const dim3 grid(col_blocks * (unsigned)((a.rows + kUpdRows - 1) / kUpdRows));
    hipLaunchKernelGGL(lora_update_kernel, grid, dim3(256), 0, st, a, a.U, a.B, a.C, col_blocks);
    return hipGetLastError();
}

hipError_t launch_lora_coldot(const LoraColDot& a, hipStream_t st) {
    if (a.K <= 0 || a.r <= 0) return hipSuccess;
    const int64_t chunk = lora_coldot_chunk(a.rows, a.K);
    const int64_t chunks = (a.rows + chunk - 1) / chunk;
    const bool vec = a.K % 4 == 0 && a.ldm % 4 == 0 && (uintptr_t)a.M % 16 == 0 && (uintptr_t)a.partial % 16 == 0;
    const int VEC = vec ? 4 : 1;
    const dim3 grid((unsigned)((a.K + 64 * VEC - 1) / (64 * VEC)), (unsigned)chunks);
    if (vec)
        hipLaunchKernelGGL(lora_coldot_kernel<4>, grid, dim3(64), 0, st, a, a.M, a.V, a.partial, chunk);
    else
        hipLaunchKernelGGL(lora_coldot_kernel<1>, grid, dim3(64), 0, st, a, a.M, a.V, a.partial, chunk);
    hipLaunchKernelGGL(lora_coldot_reduce, dim3((unsigned)((a.K * a.r + 63) / 64)), dim3(64 * kColRed), 0, st, a, chunks);
    return hipGetLastError();
}

hipError_t launch_lora_merge(const LoraMergeArgs& a, hipStream_t st) {
    if (a.in <= 0 || a.cols <= 0) return hipSuccess;
    hipLaunchKernelGGL(lora_merge_kernel, dim3(grid_for(a.in * a.cols)), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace mft
