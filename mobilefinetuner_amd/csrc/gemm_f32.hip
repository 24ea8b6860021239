// fp32 matrix products from bf16 MFMAs.
//
// An fp32 number is the sum of three bf16 numbers, each the one nearest to what
// the earlier ones leave (split3; the remainders are exact in fp32, and the
// last is a bf16 number).  With a = a1 + a2 + a3 and b likewise,
//   a b = a1 b1 + a1 b2 + a2 b1 + a2 b2 + a1 b3 + a3 b1   (+ a2 b3 + a3 b2 + a3 b3)
// and each product of two bf16 numbers is exact in the fp32 accumulator's
// multiplier.  |a2| <= 2^-8 |a| and |a3| <= 2^-17 |a|: what six products leave
// out is under 2^-23.9 of a b and as often above as below it (cut to 8 bits
// each instead of rounded, the parts have the sign of a, and up to 2^-21 is
// lost towards zero).  Six v_mfma_f32_32x32x16_bf16 do the work of eight
// v_mfma_f32_32x32x2_f32 in 6 x 32 instead of 8 x 64 cycles, and round the
// accumulator 6 times per 16 values of k instead of 16.  Those save more than
// the six products leave out from K = 3 on; what is left of a sum after whole
// stages of 16 or 32, and with it every shorter sum, goes by fp32 MFMAs.  Norm
// of the error against 64 bits in 2^-24 of the result, normal operands, beside
// fp32 MFMAs throughout: K 16 1.0 (1.2), 100 1.7 (3.0), 768 2.9 (8.3); of one
// sign, 2048 rows: K 768 4.9 (7.1), 4096 9.9 (15.9).
// (Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", ARITH 2019, split fp32 so.)
// What it gives (us, TFLOP/s of the fp32 product; rocBLAS's fp32 kernels beside
// it, one box): 512 x 16384 x 768 73 us, 176 (102 us); 512 x 768 x 16384 86 us,
// 150 (895 us); 2048 x 16384 x 1024 351 us, 196 (458 us); 509 x 2304 x 768 25 us
// (27 us), 509 x 768 x 2304 24 us (20 us).  At T = 128 (512 x 50257 x 768 and its
// two gradients) the matrix units are busy 48 to 55 percent of the cycles, at
// the 1.8 to 2 GHz that the card holds under them, the VALU, which splits, 39,
// half of that beside them, and the LDS 28 to 37; half of the waves' cycles wait
// for issue.  At T = 64 the serial chain of a stage bounds it (matrix units 14 to
// 18 percent).
// Infinities: a remainder of inf, or 0 * inf among the six products, is NaN
// where fp32 arithmetic may give inf.  A tile with a NaN that no NaN operand of
// its row or column explains is computed again, whole, by the fp32 MFMAs; a NaN
// operand costs its tiles one more pass over their operands (the LM head and
// loss at 512 x 768 x 20001 with one NaN 0.75 ms, without 0.46).  So are tiles
// with a result past the largest float (a1 may be above a), and with one under
// 2^-80: the third part of an operand under 2^-110 lies below the smallest bf16
// subnormal, and up to 2^-134 is lost.  In results from 2^-80 on that is
// under their own rounding while K max(|a|, |b|) < 2^30; operands under 2^-134
// in a result that is then 0 stay 0.
//
// A workgroup (4 waves) owns a T x T tile of C and a range of BK-deep stages
// of k (of every term in turn, so that a rank-r update is one or two more
// stages).  A stage's fp32 values are loaded to registers two to three stages
// ahead, split while the stage before is multiplied, and written to the other of two
// LDS buffers ([plane][row][BK], 16-byte chunks XOR-swizzled): one barrier per
// stage, with the split's VALU work between the MFMAs.  The waves read each
// plane once: 12 KB of LDS reads per 24 MFMAs and wave at T = 128.  Either
// operand may be stored with k contiguous (16-byte loads along k) or not
// (loads along the rows, eight k per thread, which transposes in registers).
#include "gemm_f32.h"

#include <algorithm>

#include "attn_common.h"
#include "attn_geometry.h"
#include "attn_kernels.h"
#include "prologue_kernels.h"

namespace mft {
namespace {

constexpr int kPlanes = 3;

// Four floats at any address of a float: the loads take that, and rows of an
// odd length or base cost no more than others (4096 rows of LoRA 1151 -> 1153
// 650 us by stages of single loads, 243 by these).
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

struct Args {
    GemmF32 g;
    int tiles_m, tiles_n, slices, stages, per_slice;  // stages of all terms, and of one slice
    int n0;     // stages of term 0
    FastDiv per_slice_tiles, fewer_tiles;  // division by tiles_m tiles_n and by the smaller of the two
    int whole;  // one slice: written (or added) to C directly, else to partial
};

// E values as three planes of packed bf16.
template <int E> struct Split {
    uint32_t p[kPlanes][E / 2];
};
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {  // to nearest even
    typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(bf16)lo, (bf16)hi});
}
template <int E> __device__ __forceinline__ Split<E> split3(const float* x) {
    Split<E> s;
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
        float lo = x[2 * i], hi = x[2 * i + 1];
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) {
            // what is left for the last plane is a bf16 number
            const uint32_t u = p < kPlanes - 1 ? bf16_pair(lo, hi)
                                               : __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
            s.p[p][i] = u;
            lo -= __uint_as_float(u << 16);
            hi -= __uint_as_float(u & 0xffff0000u);
        }
    }
    return s;
}

// 16-byte chunk c (8 k) of row r in a plane of BK k per row.  Eight (BK = 16)
// or four (32) rows fill the 64 banks, so the chunk turns with r / 8 or r / 4,
// and 16 rows' reads of one chunk meet no bank twice.
template <int BK> __device__ __forceinline__ int chunk_at(int r, int c) {
    return BK == 16 ? r * 2 + (c ^ ((r >> 3) & 1)) : r * 4 + (c ^ ((r >> 2) & 3));
}

// One operand's stages on their way to LDS: each of the workgroup's NT threads
// holds E = T * BK / NT consecutive k of one row.  k-contiguous storage (KC):
// thread (row t / KG, k group t % KG); else (row t % T, k group t / T), a wave
// reading 64 consecutive rows at each k.
template <int T, int BK, int NT, bool KC> struct Loader {
    static constexpr int E = T * BK / NT, KG = BK / E;
    static_assert(E == 4 || E == 8, "one 16-byte load, or two");
    int row, kg;
    const float* base;  // this thread's first element of the fast path
    int64_t step;       // elements from one stage to the next
    __device__ __forceinline__ void place(int tid) {
        row = KC ? tid / KG : tid % T;
        kg = KC ? tid % KG : tid / T;
    }
    __device__ __forceinline__ void init(int tid, const float* p, int64_t ld, int64_t r0, int64_t rows) {
        place(tid);
        const int64_t r = min(r0 + row, rows - 1);  // rows past the end are not stored
        base = KC ? p + r * ld + E * kg : p + E * kg * ld + r;
        step = KC ? BK : BK * ld;
    }
    // Stage i of the first term (whole, vector loads).
    __device__ __forceinline__ void load_fast(int64_t i, int64_t ld, float* x) const {
        const float* q = base + i * step;
        if constexpr (KC) {
#pragma unroll
            for (int v = 0; v < E / 4; ++v) {
                const f32x4_any u = reinterpret_cast<const f32x4_any*>(q)[v];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * v + e] = u[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = q[e * ld];
        }
    }
    // k in [k0, k0 + BK) of any operand, element by element: the last stage
    // of a term, and the second term.
    __device__ __forceinline__ void load_any(const float* p, int64_t ld, bool kc, int64_t r0, int64_t rows, int64_t k0,
                                             int64_t K, float* x) const {
        const int64_t sr = kc ? ld : 1, sk = kc ? 1 : ld, k = k0 + E * kg;
        const float* q = p + min(r0 + row, rows - 1) * sr;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float v = q[min(k + e, K - 1) * sk];
            x[e] = k + e < K ? v : 0.f;
        }
    }
    __device__ __forceinline__ void store(uint4* lds, const float* x) const {
        const Split<E> s = split3<E>(x);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) {
            uint4* d = lds + p * T * BK / 8 + chunk_at<BK>(row, E * kg / 8);
            if constexpr (E == 8)
                *d = make_uint4(s.p[p][0], s.p[p][1], s.p[p][2], s.p[p][3]);
            else
                reinterpret_cast<uint2*>(d)[kg & 1] = make_uint2(s.p[p][0], s.p[p][1]);
        }
    }
    __device__ __forceinline__ void store_f32(float* lds, int ld, const float* x) const {
#pragma unroll
        for (int v = 0; v < E / 4; ++v)
            *reinterpret_cast<f32x4*>(lds + row * ld + E * kg + 4 * v) =
                f32x4{x[4 * v], x[4 * v + 1], x[4 * v + 2], x[4 * v + 3]};
    }
};

// Results that the split does not vouch for (see the top): not finite, or under
// 2^-80 and not 0.  Twice the bits less one orders zeros above all others.
struct Doubt {
    uint32_t least = ~0u;
    float sum = 0.f;  // NaN once a value is not finite
    __device__ __forceinline__ void look(float x) {
        least = min(least, (__float_as_uint(x) << 1) - 1u);
        sum = fmaf(x, 0.f, sum);
    }
    __device__ __forceinline__ bool any() const { return least < ((127u - 80u) << 24) - 1u || sum != sum; }
};

// TA / TB: term 0's storage.  KW groups of 2 x 2 waves share a stage's 16-deep
// k steps; their accumulators are added through LDS at the end.
template <int T, int BK, int KW, bool TA, bool TB>
__global__ __launch_bounds__(256 * KW, 3) void gemm_f32_kernel(Args a) {
    constexpr int MT = T / 64, NT = T / 64;  // 32 x 32 tiles per wave
    constexpr int kThreads = 256 * KW, KS = BK / 16 / KW;  // k steps of a wave per stage
    constexpr int TM = T, TN = T, kBuf = kPlanes * T * BK / 8;  // uint4 per operand and buffer
    __shared__ uint4 lds[4 * kBuf];  // [buffer][A, B]
    __shared__ int votes[2][4 * KW], nan_rows[2 * T];
    const int lane = threadIdx.x & 63, w = wave_id(), n = lane & 31, hh = lane >> 5;
    const int wm = w & 1, wn = w >> 1 & 1, wk = w >> 2;

    // Tiles that share the larger operand's rows run next to each other on one
    // XCD: the smaller tile count fastest, then the other, then the k slices.
    int i = xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int slice = (int)a.per_slice_tiles.div(i);
    i -= slice * a.tiles_m * a.tiles_n;
    const bool m_fast = a.tiles_m <= a.tiles_n;
    const int slow = (int)a.fewer_tiles.div(i), fast = i - slow * (m_fast ? a.tiles_m : a.tiles_n);
    const int tm = m_fast ? fast : slow, tn = m_fast ? slow : fast;
    const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;
    const int s0 = slice * a.per_slice, s1 = min(s0 + a.per_slice, a.stages);

    const GemmF32Term &f = a.g.terms[0], &h = a.g.terms[1];
    Loader<T, BK, kThreads, !TA> ldr_a;
    Loader<T, BK, kThreads, TB> ldr_b;
    constexpr int E = decltype(ldr_a)::E;
    ldr_a.init(threadIdx.x, f.A, f.lda, m0, a.g.M);
    ldr_b.init(threadIdx.x, f.B, f.ldb, n0, a.g.N);
    // Stages [s0, sf) are whole and go by vector loads.
    const int sf = f.alpha == 1.f ? max(s0, min(s1, (int)(f.K / BK))) : s0;
    f32x16 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int k = 0; k < MT; ++k) {
            acc[j][k] = zero16();
            asm volatile("" : "+v"(acc[j][k]));  // not a literal zero (see mfma_v_first)
        }
    struct Operands {
        bf16x8 a[KS][MT][kPlanes], b[KS][NT][kPlanes];
    };
    auto read = [&](int buf) {
        const uint4* la = lds + buf * 2 * kBuf;
        const uint4* lb = la + kBuf;
        Operands o;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) {
#pragma unroll
                for (int k = 0; k < MT; ++k)
                    o.a[ks][k][p] = __builtin_bit_cast(
                        bf16x8, la[p * T * BK / 8 + chunk_at<BK>(wm * (TM / 2) + 32 * k + n, 2 * (KS * wk + ks) + hh)]);
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    o.b[ks][j][p] = __builtin_bit_cast(
                        bf16x8, lb[p * T * BK / 8 + chunk_at<BK>(wn * (TN / 2) + 32 * j + n, 2 * (KS * wk + ks) + hh)]);
            }
        return o;
    };
    // C^T = B^T A^T per 32 x 32 tile (four consecutive n per register group),
    // the smallest products first.
    auto multiply = [&](const Operands& o) {
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int k = 0; k < MT; ++k)
                        acc[j][k] = mfma_bf16(o.b[ks][j][pb[q]], o.a[ks][k][pa[q]], acc[j][k]);
    };
    float xa[2][E], xb[2][E];
    auto fetch = [&](int s, float* u, float* v) {  // a fast stage; past the last one, that again
        const int64_t i = min(s, sf - 1);
        ldr_a.load_fast(i, f.lda, u);
        ldr_b.load_fast(i, f.ldb, v);
    };
    // Stage s from LDS buffer `buf`, while stage s + 1 goes from registers to
    // the other buffer; stage s + 3 is then loaded in its place.  No branch
    // inside: the compiler's waits then count the loads of each stage.
    auto step = [&](int s, int buf, float* u, float* v) {
        const Operands o = read(buf);
        uint4* next = lds + (buf ^ 1) * 2 * kBuf;
        multiply(o);
        ldr_a.store(next, u);
        ldr_b.store(next + kBuf, v);
#pragma unroll
        // The split between the MFMAs (3 to 5 tried at T = 128, 4 to 12 at 64,
        // where loads along the rows add addresses; up to 8 percent apart).
        for (int q = 0; q < 6 * MT * NT * KS; ++q) {
            __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
            __builtin_amdgcn_sched_group_barrier(SG_VALU, MT * NT > 1 ? 5 : TB ? 6 : 8, 0);
        }
        fetch(s + 3, u, v);
        lds_barrier();
    };
    if (s0 < sf) {
        fetch(s0, xa[0], xb[0]);
        fetch(s0 + 1, xa[1], xb[1]);
        ldr_a.store(lds, xa[0]);
        ldr_b.store(lds + kBuf, xb[0]);
        fetch(s0 + 2, xa[0], xb[0]);
        lds_barrier();
        for (int s = s0; s < sf; s += 2) {
            step(s, 0, xa[1], xb[1]);
            if (s + 1 < sf) step(s + 1, 1, xa[0], xb[0]);
        }
    }
    // The other stages one at a time, in fp32 MFMAs: a term's last, partial
    // one, the second term's, and all of a term times alpha.
    // Sums of few terms are all here (see the top).  Half hh of a wave takes
    // values 4 hh .. 4 hh + 3 of each eight k, and the KW groups of waves take
    // the eights in turn.
    // What these stages and the results' addresses need is formed again here
    // (tid is opaque): kept through the loop above it costs the third workgroup
    // of a CU its registers.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int n2 = tid & 31, hh2 = tid >> 5 & 1;
    Loader<T, BK, kThreads, !TA> any_a;
    Loader<T, BK, kThreads, TB> any_b;
    any_a.place(tid), any_b.place(tid);
    constexpr int kRow = BK + 4;  // floats from one row to the next
    float* fa = reinterpret_cast<float*>(lds);
    float* fb = fa + TM * kRow;
    static_assert((TM + TN) * kRow * 4 + (KW - 1) * 4 * 16 * 64 * 4 <= sizeof(lds), "a stage in fp32 and the shares of k fit the buffers");
    // Whether x holds in any thread of the workgroup (a barrier between the two).
    auto vote = [&](int i, bool x) {
        const bool any = __any(x);
        if (lane == 0) votes[i][w] = any;
    };
    auto voted = [&](int i) {
        int v = 0;
#pragma unroll
        for (int q = 0; q < 4 * KW; ++q) v |= votes[i][q];
        return __builtin_amdgcn_readfirstlane(v) != 0;
    };
    auto load_stage = [&](int s, float* u, float* v) {  // any stage
        const bool second = s >= a.n0;
        const int64_t k0 = (int64_t)BK * (second ? s - a.n0 : s), K = second ? h.K : f.K;
        any_a.load_any(second ? h.A : f.A, second ? h.lda : f.lda, second ? h.ta == 0 : !TA, m0, a.g.M, k0, K, u);
        any_b.load_any(second ? h.B : f.B, second ? h.ldb : f.ldb, second ? h.tb != 0 : TB, n0, a.g.N, k0, K, v);
        return (int)min<int64_t>(BK, K - k0 + 7) / 8;  // eights of k that hold values
    };
    auto fp32_stages = [&](int from) {
        for (int s = from; s < s1; ++s) {
            const int eights = load_stage(s, xa[0], xb[0]);
            const float alpha = s >= a.n0 ? h.alpha : f.alpha;
#pragma unroll
            for (int e = 0; e < E; ++e) xa[0][e] *= alpha;
            lds_barrier();
            any_a.store_f32(fa, kRow, xa[0]);
            any_b.store_f32(fb, kRow, xb[0]);
            lds_barrier();
            for (int i = wk; i < eights; i += KW) {
                f32x4 va[MT], vb[NT];
#pragma unroll
                for (int k = 0; k < MT; ++k)
                    va[k] = *reinterpret_cast<const f32x4*>(fa + (wm * (TM / 2) + 32 * k + n2) * kRow + 8 * i + 4 * hh2);
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    vb[j] = *reinterpret_cast<const f32x4*>(fb + (wn * (TN / 2) + 32 * j + n2) * kRow + 8 * i + 4 * hh2);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
#pragma unroll
                        for (int k = 0; k < MT; ++k) acc[j][k] = mfma_f32(vb[j][e], va[k][e], acc[j][k]);
            }
        }
    };
    auto join = [&] {  // the waves' shares of k
        if constexpr (KW > 1) {
            static_assert(KW == 2 && MT * NT == 1, "two groups of waves, one 32 x 32 tile each");
            float* other = fb + TN * kRow + (w & 3) * 16 * 64 + lane;
            if (wk == 1)
#pragma unroll
                for (int r = 0; r < 16; ++r) other[64 * r] = acc[0][0][r];
            lds_barrier();
            if (wk == 0)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[0][0][r] += other[64 * r];
        } else {
            lds_barrier();
        }
    };
    fp32_stages(sf);
    Doubt doubt;
#pragma unroll
    for (int i = 0; i < 16 * MT * NT; ++i) doubt.look(acc[i / (16 * MT)][i / 16 % MT][i % 16]);
    vote(0, doubt.any());
    join();
    if (__builtin_expect(sf > s0 && voted(0), 0)) {
        // NaN throughout the rows of A and of B that hold one: the other elements count.
        int here = tid;
        asm volatile("" : "+v"(here));  // nothing of this is formed ahead
        for (int i = here; i < TM + TN; i += kThreads) nan_rows[i] = 0;
        lds_barrier();
        constexpr int kParts = kThreads / (TM + TN);  // threads to a row
        const int row = here % (TM + TN), part = here / (TM + TN);
        const bool of_a = row < TM;
        bool nan = false;
        for (int t = 0; t < 2; ++t) {
            const GemmF32Term& x = a.g.terms[t];
            const int e0 = t == 0 ? min(s0, a.n0) : max(s0, a.n0) - a.n0, e1 = t == 0 ? min(s1, a.n0) : max(s1, a.n0) - a.n0;
            const int64_t k1 = min((int64_t)BK * e1, x.K);
            const bool kc = of_a ? x.ta == 0 : x.tb != 0;
            const int64_t ld = of_a ? x.lda : x.ldb, r = of_a ? min(m0 + row, a.g.M - 1) : min(n0 + row - TM, a.g.N - 1);
            const float* q = (of_a ? x.A : x.B) + r * (kc ? ld : 1);
            const int64_t step = kc ? 1 : ld;
            constexpr int U = 8;  // loads in flight
            int64_t k = (int64_t)BK * e0 + U * part;
            for (; k + U <= k1; k += U * kParts) {
                float v[U];
                if (kc) {
#pragma unroll
                    for (int i = 0; i < U / 4; ++i) {
                        const f32x4_any u = *reinterpret_cast<const f32x4_any*>(q + k + 4 * i);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[4 * i + e] = u[e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < U; ++e) v[e] = q[(k + e) * step];
                }
#pragma unroll
                for (int e = 0; e < U; ++e) nan |= v[e] != v[e];
            }
            for (const int64_t last = min(k + U, k1); k < last; ++k) nan |= q[k * step] != q[k * step];
        }
        if (nan) nan_rows[row] = 1;
        lds_barrier();
        bool again = false;
        if (wk == 0)
#pragma unroll
            for (int i = 0; i < 16 * MT * NT; ++i) {
                const int j = i / (16 * MT), k = i / 16 % MT, r = i % 16;
                const int m = nan_rows[wm * (TM / 2) + 32 * k + (here & 31)],
                          c = nan_rows[TM + wn * (TN / 2) + 32 * j + row_of_reg(r, here >> 5 & 1)];
                float x = acc[j][k][r];
                asm volatile("" : "+v"(x));  // looked at anew: kept from above it costs a register each
                Doubt one;
                one.look(x);
                again |= one.any() & ((m | c) == 0);
            }
        vote(1, again);
        lds_barrier();
        if (voted(1)) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int k = 0; k < MT; ++k) {
                    acc[j][k] = zero16();
                    asm volatile("" : "+v"(acc[j][k]));  // as above
                }
            fp32_stages(s0);
            join();
        }
    }
    if (wk != 0) return;

    float* C = a.whole ? a.g.C : a.g.partial + (int64_t)slice * a.g.M * a.g.N;
    const int64_t ldc = a.whole ? a.g.ldc : a.g.N;
    const float* bias = a.whole ? a.g.bias : nullptr;
    const bool vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
    const int64_t mw = m0 + wm * (TM / 2) + n2, nw = n0 + wn * (TN / 2) + 4 * hh2;
    if (a.whole && a.g.add) {  // all of C's loads ahead of the stores
#pragma unroll
        for (int k = 0; k < MT; ++k) {
            const float* row = C + min(mw + 32 * k, a.g.M - 1) * ldc;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int64_t c0 = nw + 32 * j + 8 * q;
                    f32x4 o;
                    if (vec && a.g.N % 4 == 0) {
                        o = *reinterpret_cast<const f32x4*>(row + min(c0, a.g.N - 4));
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = row[min(c0 + e, a.g.N - 1)];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[j][k][4 * q + e] += o[e];
                }
        }
    }
#pragma unroll
    for (int k = 0; k < MT; ++k) {
        const int64_t m = mw + 32 * k;
        if (m >= a.g.M) continue;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t c0 = nw + 32 * j + 8 * q;
                f32x4 o{acc[j][k][4 * q], acc[j][k][4 * q + 1], acc[j][k][4 * q + 2], acc[j][k][4 * q + 3]};
                float* d = C + m * ldc + c0;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (bias && c0 + e < a.g.N) o[e] += bias[c0 + e];
                if (vec && c0 + 4 <= a.g.N) {
                    *reinterpret_cast<f32x4*>(d) = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (c0 + e < a.g.N) d[e] = o[e];
                }
            }
    }
}

// C (+)= the slices' partial products in slice order, + bias.
template <int VEC>
__global__ __launch_bounds__(256) void gemm_f32_reduce(Args a) {
    typedef float V __attribute__((ext_vector_type(VEC)));
    const int64_t MN = a.g.M * a.g.N, i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (i >= MN) return;
    const int64_t m = i / a.g.N, n = i - m * a.g.N;  // N is a multiple of VEC
    V sum = *reinterpret_cast<const V*>(a.g.partial + i);
#pragma unroll 8
    for (int s = 1; s < a.slices; ++s) sum += *reinterpret_cast<const V*>(a.g.partial + s * MN + i);
    float* d = a.g.C + m * a.g.ldc + n;
#pragma unroll
    for (int e = 0; e < VEC; ++e) d[e] = sum[e] + (a.g.bias ? a.g.bias[n + e] : 0.f) + (a.g.add ? d[e] : 0.f);
}

struct Plan {
    bool small;  // 64 x 64 tiles
    Args a;
};

// 128 x 128 tiles where they fill the GPU, with k cut into slices or not; else
// 64 x 64.  k is cut into slices of at least kMinSlice values until about two
// workgroups per CU run, where the tiles alone leave more than half of the GPU
// idle (each slice costs an fp32 tile written and read again), and of at
// least kFewSlice until one per CU does (33 x 768 x 768 10.8 -> 9.7 us, 64 x 768
// x 500 12.9 -> 9.7).  Where 128 x 128 tiles would need slices, a K up to
// kUncut is shorter in 64 x 64 tiles without (1024 x 1024 x 1024 29 -> 22 us,
// 2048 x 768 x 768 35 -> 24; at 2048 x 640 x 2048 52 against 44).
constexpr int kMinSlice = 256, kFewSlice = 96, kUncut = 1536;
Plan plan(const GemmF32& g) {
    Plan p{};
    const int cus = device_cus();
    auto tiles = [&](int t) { return ((g.M + t - 1) / t) * ((g.N + t - 1) / t); };
    const int64_t K = g.terms[0].K + g.terms[1].K;
    auto cut = [&](int64_t t) {
        return 2 * t >= cus ? 1
                            : (int)std::max<int64_t>({1, std::min<int64_t>(2 * cus / t, K / kMinSlice),
                                                      std::min<int64_t>(cus / t, K / kFewSlice)});
    };
    const int64_t t128 = tiles(128);
    const bool cut128 = 2 * t128 < cus;
    const int64_t c128 = cut128 ? std::max<int64_t>(1, std::min<int64_t>(2 * cus / t128, K / kMinSlice)) : 1;
    p.small = t128 * c128 < cus || (cut128 && K <= kUncut);
    const int t = p.small ? 64 : 128, bk = p.small ? 32 : 16;
    p.a.g = g;
    p.a.tiles_m = (int)((g.M + t - 1) / t);
    p.a.tiles_n = (int)((g.N + t - 1) / t);
    p.a.n0 = (int)((g.terms[0].K + bk - 1) / bk);
    const int stages = p.a.stages = p.a.n0 + (int)((g.terms[1].K + bk - 1) / bk);
    const int slices = cut(tiles(t));
    p.a.per_slice = (stages + slices - 1) / slices;
    p.a.slices = (stages + p.a.per_slice - 1) / p.a.per_slice;
    p.a.whole = p.a.slices == 1;
    p.a.per_slice_tiles = FastDiv::make((uint32_t)(p.a.tiles_m * p.a.tiles_n));
    p.a.fewer_tiles = FastDiv::make((uint32_t)std::min(p.a.tiles_m, p.a.tiles_n));
    return p;
}

template <int T, int BK, int KW>
void launch_t(const Args& a, hipStream_t st) {
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n * a.slices));
    const bool ta = a.g.terms[0].ta != 0, tb = a.g.terms[0].tb != 0;
    if (ta && tb)
        hipLaunchKernelGGL((gemm_f32_kernel<T, BK, KW, true, true>), grid, dim3(256 * KW), 0, st, a);
    else if (ta)
        hipLaunchKernelGGL((gemm_f32_kernel<T, BK, KW, true, false>), grid, dim3(256 * KW), 0, st, a);
    else if (tb)
        hipLaunchKernelGGL((gemm_f32_kernel<T, BK, KW, false, true>), grid, dim3(256 * KW), 0, st, a);
    else
        hipLaunchKernelGGL((gemm_f32_kernel<T, BK, KW, false, false>), grid, dim3(256 * KW), 0, st, a);
}

}  // namespace

size_t gemm_f32_workspace(const GemmF32& g) {
    const Plan p = plan(g);
    return !p.a.whole ? (size_t)p.a.slices * g.M * g.N * 4 : 0;
}

hipError_t launch_gemm_f32(const GemmF32& g, hipStream_t st) {
    if (g.M <= 0 || g.N <= 0) return hipSuccess;
    const Plan p = plan(g);
    if (p.small)
        launch_t<64, 32, 2>(p.a, st);
    else
        launch_t<128, 16, 1>(p.a, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.a.whole) return e;
    const int64_t MN = g.M * g.N;
    if (g.N % 4 == 0)
        hipLaunchKernelGGL(gemm_f32_reduce<4>, dim3((unsigned)((MN / 4 + 255) / 256)), dim3(256), 0, st, p.a);
    else
        hipLaunchKernelGGL(gemm_f32_reduce<1>, dim3((unsigned)((MN + 255) / 256)), dim3(256), 0, st, p.a);
    return hipGetLastError();
}

}  // namespace mft
