// product.h — the arithmetic every EXACT product kernel shares (the GEMMs and
// the GEMVs): the activation split, one kstep and one chunk of a product, and
// the operands of the affine formats. A row's bits are the same from every
// kernel because they all run these functions in the same order.
#pragma once
#include <type_traits>

#include "fmt.h"
#include "launch.h"

#define KSTEPS 4  // ksteps per chunk
#define HSTEPS 8  // half-steps per chunk

__device__ __forceinline__ f16v mfma32(half8 a, half8 b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f16v zero16() {
    f16v z;
#pragma unroll
    for (int e = 0; e < 16; e++) z[e] = 0.0f;
    return z;
}

// D-layout row of accumulator element e for lane half hh
__device__ __forceinline__ int drow(int e, int hh) { return 8 * (e >> 2) + 4 * hh + (e & 3); }

__device__ __forceinline__ float silu_f(float v) {
    // x * sigmoid(x) with the reference's stable sigmoid (src/qmat.h:31-35):
    // exp only of -|x| (never overflows); 1/(1+e) for x >= 0, e/(1+e) below.
    // Hardware exp2 and reciprocal (~1 ulp each), like the reference's own
    // -ffast-math build; every kernel applies this same function.
    const float e = __expf(-fabsf(v));
    const float r = __builtin_amdgcn_rcpf(1.0f + e);
    return v * (v >= 0.0f ? r : e * r);
}

// a double moved between lanes by one DPP pattern (its two halves)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// The wave's sum in every lane: within each row of 16 lanes by DPP (swap
// neighbours, swap pairs, mirror within 8, mirror within 16: each step adds
// two values symmetrically, so every lane holds the same sum), then across
// the four rows.
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_d<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_d<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp_d<0x141>(v);   // row_half_mirror
    v += dpp_d<0x140>(v);   // row_mirror
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}
// the maximum over the wave (N = 64) or over each half of it (32), in every lane
template <int N>
__device__ __forceinline__ float wave_max(float v) {
    auto step = [&](auto ctrl) {
        v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF,
                                                                false)));
    };
    step(std::integral_constant<int, 0xB1>{});    // (the steps of wave_sum)
    step(std::integral_constant<int, 0x4E>{});
    step(std::integral_constant<int, 0x141>{});
    step(std::integral_constant<int, 0x140>{});
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    if (N == 64) v = fmaxf(v, __shfl_xor(v, 32, 64));
    return v;
}
// 1/sqrt in double: the hardware's estimate (about 24 bits) and two Newton steps
__device__ __forceinline__ double rsqrt_d(double v) {
    double y = __builtin_amdgcn_rsq(v);
#pragma unroll
    for (int i = 0; i < 2; i++) y = y * (1.5 - 0.5 * v * y * y);
    return y;
}

// ---------------------------------------------------------------------------
// Activation split of one chunk, in the A-operand layout: lane (r = l&31,
// hh = l>>5) holds elements 16u + 8hh .. +7 of half-step u for row m. The
// chunk's largest magnitude is shared by the two lanes of a row through one
// xor shuffle (every lane of the wave must call this).
struct XChunk {
    half8 h[HSTEPS], l[HSTEPS];
    float s8[HSTEPS];  // sum of the lane's 8 scaled values of half-step u, in order
    float p;           // 2^-sh: the chunk's fold factor for this row
};

// f16(x0 - h.lo), f16(x1 - h.hi) as one packed pair: x - h is exact in f32
// (h is x rounded to f16), and v_fma_mixlo / v_fma_mixhi form it with h read as f16 in place
// and rounds it to f16 once: the value of (_Float16)(x - (float)h), in two
// instructions per pair instead of six.
__device__ __forceinline__ uint32_t lo_pair(uint32_t hpair, float x0, float x1) {
    uint32_t r;
    asm volatile("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(hpair), "v"(x0));
    asm volatile("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
                 : "+v"(r)
                 : "v"(hpair), "v"(x1));
    return r;
}

// the split of NU half-steps' values v[u][j] with shift sh
template <int NU>
__device__ __forceinline__ void split_part(const float (&v)[NU][8], int sh, half8 (&h)[NU], half8 (&l)[NU],
                                           float (&s8)[NU]) {
#pragma unroll
    for (int u = 0; u < NU; u++) {
        float acc = 0.0f;
        float xs[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            xs[j] = ldexpf(v[u][j], sh);
            h[u][j] = (_Float16)xs[j];
            acc += xs[j];
        }
        s8[u] = acc;
        uint32_t hw[4], lw[4];
        __builtin_memcpy(hw, &h[u], 16);
#pragma unroll
        for (int t = 0; t < 4; t++) lw[t] = lo_pair(hw[t], xs[2 * t], xs[2 * t + 1]);
        __builtin_memcpy(&l[u], lw, 16);
    }
}

// the split of one chunk's values v[u][j] (element 16u + 8hh + j of row m)
__device__ __forceinline__ void split_vals(const float (&v)[HSTEPS][8], XChunk &o) {
    float amax = 0.0f;
#pragma unroll
    for (int u = 0; u < HSTEPS; u++)
#pragma unroll
        for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(v[u][j]));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    const int sh = chunk_shift(amax);
    o.p = ldexpf(1.0f, -sh);
    split_part<HSTEPS>(v, sh, o.h, o.l, o.s8);
}

// VEC: K % 8 == 0 and 16-byte aligned rows (each lane's 8 elements are
// wholly inside or wholly past K), two float4 loads per half-step
template <bool VEC>
__device__ __forceinline__ void load_chunk(const float *__restrict__ x, int M, int K, int m, int c, int hh,
                                           float (&v)[HSTEPS][8]) {
    const bool live = m < M;
    const float *row = x + (size_t)(live ? m : 0) * K;
#pragma unroll
    for (int u = 0; u < HSTEPS; u++) {
        const int k0 = 128 * c + 16 * u + 8 * hh;
        if constexpr (VEC) {
            float4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
            if (live && k0 < K) {
                a = *(const float4 *)(row + k0);
                b = *(const float4 *)(row + k0 + 4);
            }
            v[u][0] = a.x; v[u][1] = a.y; v[u][2] = a.z; v[u][3] = a.w;
            v[u][4] = b.x; v[u][5] = b.y; v[u][6] = b.z; v[u][7] = b.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) v[u][j] = (live && k0 + j < K) ? row[k0 + j] : 0.0f;
        }
    }
}

template <bool VEC>
__device__ __forceinline__ void split_chunk(const float *__restrict__ x, int M, int K, int m, int c, int hh,
                                            XChunk &o) {
    float v[HSTEPS][8];
    load_chunk<VEC>(x, M, K, m, c, hh, v);
    split_vals(v, o);
}

// ---------------------------------------------------------------------------
// Weight fragments of WN column groups: per-chunk headers and per-kstep words.
// Formats whose integer sub-block factors fold into the decoded weights (the
// FHdr traits): a chunk's MFMAs then accumulate straight through its four
// ksteps, and the factors d (and the mins, through one more MFMA) apply once
// per chunk instead of once per sub-block
template <int QT> constexpr bool fold_fmt() {
    return QT == QT_Q2_K || QT == QT_Q3_K || QT == QT_Q4_K || QT == QT_Q5_K;
}
template <int QT, bool FOLD = fold_fmt<QT>()> struct KHdr { using T = typename Fmt<QT>::Hdr; };
template <int QT> struct KHdr<QT, true> { using T = typename Fmt<QT>::FHdr; };

template <int QT, int WN> struct BH { typename KHdr<QT>::T h[WN]; };
template <int QT, int WN> struct BK { typename Fmt<QT>::RawK r[WN]; };

template <int QT, int WN>
__device__ __forceinline__ void load_bh(const DevW &W, int Kc, const int (&gn)[WN], int c, int lane, BH<QT, WN> &b) {
#pragma unroll
    for (int j = 0; j < WN; j++) {
        if constexpr (fold_fmt<QT>()) Fmt<QT>::load_fhdr(W, Kc, gn[j], c, lane, b.h[j]);
        else Fmt<QT>::load_hdr(W, Kc, gn[j], c, lane, b.h[j]);
    }
}
template <int QT, int WN>
__device__ __forceinline__ void load_bk(const DevW &W, int Kc, const int (&gn)[WN], int c, int s, int lane,
                                        BK<QT, WN> &b) {
#pragma unroll
    for (int j = 0; j < WN; j++) Fmt<QT>::load_k(W, Kc, gn[j], c, s, lane, b.r[j]);
}

// A fragments of one kstep for WM row groups: the two f16 terms of its two
// half-steps
template <int WM> struct AK {
    half8 h[WM][2], l[WM][2];
};

// The exact product of one kstep into the chunk accumulator. Folded formats:
// acc += xh*(q f) + xl*(q f) for both half-steps, MFMA after MFMA; the others:
// t = the kstep's MFMAs from zero, acc = fma(sc, t, acc) per sub-block. The
// float operations each output sees, and their order, are the same in every
// caller.
//
// A1 (INT8ACT numerics): the activations are int8 values held as f16 (exact),
// one term: the xl MFMAs drop out, and every sum the MFMAs form is an exact
// integer (the kernels keep each accumulation below 2^24 in magnitude).
//
// NE: the per-element f32 work covers accumulator elements e < NE only (the
// GEMV of M rows reads elements 0 .. NE-1: rows drow(e, hh) below M); the
// elements it covers see the same operations at every NE.
template <int QT, int WM, int WN, bool A1 = false, int NE = 16>
__device__ __forceinline__ void kstep(const AK<WM> &a, const BK<QT, WN> &b, const BH<QT, WN> &hd, int s,
                                      f16v (&acc)[WM][WN]) {
    using F = Fmt<QT>;
    if constexpr (fold_fmt<QT>()) {
#pragma unroll
        for (int j = 0; j < WN; j++) {
            const half8 b0 = F::decode_f(b.r[j], s, 0, hd.h[j]), b1 = F::decode_f(b.r[j], s, 1, hd.h[j]);
#pragma unroll
            for (int i = 0; i < WM; i++) {
                acc[i][j] = mfma32(a.h[i][0], b0, acc[i][j]);
                acc[i][j] = mfma32(a.h[i][1], b1, acc[i][j]);
                if constexpr (!A1) {
                    acc[i][j] = mfma32(a.l[i][0], b0, acc[i][j]);
                    acc[i][j] = mfma32(a.l[i][1], b1, acc[i][j]);
                }
            }
        }
    } else if constexpr (QT == QT_F32) {
        static_assert(!A1, "f32 weights have no int8-activation form");
        // f32 weights: resident as (wh, wl) f16 pairs scaled per row by
        // 2^shw_n; acc += xh*wh + xh*wl + xl*wh straight into the chunk
        // accumulator (no per-kstep factor)
#pragma unroll
        for (int kh = 0; kh < 2; kh++)
#pragma unroll
            for (int j = 0; j < WN; j++)
#pragma unroll
                for (int i = 0; i < WM; i++) {
                    acc[i][j] = mfma32(a.h[i][kh], b.r[j].h[kh], acc[i][j]);
                    acc[i][j] = mfma32(a.h[i][kh], b.r[j].l[kh], acc[i][j]);
                    acc[i][j] = mfma32(a.l[i][kh], b.r[j].h[kh], acc[i][j]);
                }
    } else if constexpr (!F::SUB16) {
        static_assert(!F::MINS, "affine formats fold");
#pragma unroll
        for (int j = 0; j < WN; j++) {
            const half8 b0 = F::decode(b.r[j], s, 0), b1 = F::decode(b.r[j], s, 1);
            float sc, mn;
            F::scale(hd.h[j], s, 0, sc, mn);
#pragma unroll
            for (int i = 0; i < WM; i++) {
                f16v t = mfma32(a.h[i][0], b0, zero16());
                t = mfma32(a.h[i][1], b1, t);
                if constexpr (!A1) {
                    t = mfma32(a.l[i][0], b0, t);
                    t = mfma32(a.l[i][1], b1, t);
                }
#pragma unroll
                for (int e = 0; e < NE; e++) acc[i][j][e] = __builtin_fmaf(sc, t[e], acc[i][j][e]);
            }
        }
    } else {
        static_assert(!F::MINS, "affine formats fold");
#pragma unroll
        for (int j = 0; j < WN; j++) {
            half8 b0, b1;
            if constexpr (QT == QT_Q6_K) {   // the same values, fewer instructions
                b0 = F::decode_fast(b.r[j], s, 0);
                b1 = F::decode_fast(b.r[j], s, 1);
            } else {
                b0 = F::decode(b.r[j], s, 0);
                b1 = F::decode(b.r[j], s, 1);
            }
            float sc0, mn0, sc1, mn1;
            F::scale(hd.h[j], s, 0, sc0, mn0);
            F::scale(hd.h[j], s, 1, sc1, mn1);
#pragma unroll
            for (int i = 0; i < WM; i++) {
                f16v t0 = mfma32(a.h[i][0], b0, zero16());
                if constexpr (!A1) t0 = mfma32(a.l[i][0], b0, t0);
                f16v t1 = mfma32(a.h[i][1], b1, zero16());
                if constexpr (!A1) t1 = mfma32(a.l[i][1], b1, t1);
#pragma unroll
                for (int e = 0; e < NE; e++) {
                    acc[i][j][e] = __builtin_fmaf(sc0, t0[e], acc[i][j][e]);
                    acc[i][j][e] = __builtin_fmaf(sc1, t1[e], acc[i][j][e]);
                }
            }
        }
    }
}

// The affine folded formats' row sums as the A operand of the chunk's mins
// MFMA: sub-block sum x_j (NS per chunk: the 16-element sums (first 8 in
// order) + (next 8), for 32-element sub-blocks two of them added) scaled by
// 2^-5 (|x_j| < 2^20, so the result fits f16) and split into f16 hi_j + lo_j;
// lane half 0 carries hi_j in slot j, half 1 lo_j, slots >= NS are zero. The
// mins product is then sum_j (hi_j + lo_j) * m_j = 2^-5 * sum_j x_j m_j.
__device__ __forceinline__ _Float16 xm_part(float xsum, int hh) {
    const float v = xsum * 0.03125f;
    const _Float16 hi = (_Float16)v;
    return hh ? (_Float16)(v - (float)hi) : hi;
}
template <int NS>
__device__ __forceinline__ half8 xm_frag(const float (&s8)[HSTEPS], int hh) {
    float s16[HSTEPS];
#pragma unroll
    for (int u = 0; u < HSTEPS; u++) s16[u] = s8[u] + __shfl_xor(s8[u], 32);
    half8 r;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        if (j < NS) r[j] = xm_part(NS == 8 ? s16[j] : s16[2 * j] + s16[2 * j + 1], hh);
        else r[j] = (_Float16)0.0f;
    }
    return r;
}

// End of a chunk of a folded format: acc (= sum of x * q f over the chunk)
// becomes d * acc - dm * (mins product), the chunk result the fold takes
template <int QT, int NE = 16>
__device__ __forceinline__ void fold_finish(const half8 &xm, const typename KHdr<QT>::T &H, f16v &acc) {
    if constexpr (Fmt<QT>::MINS) {
        const f16v t2 = mfma32(xm, H.mb, zero16());
#pragma unroll
        for (int e = 0; e < NE; e++) acc[e] = __builtin_fmaf(-H.dm, t2[e], H.d * acc[e]);
    } else {
#pragma unroll
        for (int e = 0; e < NE; e++) acc[e] = H.d * acc[e];
    }
}

// the per-row weight shift of the f32 format (0 for the quantized ones)
template <int QT>
__device__ __forceinline__ int wshift(const DevW &W, int n) {
    if constexpr (QT == QT_F32) return (int)W.h2[n];
    return 0;
}

// Where a product's result goes: EPI_Y stores y (SiLU applied when act);
// EPI_PREP (the first product of the FFN) applies SiLU and, instead of
// storing the f32 intermediate, prepares it as the second product's input —
// the workgroup's 128 output columns are exactly one 128-element chunk of
// the second product's K, so the chunk's shift, split and sums are formed
// here by split_part, the same function the preparation pass runs, on the
// same f32 values (bit-identical to storing y and preparing it).
enum { EPI_Y = 0, EPI_PREP = 1 };
struct PrepOut {
    uint8_t *xp, *xm;
    float *xpf;
    int Kc, xsum;   // mins A operands (xm_frag): 0 none, 1 of 8 sub-blocks, 2 of 4
};

// The products' output epilogue on v = the product (+ its bias): act 1 SiLU, 4
// ReLU; act 2 and 3 accumulate into y, y = fmaf(1 or 1/2, v, y) (the residual
// adds x += tmp and x += tmp / 2 of the encoder layer, with their operations);
// 0 v. yv: what y holds (for act 2 and 3).
__device__ __forceinline__ bool act_res(int act) { return act == 2 || act == 3; }
__device__ __forceinline__ float epi_out(int act, float v, float yv) {
    if (act == 1) return silu_f(v);
    if (act == 4) return v < 0.0f ? 0.0f : v;
    if (act_res(act)) return fmaf(act == 3 ? 0.5f : 1.0f, v, yv);
    return v;
}

// Weight bytes per element of the resident layout (planes and headers)
template <int QT> constexpr float w_bpe() {
    return QT == QT_F32 ? 4.0f : QT == QT_INT8 ? 1.0f : QT == QT_INT4 ? 0.5625f : QT == QT_Q4_0 ? 0.5625f
         : QT == QT_Q8_0 ? 1.0625f : QT == QT_Q2_K ? 0.33f : QT == QT_Q3_K ? 0.43f : QT == QT_Q4_K ? 0.5625f
         : QT == QT_Q5_K ? 0.6875f : 0.82f;
}

// Compiler-level ordering of a wave's own LDS writes and reads (the LDS
// executes one wave's operations in issue order).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Products of few rows, K split over a workgroup's waves (gemm_ksplit.hip):
// whether M rows of `jobs` products of W's shape and format take that form (prep:
// the FFN's prepared output, as mh_launch_gemm_prep_out; a1: INT8ACT), and its launch
bool mh_use_gemm_ks(int qtype, const DevW &W, int M, int jobs, bool prep, bool a1);
hipError_t mh_launch_gemm_ks(int qtype, const GemmJobs &J, const uint8_t *xp, const float *xs16, const float *xpf, int M,
                             int act, const PrepOut *po, bool a1, hipStream_t st);

#define MH_DISPATCH(fn, qtype, ...)                                  \
    switch (qtype) {                                                 \
    case QT_F32: return fn<QT_F32>(__VA_ARGS__);                     \
    case QT_INT8: return fn<QT_INT8>(__VA_ARGS__);                   \
    case QT_INT4: return fn<QT_INT4>(__VA_ARGS__);                   \
    case QT_Q4_0: return fn<QT_Q4_0>(__VA_ARGS__);                   \
    case QT_Q8_0: return fn<QT_Q8_0>(__VA_ARGS__);                   \
    case QT_Q2_K: return fn<QT_Q2_K>(__VA_ARGS__);                   \
    case QT_Q3_K: return fn<QT_Q3_K>(__VA_ARGS__);                   \
    case QT_Q4_K: return fn<QT_Q4_K>(__VA_ARGS__);                   \
    case QT_Q5_K: return fn<QT_Q5_K>(__VA_ARGS__);                   \
    case QT_Q6_K: return fn<QT_Q6_K>(__VA_ARGS__);                   \
    }                                                                \
    return hipErrorInvalidValue;

