// encoder.hip — the steps of one FastConformer encoder layer around its
// products and its attention core (src/encoder.c:485-521 and the batched form
// :901-946): the layer norms with the residual add that precedes each of
// them, the GLU, and the depthwise convolution with its conv norm and SiLU
// (conv_module, :413-462).
//
//   k_add_ln    x += alpha * res (when res), then out = LN(x) per row
//               (layer_norm_f, :25-37; the adds of :495, 502, 507, 511)
//   k_add_ln_prep  the same, its output written as the products' prepared
//               input (EXACT numerics) instead of f32 rows
//   k_glu       g = a * sigmoid(b) over the two halves of each row  :426-432
//   k_dwconv    depthwise conv over time within each segment (causal: left
//               pad k-1; else 'same'), + dw_b, then the folded batch norm
//               x * scale + shift and SiLU when scale is given     :434-459
//   k_dwconv_tile  the same on LDS tiles, forming the GLU as it stages its
//               input
//
// and of the dw_striding subsampling in front of the layers
// (src/subsampling.c:208-268, 109-200), with activations channel-last,
// [segment][time][freq][channel], so that its pointwise convolutions and its
// final linear are this unit's products:
//   k_conv_in_dw  the full 3x3 stride-2 conv of the mel features, 1 -> C
//               channels, + bias, ReLU (:222-226), fused into the first
//               depthwise 3x3 stride-2 conv, + bias (:231-236);
//               k_conv_in_dw_mx is its form on the f32 MFMA
//   k_dw_s2     the depthwise 3x3 stride-2 conv, + bias; its input takes
//               the previous pointwise conv's bias and ReLU on load  :237-244
//   k_flatten   the last pointwise conv's bias and ReLU, then the
//               channel-major flatten [t][c * F' + f] of :249-257
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "product.h"

namespace {

// the reference's stable sigmoid (src/qmat.h:31-35): exp only of -|x|, 1 / (1 +
// e) for x >= 0, e / (1 + e) below. One exponential and one division whatever
// the sign (as two branches a wave runs both: GLU and conv of 12000 x 1024 at
// 63 us, a third of it these).
__device__ __forceinline__ float sigmoid_f(float x) {
    const float e = expf(x >= 0.0f ? -x : x);
    return (x >= 0.0f ? 1.0f : e) / (1.0f + e);
}

// One wave per row of d = 256 V4 floats (lane l holds elements 4l + 256u ..
// +3): x += alpha res (stored; res may be null), then the layer norm into
// v: mean and var in double, inv = (float)(1 / sqrt(var + 1e-5)); v = ((x -
// (float)mean) * inv) * w + b in f32, as layer_norm_f. One pass sums the
// differences to the row's first element and their squares: (x[0] - mean)^2 <= d
// var, so what cancels in the variance is at most d^2 2^-53 of it. Two passes
// are twice the chain of double sums across the wave, which is most of the time
// when rows are few (a layer of 63 x 1024, five of these: 118 -> 116 us; of 1004
// x 1024, six: 290 -> 279 us).
template <int V4>
__device__ __forceinline__ void add_ln_row(float *xr, const float *__restrict__ rr, float alpha,
                                           const float *__restrict__ w, const float *__restrict__ b, int silu, int lane,
                                           float4 (&v)[V4]) {
    constexpr int d = 256 * V4;
    float4 wv[V4], bv[V4];
#pragma unroll
    for (int u = 0; u < V4; u++) {
        const int i = 4 * lane + 256 * u;
        v[u] = *(const float4 *)(xr + i);
        wv[u] = *(const float4 *)(w + i);
        bv[u] = *(const float4 *)(b + i);
    }
    if (rr) {
#pragma unroll
        for (int u = 0; u < V4; u++) {
            const float4 a = *(const float4 *)(rr + 4 * lane + 256 * u);
            v[u].x = fmaf(alpha, a.x, v[u].x);
            v[u].y = fmaf(alpha, a.y, v[u].y);
            v[u].z = fmaf(alpha, a.z, v[u].z);
            v[u].w = fmaf(alpha, a.w, v[u].w);
            *(float4 *)(xr + 4 * lane + 256 * u) = v[u];
        }
    }
    const double x0 = (double)__int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v[0].x)));
    double s = 0.0, q = 0.0;
#pragma unroll
    for (int u = 0; u < V4; u++) {
        const double c0 = (double)v[u].x - x0, c1 = (double)v[u].y - x0;
        const double c2 = (double)v[u].z - x0, c3 = (double)v[u].w - x0;
        s += (c0 + c1) + (c2 + c3);
        q += (c0 * c0 + c1 * c1) + (c2 * c2 + c3 * c3);
    }
    s = wave_sum(s);
    q = wave_sum(q);
    constexpr double rd = 1.0 / d;
    const double m = s * rd, mu = x0 + m;
    const float inv = (float)rsqrt_d(q * rd - m * m + 1e-5);
    const float muf = (float)mu;
#pragma unroll
    for (int u = 0; u < V4; u++) {
        v[u].x = ((v[u].x - muf) * inv) * wv[u].x + bv[u].x;
        v[u].y = ((v[u].y - muf) * inv) * wv[u].y + bv[u].y;
        v[u].z = ((v[u].z - muf) * inv) * wv[u].z + bv[u].z;
        v[u].w = ((v[u].w - muf) * inv) * wv[u].w + bv[u].w;
        if (silu) v[u] = float4{silu_f(v[u].x), silu_f(v[u].y), silu_f(v[u].z), silu_f(v[u].w)};
    }
}

// Four channels per lane of row m of an EXACT product's prepared input: the
// lane's half wave holds chunk c, lane l of it elements 4l .. 4l+3. The
// arithmetic of split_chunk; 8-byte stores, which the L2 joins with those of the
// neighbouring rows (the wave's next ones).
__device__ __forceinline__ void prep_store4(float4 v, int lane, size_t m, int c, int Kc, uint8_t *__restrict__ xp,
                                            float *__restrict__ xpf) {
    const int l32 = lane & 31, hu = l32 >> 2, hh = (l32 >> 1) & 1;
    float a = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    a = wave_max<32>(a);
    const int sh = chunk_shift(a);
    const float xs[4] = {ldexpf(v.x, sh), ldexpf(v.y, sh), ldexpf(v.z, sh), ldexpf(v.w, sh)};
    const half4v h = {(_Float16)xs[0], (_Float16)xs[1], (_Float16)xs[2], (_Float16)xs[3]};
    uint2 hw;
    __builtin_memcpy(&hw, &h, 8);
    const uint2 lw = {lo_pair(hw.x, xs[0], xs[1]), lo_pair(hw.y, xs[2], xs[3])};
    uint8_t *o = xp + ((((m >> 5) * Kc + c) * 8 + hu) * 2 * 64 + (m & 31) + 32 * hh) * 16 + 8 * (lane & 1);
    *(uint2 *)o = hw;
    *(uint2 *)(o + 64 * 16) = lw;
    if (l32 == 0) xpf[((m >> 5) * Kc + c) * 32 + (m & 31)] = ldexpf(1.0f, -sh);
}

// out = LN(x += alpha res), one wave per row. out may be x.
template <int V4>
__global__ __launch_bounds__(256) void k_add_ln(float *x, const float *__restrict__ res, float alpha,
                                                const float *__restrict__ w, const float *__restrict__ b,
                                                float *out, int rows, int silu) {
    constexpr int d = 256 * V4;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= rows) return;
    float4 v[V4];
    add_ln_row<V4>(x + (size_t)r * d, res ? res + (size_t)r * d : nullptr, alpha, w, b, silu, lane, v);
    float *orow = out + (size_t)r * d;
#pragma unroll
    for (int u = 0; u < V4; u++) *(float4 *)(orow + 4 * lane + 256 * u) = v[u];
}

// LN(x += alpha res) as the products' prepared input in EXACT numerics, in
// place of the f32 rows: the split of each row's 128-element chunks that the
// products' preparation forms (the same values: shift sh from the chunk's
// largest magnitude, hi = f16(v 2^sh), lo = f16(v 2^sh - hi), fold factor
// 2^-sh), in its layout
//   xp   [row group G][chunk][half-step u][hi, lo][64 slots][16 B], slot r + 32 hh
//        holding chunk elements 16u + 8hh .. +7 of row 32G + r
//   xpf  [G][chunk][32]
// Lane l's float4 u is chunk 2u + l / 32, elements 4 (l % 32) .. +3: half-step
// (l % 32) / 4, half hh = (l / 2) % 2, the 8-byte half l % 2 of the slot. A
// workgroup holds 8 consecutive rows (8 waves): for each (chunk, half-step,
// term, hh) their slots are one 128-byte line of xp. The pieces go to LDS
// first, in that line order, so that the stores to xp are whole lines (a
// wave's store covers 8 of them). Rows rows .. Mpad-1 are the zero rows the
// preparation pads with (fold factor 1).
template <int V4>
__global__ __launch_bounds__(512) void k_add_ln_prep(float *x, const float *__restrict__ res, float alpha,
                                                     const float *__restrict__ w, const float *__restrict__ b,
                                                     int rows, int silu, uint8_t *__restrict__ xp,
                                                     float *__restrict__ xpf) {
    constexpr int d = 256 * V4, Kc = d / 128, NL = Kc * 32;   // lines of the workgroup
    __shared__ uint4 stage[NL * 8];
    const int wave = threadIdx.x >> 6, m = blockIdx.x * 8 + wave, lane = threadIdx.x & 63;
    const int G = m >> 5, r = m & 31, l32 = lane & 31;
    float4 v[V4];
    if (m < rows) {
        add_ln_row<V4>(x + (size_t)m * d, res ? res + (size_t)m * d : nullptr, alpha, w, b, silu, lane, v);
    } else {
#pragma unroll
        for (int u = 0; u < V4; u++) v[u] = float4{0.f, 0.f, 0.f, 0.f};
    }
    const int hu = l32 >> 2, hh = (l32 >> 1) & 1;
#pragma unroll
    for (int u = 0; u < V4; u++) {
        const int c = 2 * u + (lane >> 5);
        float a = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
        const int sh = chunk_shift(wave_max<32>(a));
        const float xs[4] = {ldexpf(v[u].x, sh), ldexpf(v[u].y, sh), ldexpf(v[u].z, sh), ldexpf(v[u].w, sh)};
        _Float16 hv[4], lv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            hv[j] = (_Float16)xs[j];
            lv[j] = (_Float16)(xs[j] - (float)hv[j]);
        }
        uint2 hw, lw;
        __builtin_memcpy(&hw, hv, 8);
        __builtin_memcpy(&lw, lv, 8);
        // line ((c * 8 + hu) * 2 + term) * 2 + hh, slot wave (the row within the 8)
        uint8_t *o = (uint8_t *)stage + (((((c * 8 + hu) * 2) * 2 + hh) * 8 + wave) * 16 + 8 * (lane & 1));
        *(uint2 *)o = hw;
        *(uint2 *)(o + 2 * 8 * 16) = lw;
        if (l32 == 0) xpf[((size_t)G * Kc + c) * 32 + r] = ldexpf(1.0f, -sh);
    }
    __syncthreads();
    // line L = (q * 2 + hh), q = (c * 8 + hu) * 2 + term, lies at xp offset
    // (G * Kc * 16 + q) * 1024 + hh * 512 + (8-row block) * 128
    const int rb = (blockIdx.x & 3) * 128;
    uint8_t *gx = xp + (size_t)(blockIdx.x >> 2) * Kc * 16 * 1024 + rb;
#pragma unroll
    for (int i = threadIdx.x; i < NL * 8; i += 512) {
        const int L = i >> 3, sl = i & 7;
        *(uint4 *)(gx + (size_t)(L >> 1) * 1024 + (L & 1) * 512 + sl * 16) = stage[i];
    }
}

// g[r, i] = h[r, i] * sigmoid(h[r, d + i]); thread = 4 elements
__global__ __launch_bounds__(256) void k_glu(const float *__restrict__ h, float *__restrict__ g, size_t rows,
                                             int d) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x, d4 = d / 4;
    if (idx >= rows * d4) return;
    const size_t r = idx / d4, i = 4 * (idx - r * d4);
    const float4 a = *(const float4 *)(h + r * 2 * d + i), b = *(const float4 *)(h + r * 2 * d + d + i);
    const float4 o = {a.x * sigmoid_f(b.x), a.y * sigmoid_f(b.y), a.z * sigmoid_f(b.z), a.w * sigmoid_f(b.w)};
    *(float4 *)(g + r * d + i) = o;
}

// x * sigmoid(x) with the stable sigmoid (mynah_asr_silu)
__device__ __forceinline__ float silu_e(float x) { return x * sigmoid_f(x); }

// c[t, i] = dw_b[i] + sum_j w[i, j] * g[t - pc + j, i] over the taps inside
// the segment (in tap order from j0), then, with scale: silu(c * scale +
// shift). Thread = (row, 4 channels); the weights in the reference's order
// w[i][j] (the fallback for shapes the tiled form does not take).
__global__ __launch_bounds__(256) void k_dwconv(const float *__restrict__ g, const float *__restrict__ w,
                                                const float *__restrict__ bias, const float *__restrict__ scale,
                                                const float *__restrict__ shift, float *__restrict__ out, int T,
                                                int nseq, int d, int k, int pc) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int d4 = d / 4;
    if (idx >= (size_t)nseq * T * d4) return;
    const int row = (int)(idx / d4), i = 4 * (int)(idx - (size_t)row * d4);
    const int s = row / T, t = row - s * T;
    const float *gs = g + (size_t)s * T * d;
    float4 o = bias ? *(const float4 *)(bias + i) : float4{0.f, 0.f, 0.f, 0.f};
    const int j0 = t - pc < 0 ? pc - t : 0, j1 = t - pc + k > T ? T - t + pc : k;
    for (int j = j0; j < j1; j++) {
        const float4 src = *(const float4 *)(gs + (size_t)(t - pc + j) * d + i);
        const float *wj = w + (size_t)i * k + j;
        const float4 wv = {wj[0], wj[k], wj[2 * k], wj[3 * k]};
        o.x = fmaf(wv.x, src.x, o.x);
        o.y = fmaf(wv.y, src.y, o.y);
        o.z = fmaf(wv.z, src.z, o.z);
        o.w = fmaf(wv.w, src.w, o.w);
    }
    if (scale) {
        const float4 sc = *(const float4 *)(scale + i), sh = *(const float4 *)(shift + i);
        o.x = silu_e(fmaf(o.x, sc.x, sh.x));
        o.y = silu_e(fmaf(o.y, sc.y, sh.y));
        o.z = silu_e(fmaf(o.z, sc.z, sh.z));
        o.w = silu_e(fmaf(o.w, sc.w, sh.w));
    }
    *(float4 *)(out + (size_t)row * d + i) = o;
}

// The same in tiles: a workgroup = R rows of one segment x 256 channels. The
// rows t0 - pc .. t0 + R - 1 - pc + k - 1 of the GLU (zero outside the segment) are
// staged in LDS once, so each input row is read from memory once per tile
// instead of once per tap; wave w = rows R/4 w .. of the tile, lane = 4
// channels. Per output the operations and their order are those of k_dwconv
// (taps outside the segment skipped, not added as zeros).
// The GLU is formed from pw1's output h [rows][2d] as it is staged (k_glu's
// operations; the halo rows' values are formed again by the next tile).
// PREP: the output rows are written as the EXACT products' prepared input
// (xp, xpf, for M = nseq T rows padded to 64, as k_add_ln_prep writes it)
// instead of into out: per (row, 128-channel chunk: 32 lanes) the split the
// preparation forms, held in registers until the tile is done, then staged
// in the input rows' LDS so the stores run along rows.
//
// K: the kernel width where it is known at compile time (0: at run time). Then
// a tile that touches no segment end keeps its taps in registers and slides
// along its rows, reading each staged row once per wave instead of once per tap.
// R: 32 rows, or 8 when 32-row tiles are fewer than the CUs (a segment of 63
// frames is 8 tiles of 32 rows: each one long chain of loads; the halo, 8 rows
// per tile at width 9, is then read twice as often, from L2).
template <bool PREP, int R, int K>
__global__ __launch_bounds__(256) void k_dwconv_tile(const float *__restrict__ g, const float *__restrict__ w,
                                                     const float *__restrict__ bias, const float *__restrict__ scale,
                                                     const float *__restrict__ shift, float *__restrict__ out,
                                                     int T, int d, int kr, int pc, uint8_t *__restrict__ xp,
                                                     float *__restrict__ xpf) {
    // [R + k - 1][64] rows of g, then [k][64] taps; PREP, once the tile is
    // done: the staged slots [R rows][2 chunks][8 half-steps][2 terms][2
    // halves] over the rows, the fold factors [R][2] over the taps
    extern __shared__ float4 dws[];
    constexpr int RW = R / 4;   // rows per wave
    uint2 ph[PREP ? RW : 1], pl[PREP ? RW : 1];
    float pf[PREP ? RW : 1];
    const int k = K ? K : kr;
    const int tid = threadIdx.x, q = tid & 63, t0 = blockIdx.x * R, c0 = blockIdx.y * 256;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrow = R + k - 1;
    const int gw = 2 * d;   // the input's row width
    const float *gs = g + (size_t)blockIdx.z * T * gw + c0;
    float4 *taps = dws + nrow * 64;
    // the taps of w [d][k] written tap-major (each tap of 4 channels one
    // float4): thread = channel c0 + tid, its k taps, loaded ahead of the rows
    constexpr int KT = K ? K : 16;
    float tv[KT];
    const float *wc = w + (size_t)(c0 + tid) * k;
#pragma unroll
    for (int j = 0; j < KT; j++) tv[j] = j < k ? wc[j] : 0.0f;
    constexpr int UB = 4;   // rows of a wave in flight
    for (int i0 = wave; i0 < nrow; i0 += 4 * UB) {
        float4 a[UB], b[UB];
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const int r = i0 + 4 * u, t = t0 - pc + r;
            a[u] = float4{0.f, 0.f, 0.f, 0.f};
            b[u] = a[u];
            if (r < nrow && t >= 0 && t < T) {
                const float *p = gs + (size_t)t * gw + 4 * q;
                a[u] = *(const float4 *)p;
                b[u] = *(const float4 *)(p + d);
            }
        }
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const int r = i0 + 4 * u, t = t0 - pc + r;
            if (r >= nrow) continue;
            float4 o = a[u];
            if (t >= 0 && t < T)
                o = float4{o.x * sigmoid_f(b[u].x), o.y * sigmoid_f(b[u].y), o.z * sigmoid_f(b[u].z),
                           o.w * sigmoid_f(b[u].w)};
            dws[r * 64 + q] = o;
        }
    }
    {
        float *tf = (float *)taps;
#pragma unroll
        for (int j = 0; j < KT; j++)
            if (j < k) tf[j * 256 + tid] = tv[j];
    }
    const int i = c0 + 4 * q;
    const float4 b0 = bias ? *(const float4 *)(bias + i) : float4{0.f, 0.f, 0.f, 0.f};
    float4 sc = {0.f, 0.f, 0.f, 0.f}, sh = sc;
    if (scale) {
        sc = *(const float4 *)(scale + i);
        sh = *(const float4 *)(shift + i);
    }
    __syncthreads();
    float *os = out + (size_t)blockIdx.z * T * d + i;
    const int r0 = RW * wave;
    float4 o[RW];
#pragma unroll
    for (int u = 0; u < RW; u++) o[u] = b0;
    auto tap = [](float4 &acc, const float4 &wv, const float4 &src) {
        acc.x = fmaf(wv.x, src.x, acc.x);
        acc.y = fmaf(wv.y, src.y, acc.y);
        acc.z = fmaf(wv.z, src.z, acc.z);
        acc.w = fmaf(wv.w, src.w, acc.w);
    };
    if (K && t0 >= pc && t0 + R - 1 - pc + k - 1 < T && t0 + R <= T) {
        float4 wv[K ? K : 1];
#pragma unroll
        for (int j = 0; j < K; j++) wv[j] = taps[j * 64 + q];
#pragma unroll
        for (int r = 0; r < RW + K - 1; r++) {
            const float4 src = dws[(r0 + r) * 64 + q];
#pragma unroll
            for (int u = 0; u < RW; u++)
                if (r - u >= 0 && r - u < K) tap(o[u], wv[r - u], src);
        }
    } else {
#pragma unroll
        for (int u = 0; u < RW; u++) {
            const int t = t0 + r0 + u;
            const int j0 = t - pc < 0 ? pc - t : 0, j1 = t - pc + k > T ? T - t + pc : k;
            if (t < T)
                for (int j = j0; j < j1; j++) tap(o[u], taps[j * 64 + q], dws[(r0 + u + j) * 64 + q]);
        }
    }
#pragma unroll
    for (int u = 0; u < RW; u++) {
        const int t = t0 + r0 + u;
        if (t >= T) break;
        if (scale) {
            o[u].x = silu_e(fmaf(o[u].x, sc.x, sh.x));
            o[u].y = silu_e(fmaf(o[u].y, sc.y, sh.y));
            o[u].z = silu_e(fmaf(o[u].z, sc.z, sh.z));
            o[u].w = silu_e(fmaf(o[u].w, sc.w, sh.w));
        }
        if constexpr (PREP) {
            // lanes 32 cl .. 32 cl + 31 hold chunk cl's 128 channels of row t
            float a = fmaxf(fmaxf(fabsf(o[u].x), fabsf(o[u].y)), fmaxf(fabsf(o[u].z), fabsf(o[u].w)));
#pragma unroll
            for (int off = 16; off > 0; off >>= 1) a = fmaxf(a, __shfl_xor(a, off, 64));
            const int shf = chunk_shift(a);
            const float xs[4] = {ldexpf(o[u].x, shf), ldexpf(o[u].y, shf), ldexpf(o[u].z, shf), ldexpf(o[u].w, shf)};
            _Float16 hv[4], lv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                hv[j] = (_Float16)xs[j];
                lv[j] = (_Float16)(xs[j] - (float)hv[j]);
            }
            __builtin_memcpy(&ph[u], hv, 8);
            __builtin_memcpy(&pl[u], lv, 8);
            pf[u] = ldexpf(1.0f, -shf);
        } else {
            *(float4 *)(os + (size_t)t * d) = o[u];
        }
    }
    if constexpr (PREP) {
        __syncthreads();   // every wave is done with the input rows and the taps
        float4 *stage = dws;
        float *fold = (float *)(dws + R * 64);
        {
            const int l32 = q & 31, cl = q >> 5, hu = l32 >> 2, hh = (l32 >> 1) & 1;
#pragma unroll
            for (int u = 0; u < RW; u++) {
                const int rr = r0 + u;
                if (t0 + rr >= T) break;
                uint8_t *o8 = (uint8_t *)(stage + (((rr * 2 + cl) * 8 + hu) * 2) * 2 + hh) + 8 * (l32 & 1);
                *(uint2 *)o8 = ph[u];
                *(uint2 *)(o8 + 2 * 16) = pl[u];   // term 1: two slots on
                if (l32 == 0) fold[rr * 2 + cl] = pf[u];
            }
        }
        __syncthreads();
        const int Kc = d / 128;
        const size_t mb = (size_t)blockIdx.z * T;
        // 64 slots per row; consecutive threads run along the rows
        for (int p = tid; p < R * 64; p += 256) {
            const int rr = p % R, rest = p / R;
            const int cl = rest >> 5, hu = (rest >> 2) & 7, term = (rest >> 1) & 1, hh = rest & 1;
            const int t = t0 + rr;
            if (t < T) {
                const size_t m = mb + t;
                const int chunk = 2 * blockIdx.y + cl;
                *(float4 *)(xp + ((((m >> 5) * Kc + chunk) * 8 + hu) * 2 * 64 + term * 64 + (m & 31) + 32 * hh) * 16) =
                    stage[(((rr * 2 + cl) * 8 + hu) * 2 + term) * 2 + hh];
            }
        }
        if (tid < 2 * R) {
            const int rr = tid % R, cl = tid / R, t = t0 + rr;
            if (t < T) {
                const size_t m = mb + t;
                xpf[((m >> 5) * Kc + 2 * blockIdx.y + cl) * 32 + (m & 31)] = fold[rr * 2 + cl];
            }
        }
        // the rows past M up to the 64-row padding: zeros (fold factor 1), as
        // the preparation pads; by the last tile of the last segment
        if (blockIdx.z == gridDim.z - 1 && blockIdx.x == gridDim.x - 1) {
            const size_t M = (size_t)gridDim.z * T, Mp = (M + 63) / 64 * 64;
            for (size_t i = tid; i < (Mp - M) * 64; i += 256) {
                const size_t m = M + (i >> 6);
                const int rest = (int)(i & 63), cl = rest >> 5, hu = (rest >> 2) & 7, term = (rest >> 1) & 1,
                          hh = rest & 1;
                const int chunk = 2 * blockIdx.y + cl;
                *(float4 *)(xp + ((((m >> 5) * Kc + chunk) * 8 + hu) * 2 * 64 + term * 64 + (m & 31) + 32 * hh) * 16) =
                    float4{0.f, 0.f, 0.f, 0.f};
                if (rest == 0 || rest == 32) xpf[((m >> 5) * Kc + chunk) * 32 + (m & 31)] = 1.0f;
            }
        }
    }
}

// The first two stages in one pass: out[s][to][fo][c] = the depthwise 3x3
// stride-2 conv (+ b1) of y = relu(conv_in(x) + b0), the 1 -> C 3x3 stride-2
// conv of the mel features (subsampling.c:222-226, 231-236). y is formed
// where a depthwise tap reads it and never stored (at config 5 it would be
// 2 GB written and read back). Per tap the operations are those of the
// conv alone (nine fmas from zero in tap order, + b0, ReLU) and of the
// depthwise conv (a product, then eight fmas, + b1 last); a tap outside
// y's [T1, F1] reads zero (the depthwise conv's pad), and a mel sample
// outside [T, F] reads zero (the first conv's pad).
//
// One wave per output row (s, to) and run of FS columns fo, its lanes over the
// channels 4 at a time, sliding along fo: the 3 x 3 window of y a depthwise
// output reads stays in registers, and each step forms y's two new columns (y
// column 2 of one step is column 0 of the next). Each lane holds its channels'
// 2 x 9 taps. The 7 mel rows the wave reads lie in its own LDS with the pads as
// zeros, column k at word k + 1, so that a step reads its four new columns of a
// row as one 16-byte broadcast (the fifth is the last step's last). Loads of
// single mel samples behind their bounds, through the scalar cache, made a step
// a chain of about 30 waits: 138 us at 4 segments of 6000 frames (6000 rows of
// 20 columns, 256 channels), where its fmas take 55.
// For channels that are no multiple of 128; the others take k_conv_in_dw_mx.
// Weights tap-major, w0[j][C] and w1[j][C].
constexpr int CI_FS = 32;   // columns per wave at most
__global__ __launch_bounds__(256) void k_conv_in_dw(const float *__restrict__ x, const float *__restrict__ w0,
                                                    const float *__restrict__ b0, const float *__restrict__ w1,
                                                    const float *__restrict__ b1, float *__restrict__ out, int nseq,
                                                    int T, int F, int T1, int F1, int To, int Fo, int C, int pl,
                                                    int FS, int parts) {
    constexpr int WC = 4 * CI_FS + 4;
    __shared__ __align__(16) float win[4][7][WC];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + wave), wrow = wid / parts;
    if (wrow >= nseq * To) return;   // (no workgroup barrier follows)
    const int to = wrow % To, s = wrow / To, f0 = (wid - wrow * parts) * FS, f9 = min(f0 + FS, Fo);
    const float *xs = x + (size_t)s * T * F;
    // window column k: mel f = 4 f0 - 3 pl + k; window row j: mel t = 4 to - 3 pl + j
    const int cols = 4 * (f9 - f0) + 4;
    for (int k = lane; k < cols; k += 64) {
        const int f = 4 * f0 - 3 * pl + k - 1;
#pragma unroll
        for (int j = 0; j < 7; j++) {
            const int t = 4 * to - 3 * pl + j;
            win[wave][j][k] = t >= 0 && t < T && f >= 0 && f < F ? xs[(size_t)t * F + f] : 0.0f;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int c = 4 * lane; c < C; c += 256) {
        float4 wa[9], wb[9];
#pragma unroll
        for (int j = 0; j < 9; j++) {
            wa[j] = *(const float4 *)(w0 + (size_t)j * C + c);
            wb[j] = *(const float4 *)(w1 + (size_t)j * C + c);
        }
        const float4 bb0 = *(const float4 *)(b0 + c), bb1 = *(const float4 *)(b1 + c);
        float mel[7][5];   // columns 4i+2 .. 4i+6 of step i
        // y at (t1 = 2 to - pl + r, f1): relu(b0 + conv_in) over the mel columns
        // from m0 of the step, zero outside [T1, F1]
        auto yat = [&](int r, int f1, int m0) {
            const int t1 = 2 * to - pl + r;
            float4 ci = {0.f, 0.f, 0.f, 0.f};
            if (t1 >= 0 && t1 < T1 && f1 >= 0 && f1 < F1) {
#pragma unroll
                for (int dt = 0; dt < 3; dt++)
#pragma unroll
                    for (int df = 0; df < 3; df++) {
                        const float v = mel[2 * r + dt][m0 + df];
                        const float4 wv = wa[3 * dt + df];
                        ci.x = fmaf(wv.x, v, ci.x);
                        ci.y = fmaf(wv.y, v, ci.y);
                        ci.z = fmaf(wv.z, v, ci.z);
                        ci.w = fmaf(wv.w, v, ci.w);
                    }
                ci = float4{fmaxf(ci.x + bb0.x, 0.0f), fmaxf(ci.y + bb0.y, 0.0f), fmaxf(ci.z + bb0.z, 0.0f),
                            fmaxf(ci.w + bb0.w, 0.0f)};
            }
            return ci;
        };
        float4 yw[3][3];
#pragma unroll
        for (int j = 0; j < 7; j++) {   // columns 0, 1, 2
            const float4 a = *(const float4 *)&win[wave][j][0];
            mel[j][0] = a.y, mel[j][1] = a.z, mel[j][2] = a.w;
        }
#pragma unroll
        for (int r = 0; r < 3; r++) yw[r][2] = yat(r, 2 * f0 - pl, 0);
#pragma unroll
        for (int j = 0; j < 7; j++) mel[j][4] = mel[j][2];
        for (int fo = f0; fo < f9; fo++) {
#pragma unroll
            for (int j = 0; j < 7; j++) {
                mel[j][0] = mel[j][4];
                const float4 a = *(const float4 *)&win[wave][j][4 * (fo - f0) + 4];
                mel[j][1] = a.x, mel[j][2] = a.y, mel[j][3] = a.z, mel[j][4] = a.w;
            }
#pragma unroll
            for (int r = 0; r < 3; r++) {
                yw[r][0] = yw[r][2];
                yw[r][1] = yat(r, 2 * fo - pl + 1, 0);
                yw[r][2] = yat(r, 2 * fo - pl + 2, 2);
            }
            float4 acc = {wb[0].x * yw[0][0].x, wb[0].y * yw[0][0].y, wb[0].z * yw[0][0].z, wb[0].w * yw[0][0].w};
#pragma unroll
            for (int j = 1; j < 9; j++) {
                const float4 wv = wb[j], y = yw[j / 3][j % 3];
                acc.x = fmaf(wv.x, y.x, acc.x);
                acc.y = fmaf(wv.y, y.y, acc.y);
                acc.z = fmaf(wv.z, y.z, acc.z);
                acc.w = fmaf(wv.w, y.w, acc.w);
            }
            acc = float4{bb1.x + acc.x, bb1.y + acc.y, bb1.z + acc.z, bb1.w + acc.w};
            const size_t m = (size_t)wrow * Fo + fo;
            *(float4 *)(out + m * C + c) = acc;
        }
    }
}

// The same for channels that are a multiple of 128, with the first conv on the
// f32 MFMA. A workgroup is 32 consecutive output rows m = (s, to, fo) by 128
// channels, wave w channels 32w .. 32w + 31: for each of the nine depthwise
// taps y comes as five 32 x 32 x 2 MFMAs (rows = channels, columns = output
// rows, K = the nine mel samples and a zero), starting from b0, and goes into
// the tap's fma where it lies. Each lane holds 16 channels of one output row, so
// nothing moves between lanes, and rows of any T and F fill the tiles. The mel
// samples come to LDS once per workgroup in the B operand's order.
// On the VALU the first conv's fmas alone are 216 of about 330 instructions per
// wave and step, which bounds k_conv_in_dw: 95 us at 4 segments of 6000 frames of
// 80 features, 256 channels, 87 here (both traced; the whole subsampling 330 ->
// 314 us). The 45 MFMAs of a tile are 35 us of it at the
// f32 MFMA's nominal rate and the rows' 123 MB 25; what is left is the chain of
// a tap (five dependent MFMAs, then their fmas). A neighbour's column would
// save a third of the MFMAs but lies in other lanes.
// PREP: the pointwise product's prepared input, its 64-row padding as zeros: the
// arithmetic of prep_store4, the chunk's maximum over the four waves.
template <bool PREP>
__global__ __launch_bounds__(256, 4) void k_conv_in_dw_mx(const float *__restrict__ x, const float *__restrict__ w0,
                                                       const float *__restrict__ b0, const float *__restrict__ w1,
                                                       const float *__restrict__ b1, float *__restrict__ out, int M,
                                                       int T, int F, int T1, int F1, int To, int Fo, int C, int pl,
                                                       uint8_t *__restrict__ xp, float *__restrict__ xpf) {
    __shared__ float win[7][7][32];   // mel rows 4 to - 3 pl .., columns 4 fo - 3 pl .. of each output row
    __shared__ __align__(16) float wd[9][128];
    __shared__ float wm[4][32];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = (int)blockIdx.x * 32 + l32, c0 = 128 * (int)blockIdx.y, cw = c0 + 32 * wave;
    const bool live = m < M;
    const unsigned mm = live ? m : 0, row = mm / (unsigned)Fo, s = row / (unsigned)To;
    const int fo = (int)(mm - row * Fo), to = (int)(row - s * To);
    // half wave g takes window row g: all loads go out before the first is stored
    const int g7 = 2 * wave + hh, t = 4 * to - 3 * pl + g7;
    const bool tin = live && g7 < 7 && (unsigned)t < (unsigned)T;
    const float *xr = x + (tin ? ((size_t)s * T + t) * F : 0);
    float v[7];
#pragma unroll
    for (int u = 0; u < 7; u++) {
        const int f = 4 * fo - 3 * pl + u;
        const bool in = tin && (unsigned)f < (unsigned)F;
        const float e = xr[in ? f : 0];
        v[u] = in ? e : 0.0f;
    }
    float a[5];   // A operand: channel l32, sample 2j + hh
#pragma unroll
    for (int j = 0; j < 5; j++) a[j] = 2 * j + hh < 9 ? w0[(size_t)(2 * j + hh) * C + cw + l32] : 0.0f;
    f16v bias;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const float4 b = *(const float4 *)(b0 + cw + 8 * g + 4 * hh);
        bias[4 * g] = b.x, bias[4 * g + 1] = b.y, bias[4 * g + 2] = b.z, bias[4 * g + 3] = b.w;
    }
    for (int i = tid; i < 9 * 32; i += 256)
        *(float4 *)&wd[i >> 5][4 * (i & 31)] = *(const float4 *)(w1 + (size_t)(i >> 5) * C + c0 + 4 * (i & 31));
    if (g7 < 7)
#pragma unroll
        for (int u = 0; u < 7; u++) win[g7][u][l32] = v[u];
    __syncthreads();
    const float *bp[5];   // B operand: output row l32, sample 2j + hh of tap (0, 0)
#pragma unroll
    for (int j = 0; j < 5; j++) bp[j] = 2 * j + hh < 9 ? &win[(2 * j + hh) / 3][(2 * j + hh) % 3][l32] : &win[0][0][l32];
    float4 o[4];
#pragma unroll
    for (int g = 0; g < 4; g++) o[g] = float4{0.f, 0.f, 0.f, 0.f};
    // (unrolled, the compiler reads every tap ahead at one wave per SIMD: the whole
    // subsampling 408 us; three taps unrolled at three waves: 323; rolled, the
    // waves of a SIMD overlap each other's MFMAs and fmas)
#pragma unroll 1
    for (int y = 0; y < 9; y++) {
        f16v acc = bias;
        const int r = y / 3, cc = y - 3 * r, at = (2 * r * 7 + 2 * cc) * 32;
        float bv[5];
#pragma unroll
        for (int j = 0; j < 5; j++) bv[j] = bp[j][at];
        __builtin_amdgcn_sched_barrier(0);   // (one wait for all five, not one in front of each MFMA)
        bv[4] = hh ? 0.0f : bv[4];   // (the tenth sample)
#pragma unroll
        for (int j = 0; j < 5; j++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], bv[j], acc, 0, 0, 0);
        // ReLU; zero outside y's [T1, F1]
        const bool yin = (unsigned)(2 * to - pl + r) < (unsigned)T1 && (unsigned)(2 * fo - pl + cc) < (unsigned)F1;
        const float lim = yin ? INFINITY : 0.0f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4 wv = *(const float4 *)&wd[y][32 * wave + 8 * g + 4 * hh];
            const float4 yv = {__builtin_amdgcn_fmed3f(acc[4 * g], 0.0f, lim),
                               __builtin_amdgcn_fmed3f(acc[4 * g + 1], 0.0f, lim),
                               __builtin_amdgcn_fmed3f(acc[4 * g + 2], 0.0f, lim),
                               __builtin_amdgcn_fmed3f(acc[4 * g + 3], 0.0f, lim)};
            o[g].x = fmaf(wv.x, yv.x, o[g].x);
            o[g].y = fmaf(wv.y, yv.y, o[g].y);
            o[g].z = fmaf(wv.z, yv.z, o[g].z);
            o[g].w = fmaf(wv.w, yv.w, o[g].w);
        }
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const float4 b = *(const float4 *)(b1 + cw + 8 * g + 4 * hh);
        o[g] = float4{b.x + o[g].x, b.y + o[g].y, b.z + o[g].z, b.w + o[g].w};
        if constexpr (!PREP)
            if (live) *(float4 *)(out + (size_t)m * C + cw + 8 * g + 4 * hh) = o[g];
    }
    if constexpr (PREP) {
        float am = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            if (!live) o[g] = float4{0.f, 0.f, 0.f, 0.f};
            am = fmaxf(am, fmaxf(fmaxf(fabsf(o[g].x), fabsf(o[g].y)), fmaxf(fabsf(o[g].z), fabsf(o[g].w))));
        }
        am = fmaxf(am, __shfl_xor(am, 32, 64));
        if (hh == 0) wm[wave][l32] = am;
        __syncthreads();
        am = fmaxf(fmaxf(wm[0][l32], wm[1][l32]), fmaxf(wm[2][l32], wm[3][l32]));
        const int sh = chunk_shift(am), Kc = C / 128;
        const size_t mc = (size_t)blockIdx.x * Kc + blockIdx.y;   // (32 rows, chunk)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float xv[4] = {ldexpf(o[g].x, sh), ldexpf(o[g].y, sh), ldexpf(o[g].z, sh), ldexpf(o[g].w, sh)};
            const half4v h = {(_Float16)xv[0], (_Float16)xv[1], (_Float16)xv[2], (_Float16)xv[3]};
            uint2 hw;
            __builtin_memcpy(&hw, &h, 8);
            const uint2 lw = {lo_pair(hw.x, xv[0], xv[1]), lo_pair(hw.y, xv[2], xv[3])};
            // channels 32 wave + 8 g + 4 hh ..: half-step 2 wave + g / 2, slot half g % 2
            uint8_t *p = xp + ((mc * 8 + 2 * wave + (g >> 1)) * 2 * 64 + l32 + 32 * (g & 1)) * 16 + 8 * hh;
            *(uint2 *)p = hw;
            *(uint2 *)(p + 64 * 16) = lw;
        }
        if (tid < 32) xpf[mc * 32 + l32] = ldexpf(1.0f, -sh);
    }
}

// out[s][to][fo][c] = b[c] + sum w[c][3 dt + df] in[s][2 to - pl + dt][2 fo - pl + df][c],
// in the reference's term order (the nine products summed left to right,
// subsampling.c:96-98); with pb, each input value is relu(in + pb[c]) first.
// The weights tap-major, wt[j][c].
// PREP (C of 256: a wave is 256 channels of one row): as the next product's
// prepared input, with its padding rows.
template <bool PREP>
__global__ __launch_bounds__(256) void k_dw_s2(const float *__restrict__ in, const float *__restrict__ pb,
                                               const float *__restrict__ wt, const float *__restrict__ b,
                                               float *__restrict__ out, int nseq, int T, int F, int To, int Fo,
                                               int C, int pl, uint8_t *__restrict__ xp, float *__restrict__ xpf) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int C4 = C / 4, lane = threadIdx.x & 63;
    const size_t row = idx / C4, rows = (size_t)nseq * To * Fo;
    const int c = 4 * (int)(idx - row * C4);
    if (row >= rows) {
        if constexpr (PREP)
            if (row < (rows + 63) / 64 * 64) prep_store4(float4{0.f, 0.f, 0.f, 0.f}, lane, row, c >> 7, C / 128, xp, xpf);
        return;
    }
    const int fo = (int)(row % Fo), to = (int)((row / Fo) % To), s = (int)(row / ((size_t)Fo * To));
    const float *is = in + (size_t)s * T * F * C;
    const float4 pbv = pb ? *(const float4 *)(pb + c) : float4{0.f, 0.f, 0.f, 0.f};
    float4 v[9];
#pragma unroll
    for (int dt = 0; dt < 3; dt++)
#pragma unroll
        for (int df = 0; df < 3; df++) {
            const int t = 2 * to - pl + dt, f = 2 * fo - pl + df;
            float4 a = {0.f, 0.f, 0.f, 0.f};
            if (t >= 0 && t < T && f >= 0 && f < F) {
                a = *(const float4 *)(is + ((size_t)t * F + f) * C + c);
                if (pb) {
                    a.x = fmaxf(a.x + pbv.x, 0.0f);
                    a.y = fmaxf(a.y + pbv.y, 0.0f);
                    a.z = fmaxf(a.z + pbv.z, 0.0f);
                    a.w = fmaxf(a.w + pbv.w, 0.0f);
                }
            }
            v[3 * dt + df] = a;
        }
    float4 wv = *(const float4 *)(wt + c);
    float4 acc = {wv.x * v[0].x, wv.y * v[0].y, wv.z * v[0].z, wv.w * v[0].w};
#pragma unroll
    for (int j = 1; j < 9; j++) {
        wv = *(const float4 *)(wt + (size_t)j * C + c);
        acc.x = fmaf(wv.x, v[j].x, acc.x);
        acc.y = fmaf(wv.y, v[j].y, acc.y);
        acc.z = fmaf(wv.z, v[j].z, acc.z);
        acc.w = fmaf(wv.w, v[j].w, acc.w);
    }
    const float4 bb = *(const float4 *)(b + c);
    acc = float4{bb.x + acc.x, bb.y + acc.y, bb.z + acc.z, bb.w + acc.w};
    if constexpr (PREP) prep_store4(acc, lane, row, c >> 7, C / 128, xp, xpf);
    else *(float4 *)(out + row * C + c) = acc;
}

// flat[s * To + t][c * Fo + f] = relu(in[s][t][f][c] + pb[c]); thread = one
// output element, consecutive threads along f then c (coalesced writes)
__global__ __launch_bounds__(256) void k_flatten(const float *__restrict__ in, const float *__restrict__ pb,
                                                 float *__restrict__ flat, size_t rows, int Fo, int C) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t CF = (size_t)C * Fo;
    if (idx >= rows * CF) return;
    const size_t r = idx / CF;
    const int j = (int)(idx - r * CF), c = j / Fo, f = j - c * Fo;
    const float v = in[(r * Fo + f) * C + c] + pb[c];
    flat[idx] = v < 0.0f ? 0.0f : v;
}

// The same as the linear's prepared input (C of 256): a workgroup takes one row,
// read along c into LDS and written along c * Fo + f by half waves of one
// chunk each; the workgroups past the rows write the padding.
__global__ __launch_bounds__(256) void k_flatten_prep(const float *__restrict__ in, const float *__restrict__ pb,
                                                      int rows, int Fo, int C, uint8_t *__restrict__ xp,
                                                      float *__restrict__ xpf) {
    extern __shared__ float row[];   // [Fo][C + 1]
    const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, CF = C * Fo;
    if (r < rows) {
        for (int i = 4 * tid; i < CF; i += 1024) {
            const int f = i / C, c = i - f * C;
            const float4 a = *(const float4 *)(in + (size_t)r * CF + i);
            const float v[4] = {a.x + pb[c], a.y + pb[c + 1], a.z + pb[c + 2], a.w + pb[c + 3]};
#pragma unroll
            for (int j = 0; j < 4; j++) row[f * (C + 1) + c + j] = v[j] < 0.0f ? 0.0f : v[j];
        }
        __syncthreads();
    }
    for (int j = 4 * tid; j < CF; j += 1024) {   // (CF of 256: whole waves)
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int c = (j + u) / Fo, f = j + u - c * Fo;
            v[u] = r < rows ? row[f * (C + 1) + c] : 0.0f;
        }
        prep_store4(float4{v[0], v[1], v[2], v[3]}, lane, (size_t)r, j >> 7, CF / 128, xp, xpf);
    }
}

// wt[z][j][c] = w_z[c][j] for w_z [C][9]: the per-channel taps of the three
// 3 x 3 convs tap-major, in one launch
__global__ __launch_bounds__(256) void k_transpose(const float *__restrict__ wa, const float *__restrict__ wb,
                                                   const float *__restrict__ wc, float *__restrict__ wt, int C) {
    const int idx = blockIdx.x * 256 + threadIdx.x, z = blockIdx.y;
    if (idx >= C * 9) return;
    const int j = idx / C, c = idx - j * C;
    const float *w = z == 0 ? wa : (z == 1 ? wb : wc);
    wt[(size_t)z * C * 9 + idx] = w[(size_t)c * 9 + j];
}

// y[r][i] = (y[r][i] + b[i]) * scale (the subsampling's linear bias, then
// the layer input scale: encoder.c:958-959)
__global__ __launch_bounds__(256) void k_bias_scale(float *__restrict__ y, const float *__restrict__ b, size_t rows,
                                                    int d, float scale) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * d) return;
    const int i = (int)(idx % d);
    const float v = y[idx] + b[i];
    y[idx] = scale != 1.0f ? v * scale : v;
}

}  // namespace

// the widths k_add_ln is instantiated for: 256 V4 with V4 = 1..8, 12, 16
bool mh_enc_d_supported(int d) {
    if (d <= 0 || d % 256) return false;
    const int v = d / 256;
    return v <= 8 || v == 12 || v == 16;
}

hipError_t mh_launch_add_ln(float *x, const float *res, float alpha, const float *w, const float *b, float *out,
                            int rows, int d, bool silu, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    if (!mh_enc_d_supported(d)) return hipErrorInvalidValue;
    const dim3 grid((rows + 3) / 4), blk(256);
    switch (d / 256) {
    case 1: hipLaunchKernelGGL(k_add_ln<1>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 2: hipLaunchKernelGGL(k_add_ln<2>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 3: hipLaunchKernelGGL(k_add_ln<3>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 4: hipLaunchKernelGGL(k_add_ln<4>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 5: hipLaunchKernelGGL(k_add_ln<5>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 6: hipLaunchKernelGGL(k_add_ln<6>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 7: hipLaunchKernelGGL(k_add_ln<7>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 8: hipLaunchKernelGGL(k_add_ln<8>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 12: hipLaunchKernelGGL(k_add_ln<12>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    case 16: hipLaunchKernelGGL(k_add_ln<16>, grid, blk, 0, st, x, res, alpha, w, b, out, rows, silu); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// d = 256 .. 2048 (wider rows would spill at two waves per SIMD)
bool mh_add_ln_prep_supported(int d) { return d > 0 && d % 256 == 0 && d / 256 <= 8; }

hipError_t mh_launch_add_ln_prep(float *x, const float *res, float alpha, const float *w, const float *b, int rows,
                                 int d, bool silu, uint8_t *xp, float *xpf, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    if (!mh_add_ln_prep_supported(d)) return hipErrorInvalidValue;
    const dim3 grid(mh_mpad(rows) / 8), blk(512);
    switch (d / 256) {
#define LNP(V) \
    case V: hipLaunchKernelGGL(k_add_ln_prep<V>, grid, blk, 0, st, x, res, alpha, w, b, rows, silu, xp, xpf); break;
    LNP(1) LNP(2) LNP(3) LNP(4) LNP(5) LNP(6) LNP(7) LNP(8)
#undef LNP
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t mh_launch_glu(const float *h, float *g, size_t rows, int d, hipStream_t st) {
    if (!rows) return hipSuccess;
    if (d % 4) return hipErrorInvalidValue;
    const size_t n = rows * (size_t)(d / 4);
    hipLaunchKernelGGL(k_glu, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, h, g, rows, d);
    return hipGetLastError();
}

constexpr int DW_R = 32;   // rows of a large tile

bool mh_glu_dwconv_supported(int d, int k) {
    return d > 0 && d % 256 == 0 && k > 0 && sizeof(float4) * 64 * (size_t)(DW_R + 2 * k - 1) <= 64 * 1024;
}

// odd widths up to 15 with the width known at compile time, the rest (even
// widths and 1) at run time; 8-row tiles when 32-row ones are fewer than the CUs
template <bool PREP, int R>
static hipError_t dwconv_tile(const float *g, const float *w, const float *bias, const float *scale, const float *shift,
                              float *out, int T, int nseq, int d, int k, int pc, uint8_t *xp, float *xpf,
                              hipStream_t st) {
    // (>= the staged slots and folds: R rows and 2 R floats, which the taps' rows cover only for k > 1)
    const size_t lds = sizeof(float4) * 64 * (size_t)(R + 2 * k - 1);
    const dim3 grid((unsigned)((T + R - 1) / R), d / 256, nseq);
    switch (k) {
#define DWK(K)                                                                                                        \
    case K:                                                                                                           \
        hipLaunchKernelGGL((k_dwconv_tile<PREP, R, K>), grid, dim3(256), lds, st, g, w, bias, scale, shift, out, \
                           T, d, k, pc, xp, xpf);                                                                     \
        break;
        DWK(3) DWK(5) DWK(7) DWK(9) DWK(11) DWK(13) DWK(15)
#undef DWK
    default:
        hipLaunchKernelGGL((k_dwconv_tile<PREP, R, 0>), grid, dim3(256), lds, st, g, w, bias, scale, shift, out, T, d,
                           k, pc, xp, xpf);
    }
    return hipGetLastError();
}

template <bool PREP>
static hipError_t dwconv_rows(const float *g, const float *w, const float *bias, const float *scale, const float *shift,
                              float *out, int T, int nseq, int d, int k, int pc, uint8_t *xp, float *xpf,
                              hipStream_t st) {
    if ((long)((T + DW_R - 1) / DW_R) * (d / 256) * nseq < 256)
        return dwconv_tile<PREP, 8>(g, w, bias, scale, shift, out, T, nseq, d, k, pc, xp, xpf, st);
    return dwconv_tile<PREP, DW_R>(g, w, bias, scale, shift, out, T, nseq, d, k, pc, xp, xpf, st);
}

hipError_t mh_launch_glu_dwconv(const float *h, const float *w, const float *bias, const float *scale,
                                const float *shift, float *out, int T, int nseq, int d, int k, int causal,
                                uint8_t *xp, float *xpf, hipStream_t st) {
    if (T <= 0 || nseq <= 0) return hipSuccess;
    if (!mh_glu_dwconv_supported(d, k)) return hipErrorInvalidValue;
    const int pc = causal ? k - 1 : (k - 1) / 2;
    if (xp) return dwconv_rows<true>(h, w, bias, scale, shift, out, T, nseq, d, k, pc, xp, xpf, st);
    return dwconv_rows<false>(h, w, bias, scale, shift, out, T, nseq, d, k, pc, nullptr, nullptr, st);
}

hipError_t mh_launch_dwconv(const float *g, const float *w, const float *bias, const float *scale,
                            const float *shift, float *out, int T, int nseq, int d, int k, int causal,
                            hipStream_t st) {
    if (T <= 0 || nseq <= 0) return hipSuccess;
    if (d % 4 || k <= 0) return hipErrorInvalidValue;
    const int pc = causal ? k - 1 : (k - 1) / 2;
    const size_t n = (size_t)nseq * T * (d / 4);
    hipLaunchKernelGGL(k_dwconv, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, w, bias, scale, shift, out,
                       T, nseq, d, k, pc);
    return hipGetLastError();
}

int mh_ss_out_len(int n, int causal) {
    // (n + pl + pr - 3) / 2 + 1 with pads (2, 1) causal, (1, 1) otherwise
    const int p = causal ? 3 : 2;
    return (n + p - 3) / 2 + 1;
}

hipError_t mh_launch_conv_in_dw(const float *x, const float *w0, const float *b0, const float *w1, const float *b1,
                                float *out, int nseq, int T, int F, int C, int causal, uint8_t *xp, float *xpf,
                                hipStream_t st) {
    if (C % 4 || (xp && C % 128)) return hipErrorInvalidValue;
    const int T1 = mh_ss_out_len(T, causal), F1 = mh_ss_out_len(F, causal);
    const int To = mh_ss_out_len(T1, causal), Fo = mh_ss_out_len(F1, causal), pl = causal ? 2 : 1;
    if (T1 <= 0 || F1 <= 0 || To <= 0 || Fo <= 0) return hipSuccess;
    const size_t rows = (size_t)nseq * To, M = rows * Fo;   // output rows (s, to), and (s, to, fo)
    if (!rows) return hipSuccess;
    if (M > 0x7fffff00) return hipErrorInvalidValue;
    if (C % 128 == 0) {
        if (C / 128 > 65535) return hipErrorInvalidValue;
        const dim3 grid((unsigned)(xp ? (M + 63) / 64 * 2 : (M + 31) / 32), C / 128);
        if (xp)
            hipLaunchKernelGGL(k_conv_in_dw_mx<true>, grid, dim3(256), 0, st, x, w0, b0, w1, b1, out, (int)M, T, F, T1,
                               F1, To, Fo, C, pl, xp, xpf);
        else
            hipLaunchKernelGGL(k_conv_in_dw_mx<false>, grid, dim3(256), 0, st, x, w0, b0, w1, b1, out, (int)M, T, F, T1,
                               F1, To, Fo, C, pl, xp, xpf);
        return hipGetLastError();
    }
    // A wave takes whole rows while they fill the chip (1024 SIMDs, 3 waves
    // each), else part of one: a part forms one column of y more
    int FS = Fo < CI_FS ? Fo : CI_FS;
    while (FS > 4 && rows * ((Fo + FS - 1) / FS) < 2048) FS = (FS + 1) / 2;
    const int parts = (Fo + FS - 1) / FS;
    if (rows * parts > 0x7fffff00) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_conv_in_dw, dim3((unsigned)((rows * parts + 3) / 4)), dim3(256), 0, st, x, w0, b0, w1, b1, out,
                       nseq, T, F, T1, F1, To, Fo, C, pl, FS, parts);
    return hipGetLastError();
}

hipError_t mh_launch_dw_s2(const float *in, const float *pb, const float *w, const float *b, float *out, int nseq,
                           int T, int F, int C, int causal, uint8_t *xp, float *xpf, hipStream_t st) {
    if (C % 4 || (xp && C % 256)) return hipErrorInvalidValue;
    const int To = mh_ss_out_len(T, causal), Fo = mh_ss_out_len(F, causal), pl = causal ? 2 : 1;
    const size_t rows = (size_t)nseq * To * Fo;
    if (!rows) return hipSuccess;
    const size_t n = (xp ? (rows + 63) / 64 * 64 : rows) * (C / 4);
    const dim3 grid((unsigned)((n + 255) / 256));
    if (xp)
        hipLaunchKernelGGL(k_dw_s2<true>, grid, dim3(256), 0, st, in, pb, w, b, out, nseq, T, F, To, Fo, C, pl, xp, xpf);
    else
        hipLaunchKernelGGL(k_dw_s2<false>, grid, dim3(256), 0, st, in, pb, w, b, out, nseq, T, F, To, Fo, C, pl, xp,
                           xpf);
    return hipGetLastError();
}

// the row k_flatten_prep holds in LDS, with its padding
bool mh_flatten_prep_supported(int Fo, int C) { return C % 256 == 0 && (size_t)Fo * (C + 1) * 4 <= 65536; }

hipError_t mh_launch_flatten_prep(const float *in, const float *pb, size_t rows, int Fo, int C, uint8_t *xp,
                                  float *xpf, hipStream_t st) {
    if (!mh_flatten_prep_supported(Fo, C) || rows > 0x7fffff00) return hipErrorInvalidValue;
    if (!rows) return hipSuccess;
    hipLaunchKernelGGL(k_flatten_prep, dim3((unsigned)((rows + 63) / 64 * 64)), dim3(256),
                       (size_t)Fo * (C + 1) * sizeof(float), st, in, pb, (int)rows, Fo, C, xp, xpf);
    return hipGetLastError();
}

hipError_t mh_launch_flatten(const float *in, const float *pb, float *flat, size_t rows, int Fo, int C,
                             hipStream_t st) {
    const size_t n = rows * (size_t)C * Fo;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_flatten, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, pb, flat, rows, Fo, C);
    return hipGetLastError();
}

hipError_t mh_launch_bias_scale(float *y, const float *b, size_t rows, int d, float scale, hipStream_t st) {
    const size_t n = rows * (size_t)d;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_bias_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, b, rows, d, scale);
    return hipGetLastError();
}

hipError_t mh_launch_transpose_taps(const float *wa, const float *wb, const float *wc, float *wt, int C,
                                    hipStream_t st) {
    if (C <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_transpose, dim3((C * 9 + 255) / 256, 3), dim3(256), 0, st, wa, wb, wc, wt, C);
    return hipGetLastError();
}
