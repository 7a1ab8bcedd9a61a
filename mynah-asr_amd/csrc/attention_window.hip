// attention_window.hip — the relative-position self-attention core for
// chunked-limited windows (the reference's src/encoder.c:220-313; the windows of
// :373-381), on the f32 MFMA of gfx950 (v_mfma_f32_16x16x4_f32).
//
// Per head h (columns h*DK .. h*DK+DK-1 of the [T, d] buffers), chunk = right +
// 1 and lc = left / chunk, row t (chunk t/chunk) sees the keys
// [(t/chunk - lc) * chunk, (t/chunk + 1) * chunk) clipped to [0, T):
//   s[t, j] = ((q[t] + bias_u) . k[j] + (q[t] + bias_v) . rk[T-1 + j - t]) / sqrt(DK)
//   ctx[t]  = sum_j softmax_j(s[t, j]) v[j]
// rk = pe . relk_w^T is [2T-1, d] (shared by the segments of one call).
//
// f32 products and sums throughout, and no workspace: a (finite) key outside a
// row's window meets a probability of exactly 0, so a row's bits depend on the
// keys it sees and on nothing else; calls on several streams share nothing, and a
// call under stream capture allocates nothing.
// Not on full attention's f16 hi + lo operands (attention.hip): [70, 13], 16 x 750
// frames, d 1024, 8 heads take 134 us there and 172 here (a layer of 4 x 251
// frames 287 and 297 us), but its V split has one exponent per 32 keys and
// feature, so keys that a row does not see take bits from those it does (hidden
// rows 2^20 times larger: off by more than the header's bound), and its planes
// need a workspace, which calls on two streams, or replays of two graphs, share.
//
// Sums. A score is two sums of DK / 2 products, added; a tile's P . V is summed
// from zero and then joins the context. Relative error against 64 bits (2-norm,
// N(0, 1) inputs) at [70, 13], 750 frames, d 1024, 8 heads: 2.8e-7, with one chain
// each 4.2e-7 (3.1e-7 on the split operands); at [200, 50], 1000 frames, d 512
// 3.2e-7, 5.1e-7 (3.5e-7). It costs 3% of the call.
//
// One workgroup = two waves = 32 query rows of one head of one segment; wave w
// owns rows t0 + 16w .. +15 (wider blocks visit more keys that their rows cannot
// see). Keys are visited in tiles of 32 from the first one the block's rows see;
// each tile's K and V are staged in LDS, and the 48 rk rows of the block's
// position columns stay in an LDS ring that takes 32 new rows per tile; every
// wave
//   1. forms the content scores (16 x 32) with its (q + bias_u) held in registers,
//   2. forms the position scores (q + bias_v) . rk for its 16 rows in tiles of
//      16 offsets delta = j - t: a key tile needs 47 offsets (three tiles),
//      the first of which the previous key tile computed as its last (carried
//      in registers), so each key tile costs two position tiles, no more MFMA
//      work than the content scores,
//   3. applies the rel-shift through a per-wave LDS scratch (row i, key jj
//      reads band column jj - i + 15),
//   4. runs an online softmax (running row max and sum, base-2 exponentials of
//      scores pre-scaled by log2(e)/sqrt(DK)), and
//   5. multiplies the probabilities (re-laid out as an MFMA A operand through
//      LDS) by the V tile and adds that to its 16 x DK context, rescaled.
//
// MFMA 16x16x4 f32 operand layout (lane l, c = l & 15, g = l >> 4):
//   A: row c, k-slot g;  B: column c, k-slot g;  D: rows 4g + e (e = 0..3), column c.
// The reduction index of the score products is permuted so each lane reads a
// contiguous run: step s, slot g carries feature NS*g + s (NS = DK / 4).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "product.h"

namespace {

constexpr int KT = 32;          // keys per tile
constexpr int NW = 2;           // waves per workgroup, 16 query rows each
constexpr int NTH = 64 * NW;
constexpr int RB = 16 * NW;     // query rows per workgroup
constexpr int NB = RB + KT - 16;   // rk rows a key tile reads (all waves' position columns): the ring

template <int DK> struct WinLds {
    static constexpr int KS = DK + 4;   // K / rk row stride (16-byte rows, conflict-free b128 reads)
    static constexpr int VT = KT + 4;   // V is stored transposed, [DK][VT]: conflict-free b128 reads
    static constexpr int BS = 53;       // band scratch row stride
    static constexpr int PS = 36;       // probability scratch row stride
    static constexpr int K0 = 0;
    static constexpr int V0 = K0 + KT * KS;
    static constexpr int R0 = V0 + DK * VT;
    static constexpr int W0 = R0 + NB * KS;
    static constexpr int WSZ = 16 * BS;   // the probabilities reuse the band scratch
    static constexpr int TOTAL = W0 + NW * WSZ;   // floats
    static_assert(R0 % 4 == 0 && W0 % 4 == 0 && WSZ % 4 == 0, "16-byte rows");
};

__device__ __forceinline__ f4 mfma16(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Reductions over the 16 lanes of a DPP row (the lanes holding one score row):
// swap neighbours, swap pairs, mirror within 8, mirror within 16. Every lane
// ends with the same value (each step combines a and b symmetrically).
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float max16(float x) {
    x = fmaxf(x, dpp<0xB1>(x));    // quad_perm [1,0,3,2]
    x = fmaxf(x, dpp<0x4E>(x));    // quad_perm [2,3,0,1]
    x = fmaxf(x, dpp<0x141>(x));   // row_half_mirror
    x = fmaxf(x, dpp<0x140>(x));   // row_mirror
    return x;
}
__device__ __forceinline__ float sum16(float x) {
    x += dpp<0xB1>(x);
    x += dpp<0x4E>(x);
    x += dpp<0x141>(x);
    x += dpp<0x140>(x);
    return x;
}

struct Window {
    int chunk, lc, T;
    __device__ int j0(int t) const { return max((t / chunk - lc) * chunk, 0); }
    __device__ int j1(int t) const { return min((t / chunk + 1) * chunk, T); }
};

template <int DK>
__global__ __launch_bounds__(NTH, 1) void k_attn_win(const float *__restrict__ q, const float *__restrict__ k,
                                                     const float *__restrict__ v, const float *__restrict__ rk,
                                                     const float *__restrict__ bu, const float *__restrict__ bv,
                                                     float *__restrict__ ctx, int T, int d, int left, int right,
                                                     float kscale) {
    using L = WinLds<DK>;
    constexpr int NS = DK / 4;    // reduction steps of a score product
    constexpr int NT = DK / 16;   // context column tiles
    extern __shared__ __attribute__((aligned(16))) float wlds[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int c = lane & 15, g = lane >> 4;
    // XCD-aware order (query block bx, head by, segment bz): the query blocks
    // of one (segment, head) read the same K and V rows, and the segments of
    // one head the same rk rows, so they run on one XCD and share its L2
    int bx, by, bz;
    xcd_order(bx, by, bz);
    const int ho = by * DK;
    const size_t so = (size_t)bz * (size_t)T * (size_t)d;
    q += so;
    k += so;
    v += so;
    ctx += so;
    const int t0 = bx * RB, tw = t0 + 16 * w;
    const Window win{right + 1, left / (right + 1), T};
    const int ja = win.j0(t0), jb = win.j1(min(t0 + RB - 1, T - 1));

    // (q + bias_u), (q + bias_v) of query row tw + c, features NS*g .. NS*g + NS-1
    float qa[NS], qb[NS];
    {
        const int t = tw + c;
        const int f = ho + NS * g;
#pragma unroll
        for (int i = 0; i < NS / 4; i++) {
            f4 x = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
            if (t < T) {
                x = *(const f4 *)(q + (size_t)t * d + f + 4 * i);
                u = x + *(const f4 *)(bu + f + 4 * i);
                b = x + *(const f4 *)(bv + f + 4 * i);
            }
            qa[4 * i + 0] = u.x; qa[4 * i + 1] = u.y; qa[4 * i + 2] = u.z; qa[4 * i + 3] = u.w;
            qb[4 * i + 0] = b.x; qb[4 * i + 1] = b.y; qb[4 * i + 2] = b.z; qb[4 * i + 3] = b.w;
        }
    }
    // this lane's output rows tw + 4g + e and their windows
    int rj0[4], rj1[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = min(tw + 4 * g + e, T - 1);
        rj0[e] = win.j0(t);
        rj1[e] = win.j1(t);
    }
    float m[4], l[4];
    f4 acc[NT];
#pragma unroll
    for (int e = 0; e < 4; e++) m[e] = -1e30f, l[e] = 0.f;
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = f4{0.f, 0.f, 0.f, 0.f};

    float *Ks = wlds + L::K0, *Vs = wlds + L::V0, *Rs = wlds + L::R0;
    float *Bw = wlds + L::W0 + w * L::WSZ, *Pw = Bw;
    const int P = 2 * T - 1;

    // The next tile's K, V and rk rows are loaded into registers while the
    // current tile computes, then written to LDS between two barriers. Rows
    // past the ends are clamped, not zeroed: a key j outside [0, T) is masked
    // out of every score, and an rk row p outside [0, 2T-2] only pairs a query
    // row t >= T (never stored) or a masked key.
    //
    // The rk rows form a ring of NB rows: key tile ti (0 = the tile before
    // the first) reads window rows 32 ti .. 32 ti + NB - 1 (absolute rk row
    // pb0 + v for window row v), in slot v mod NB; moving to the next tile
    // retires the 32 lowest and stages 32 new ones into their slots.
    constexpr int UKV = KT * DK / 4 / NTH;
    static_assert(UKV * NTH == KT * DK / 4, "staging split");
    f4 gk[UKV], gv[UKV], gr[UKV];
    const int pb0 = T + (ja - KT) - t0 - (RB - 16);
    auto gload = [&](int jt, int ti) {
#pragma unroll
        for (int u = 0; u < UKV; u++) {
            const int i = tid + NTH * u;
            const int r = i / (DK / 4), cc = 4 * (i % (DK / 4));
            const int kr = min(max(jt + r, 0), T - 1);
            gk[u] = *(const f4 *)(k + (unsigned)(kr * d + ho + cc));   // (< 2^31: checked at launch)
            const int rv = i % KT, cv = 4 * (i / KT);   // V: lanes along keys (transposed store)
            gv[u] = *(const f4 *)(v + (unsigned)(min(max(jt + rv, 0), T - 1) * d + ho + cv));
        }
#pragma unroll
        for (int u = 0; u < UKV; u++) {
            const int i = tid + NTH * u, r = i / (DK / 4), cc = 4 * (i % (DK / 4));
            const int p = min(max(pb0 + 32 * ti + NB - 32 + r, 0), P - 1);
            gr[u] = *(const f4 *)(rk + (unsigned)(p * d + ho + cc));
        }
    };
    auto lstore = [&](int ti) {
#pragma unroll
        for (int u = 0; u < UKV; u++) {
            const int i = tid + NTH * u, r = i / (DK / 4), cc = 4 * (i % (DK / 4));
            *(f4 *)(Ks + r * L::KS + cc) = gk[u];
            const int rv = i % KT, cv = 4 * (i / KT);
#pragma unroll
            for (int e = 0; e < 4; e++) Vs[(cv + e) * L::VT + rv] = gv[u][e];
        }
#pragma unroll
        for (int u = 0; u < UKV; u++) {
            const int i = tid + NTH * u, r = i / (DK / 4), cc = 4 * (i % (DK / 4));
            const int slot = (32 * ti + NB - 32 + r) % NB;
            *(f4 *)(Rs + slot * L::KS + cc) = gr[u];
        }
    };
    // Position columns are computed in tiles of 16 offsets delta = j - t.
    // For key tile jt the wave needs delta in [b, b+47), b = jt - tw - 15:
    // tiles D0 = [b, b+16), D1, D2. The next key tile's D0 is this tile's D2,
    // so it is carried in registers and every tile computes only D1 and D2
    // (rk rows T-1 + b + 16 .. + 47: staged row (RB - 16) - 16w + col).
    const int prow = (RB - 16) - 16 * w;
    f4 carry = {0.f, 0.f, 0.f, 0.f};
    {
        // D0 of the first tile = D2 of the tile before it: tile 0's whole
        // window of rk rows (slots 0 .. NB-1), then its position tile D2
        for (int i = tid; i < NB * DK / 4; i += NTH) {
            const int r = i / (DK / 4), cc = 4 * (i % (DK / 4));
            const int p = min(max(pb0 + r, 0), P - 1);
            *(f4 *)(Rs + r * L::KS + cc) = *(const f4 *)(rk + (size_t)p * d + ho + cc);
        }
        __syncthreads();
        const float *rw = Rs + ((prow + 16 + c) % NB) * L::KS + NS * g;
        f4 cp[2] = {carry, carry};
#pragma unroll
        for (int i = 0; i < NS / 4; i++) {
            const f4 rx = *(const f4 *)(rw + 4 * i);
#pragma unroll
            for (int u = 0; u < 4; u++) cp[i / (NS / 8)] = mfma16(qb[4 * i + u], rx[u], cp[i / (NS / 8)]);
        }
        carry = cp[0] + cp[1];
        gload(ja, 1);
    }

    // ring slots of this lane's window rows at tile ti, carried from tile to
    // tile (each tile moves them 32 rows on)
    int rb0 = (32 + prow + c) % NB;
    for (int jt = ja, ti = 1; jt < jb; jt += KT, ti++) {
        const int rr[2] = {rb0, rb0 + 16 >= NB ? rb0 + 16 - NB : rb0 + 16};
        rb0 = rb0 + 32 >= NB ? rb0 + 32 - NB : rb0 + 32;
        __syncthreads();   // every wave is done with the previous tile
        lstore(ti);
        __syncthreads();
        if (jt + KT < jb) gload(jt + KT, ti + 1);

        // 1. content scores (16 rows x 32 keys), 2. position tiles D1, D2
        f4 sp[2][2], bp[2][2];   // [half of the features][tile of 16]
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int n = 0; n < 2; n++) sp[h][n] = bp[h][n] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NS / 4; i++) {
            f4 kx[2], rx[2];
#pragma unroll
            for (int n = 0; n < 2; n++) kx[n] = *(const f4 *)(Ks + (16 * n + c) * L::KS + NS * g + 4 * i);
#pragma unroll
            for (int n = 0; n < 2; n++) rx[n] = *(const f4 *)(Rs + rr[n] * L::KS + NS * g + 4 * i);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int h = i / (NS / 8);
                sp[h][0] = mfma16(qa[4 * i + u], kx[0][u], sp[h][0]);
                sp[h][1] = mfma16(qa[4 * i + u], kx[1][u], sp[h][1]);
                bp[h][0] = mfma16(qb[4 * i + u], rx[0][u], bp[h][0]);
                bp[h][1] = mfma16(qb[4 * i + u], rx[1][u], bp[h][1]);
            }
        }
        const f4 s[2] = {sp[0][0] + sp[1][0], sp[0][1] + sp[1][1]};
        const f4 bd[2] = {bp[0][0] + bp[1][0], bp[0][1] + bp[1][1]};
        // 3. rel-shift: row i = 4g + e, key jj = 16n + c takes band column jj - i + 15
        //    (delta = jt + jj - (tw + i) = b + (jj - i + 15))
#pragma unroll
        for (int e = 0; e < 4; e++) {
            Bw[(4 * g + e) * L::BS + c] = carry[e];
            Bw[(4 * g + e) * L::BS + 16 + c] = bd[0][e];
            Bw[(4 * g + e) * L::BS + 32 + c] = bd[1][e];
        }
        carry = bd[1];
        wave_lds_order();
        float sv[2][4];
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int i = 4 * g + e, j = jt + 16 * n + c;
                const float x = (s[n][e] + Bw[i * L::BS + 16 * n + c - i + 15]) * kscale;
                sv[n][e] = (unsigned)(j - rj0[e]) < (unsigned)(rj1[e] - rj0[e]) ? x : -INFINITY;
            }
        // 4. online softmax over the tile
        float alpha[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float mx = max16(fmaxf(sv[0][e], sv[1][e]));
            const float mn = fmaxf(m[e], mx);
            alpha[e] = exp2f(m[e] - mn);
            m[e] = mn;
            sv[0][e] = exp2f(sv[0][e] - mn);
            sv[1][e] = exp2f(sv[1][e] - mn);
            l[e] = l[e] * alpha[e] + sum16(sv[0][e] + sv[1][e]);
        }
        // 5. probabilities to the A layout (row c, keys 8g .. 8g+7), then P . V
        wave_lds_order();   // the band reads above precede these writes
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int e = 0; e < 4; e++) Pw[(4 * g + e) * L::PS + 16 * n + c] = sv[n][e];
        wave_lds_order();
        const f4 pa0 = *(const f4 *)(Pw + c * L::PS + 8 * g);
        const f4 pa1 = *(const f4 *)(Pw + c * L::PS + 8 * g + 4);
        const float pa[8] = {pa0.x, pa0.y, pa0.z, pa0.w, pa1.x, pa1.y, pa1.z, pa1.w};
        // B operand: column 16n + c, keys 8g .. 8g+7 of the transposed V tile
        f4 vb[2][2];
        auto rdv = [&](int n, f4 *vx) {
            const float *vr = Vs + (16 * n + c) * L::VT + 8 * g;
            vx[0] = *(const f4 *)vr;
            vx[1] = *(const f4 *)(vr + 4);
        };
        rdv(0, vb[0]);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            if (n + 1 < NT) rdv(n + 1, vb[(n + 1) & 1]);
            const f4 *vx = vb[n & 1];
            f4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 8; u++) o = mfma16(pa[u], vx[u >> 2][u & 3], o);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[n][e] = fmaf(acc[n][e], alpha[e], o[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = tw + 4 * g + e;
        if (t < T) {
            const float inv = 1.0f / l[e];
            float *o = ctx + (size_t)t * d + ho + c;
#pragma unroll
            for (int n = 0; n < NT; n++) o[16 * n] = acc[n][e] * inv;
        }
    }
}

template <int DK>
hipError_t launch_win(const float *q, const float *k, const float *v, const float *rk, const float *bu, const float *bv,
                      float *ctx, int T, int d, int H, int left, int right, int nseq, hipStream_t st) {
    if ((size_t)(2 * (size_t)T) * d >= 0x7fffffffu) return hipErrorInvalidValue;   // 32-bit row offsets
    constexpr int bytes = sizeof(float) * WinLds<DK>::TOTAL;
    // set once per instantiation (thread-safe static initialisation)
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)k_attn_win<DK>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return attr;
    // exponentials are base 2: scores carry log2(e) / sqrt(DK)
    const float kscale = (1.0f / sqrtf((float)DK)) * 1.4426950408889634f;
    hipLaunchKernelGGL((k_attn_win<DK>), dim3((T + RB - 1) / RB, H, nseq), dim3(NTH), bytes, st, q, k, v, rk, bu, bv,
                       ctx, T, d, left, right, kscale);
    return hipGetLastError();
}

}  // namespace

hipError_t mh_launch_relpos_attn_win(const float *q, const float *k, const float *v, const float *rk,
                                     const float *bias_u, const float *bias_v, float *ctx, int T, int d, int H,
                                     int left, int right, int nseq, hipStream_t st) {
    if (d / H == 128)
        return launch_win<128>(q, k, v, rk, bias_u, bias_v, ctx, T, d, H, left, right, nseq, st);
    if (d / H == 64)
        return launch_win<64>(q, k, v, rk, bias_u, bias_v, ctx, T, d, H, left, right, nseq, st);
    return hipErrorInvalidValue;
}
