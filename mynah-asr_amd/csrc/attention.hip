// attention.hip — the relative-position self-attention core of the FastConformer
// encoder layer over the full window (the reference's src/encoder.c:315-410), on
// the f16 MFMA of gfx950 from split operands. Chunked-limited windows take
// attention_window.hip.
//
// Per head h (columns h*DK .. h*DK+DK-1 of the [T, d] buffers):
//   s[t, j] = ((q[t] + bias_u) . k[j] + (q[t] + bias_v) . rk[T-1 + j - t]) / sqrt(DK)
//   ctx[t]  = sum_j softmax_j(s[t, j]) v[j],  j over [0, T)
// rk = pe . relk_w^T is [2T-1, d] (the pos projection's output, shared by the
// segments of one call).
//
// Operands. Each row of q + bias, K and rk (per head) is scaled by the power of
// two 2^e that puts its largest magnitude in [2^14, 2^15) and split into f16
// pairs hi + lo (hi = f16(x 2^e), lo = f16(x 2^e - hi)), which hold x to 2^-22
// of the row's maximum; a score is hi.hi + hi.lo + lo.hi summed in f32 (the
// dropped lo.lo is below 2^-22 of the same scale) and multiplied by 2^-(e_q +
// e_k), which is exact. V is split likewise per (tile of 32 keys, feature), the
// probabilities (<= 256: the running maximum moves only by steps above 2^8) at
// the fixed scale 2^6; one exact power of two per tile and feature undoes both.
// The softmax is fp32.
//
// k_attn_split writes K, rk and V once per call in the order the MFMAs read
// them (one 16-byte fragment per lane, 1 KiB per load), so the attention kernel
// needs no LDS staging for them and its waves no barriers between tiles.
//
// k_attn: a workgroup = 32 query rows of one head of one segment; its NW waves
// share the rows' split q + bias (in LDS) and take contiguous runs of the key
// tiles (32 keys) side by side, each with its own running maximum, sum and 32 x
// DK context; these meet in LDS at the end. Per tile a wave
//   1. forms the content scores transposed, K . q^T (lane = one query, 16 keys),
//   2. forms the position scores rk . (q + bias_v)^T of 32 offsets delta = j -
//      t: a tile needs 63 of them (two blocks of 32), the first of which are the
//      previous tile's, so a tile costs one block, the MFMA work of the content,
//   3. shifts them through a 64-key ring of LDS per wave (the block's offset
//      delta of query c belongs to key delta + c),
//   4. runs the online softmax: in-lane over 16 keys and one cross-lane step,
//   5. multiplies the probabilities, already the MFMA's A operand (V's fragments
//      hold a tile's keys in that order), by the V tile into the context.
// What bounds it: the fragments, 48 KiB per wave and tile (DK 128) through the
// 64 B/clk L1 path (6100 of the 7800 cycles that eight waves of a CU take for a
// tile each), then the MFMAs (72 of 32 cycles, 4600 cycles on each SIMD) and
// about 400 VALU instructions. At T = 750 a workgroup takes 65 100 cycles: 13 750
// until its first tile (rows, first operands and position block), 46 500 for the
// tiles, 4600 to join the contexts. The chip holds 1.73 to 1.83 GHz meanwhile, so
// the six rounds of 512 workgroups of 16 x 750 frames are 220 of the kernel's 240
// us; the rest is their start and end.
// Measured, d 1024, 8 heads, full window, with the splits: 16 x 750 frames 430 ->
// 275 us, 1 x 750 118 -> 36, 1 x 63 28 -> 13 (before: 128-row blocks staging K, V
// and rk in LDS). No faster, each measured: eight waves per workgroup (15% slower
// at 16 x 750), two query blocks per workgroup sharing K and V through L1, two
// MFMA chains per product, the products' loads two phases ahead.
//
// MFMA 32x32x16 f16 operands (lane l, c = l & 31, hh = l >> 5): A row c, B column
// c, k-slots 8 hh + j (j = 0..7); D column c, rows 8i + 4hh + jj in element 4i + jj.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "product.h"

namespace {

constexpr int KT = 32;   // keys per tile, query rows per workgroup
constexpr int NW = 4;    // waves per workgroup, two workgroups per CU

// The exponent s that puts a row's largest magnitude amax in [2^14, 2^15)
// (0 for a row of zeros or a non-finite amax: its products are then what
// f16 makes of them, as the f32 products would be infinite or NaN)
__device__ __forceinline__ int row_exp(float amax) {
    if (!(amax > 0.0f) || !(amax < INFINITY)) return 0;
    int E;
    (void)frexpf(amax, &E);
    return min(max(15 - E, -120), 120);
}

// x[j] * 2^s as f16 pairs: hi = f16(y), lo = f16(y - hi); y - hi is exact in
// f32, so hi + lo keeps 22 bits of x
__device__ __forceinline__ void split8u(const float (&y)[8], half8 &h, half8 &l) {
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int j = 0; j < 8; j++) h[j] = (_Float16)y[j];
    __builtin_memcpy(hw, &h, 16);
#pragma unroll
    for (int t = 0; t < 4; t++) lw[t] = lo_pair(hw[t], y[2 * t], y[2 * t + 1]);
    __builtin_memcpy(&l, lw, 16);
}
__device__ __forceinline__ void split8(const float (&x)[8], int s, half8 &h, half8 &l) {
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; j++) y[j] = ldexpf(x[j], s);
    split8u(y, h, l);
}

// The split operands in fragment order. A tile is [DK/16 half-steps][hi, lo]
// [64 lanes][16 B]: lane (r, hh) of half-step u holds features 16u + 8hh .. +7
// of row r.
//   k   [segment][head][tile], keys 32 tile + r;  ke [..][32]: minus each row's e
//   r   [head][2 ntile blocks], block b = offsets' rows T + 32 (b - ntile) + r of
//       rk (zeros outside [0, 2T-2]);             re [..][32] likewise
//   v   [segment][head][tile] as [DK/32 feature groups][2 k-steps][hi, lo][64]
//       [16 B]: lane (f, hh) of k-step u holds feature f of the group and keys 16u +
//       8 (j >> 2) + 4hh + (j & 3) of the tile;   vs [..][DK]: 2^-(6 + e)
// xp (DK = 128, may be null): the context is written as the EXACT products'
// prepared input (the f16 split of each row's 128-element chunks, a chunk
// being one head, with the fold factors xpf, for M = nseq T rows padded to
// mh_mpad(M)) in place of ctx, for the output projection.
struct Planes {
    half8 *k, *r, *v;
    int *ke, *re;
    float *vs;
    int ntile;
    uint8_t *xp;
    float *xpf;
};

template <int DK> struct AttnLds {
    static constexpr int NU = DK / 16;
    static constexpr int Q = 2 * NU * 2 * 1024;          // [u, v bias][NU][hi, lo][64][16 B]
    static constexpr int RING = 64 * 32 * 4;             // per wave: [64 keys][32 queries]
    static constexpr int OS = DK + 8;                    // context row stride: the lane halves' rows 4 apart
    static constexpr int O = NW * 32 * OS * 4;           // (over Q and the rings, once the tiles are done)
    static constexpr int BODY = Q + NW * RING > O ? Q + NW * RING : O;
    // row maxima [2][2 NU][32], exponents [2][32], the waves' maxima and sums
    // [NW][32], the waves' tile exponents [NW][32]
    static constexpr int X = (4 * NU + 2 + 3 * NW) * 32 * 4;
    static constexpr int BYTES = BODY + X;
};

template <int DK>
__global__ __launch_bounds__(64 * NW, 2) void k_attn(const float *__restrict__ q, const float *__restrict__ bu,
                                                     const float *__restrict__ bv, float *__restrict__ ctx, int T,
                                                     int d, float kscale, Planes P) {
    using L = AttnLds<DK>;
    constexpr int NU = L::NU, NF = DK / 32, NUW = (NU + NW - 1) / NW;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    half8 *Q = (half8 *)lds;
    float *X = (float *)(lds + L::BODY);
    int *EQ = (int *)(X + 4 * NU * 32);
    float *ML = X + (4 * NU + 2) * 32;
    const int c = lane & 31, hh = lane >> 5;
    // XCD-aware order (query block bx, head by, segment bz): the query blocks
    // of one (segment, head) read the same K and V planes, and the segments of
    // one head the same rk rows, so they run on one XCD and share its L2
    int bx, by, bz;
    xcd_order(bx, by, bz);
    const int H = gridDim.y, ho = by * DK, t0 = 32 * bx, n = P.ntile;
    const int ta = n * w / NW, tb = n * (w + 1) / NW;   // this wave's key tiles [ta, tb)
    float *ring = (float *)(lds + L::Q + w * L::RING);
    const size_t bh = (size_t)bz * H + by;
    // (uniform bases and one 32-bit lane offset: scalar address arithmetic)
    const uint8_t *kp = (const uint8_t *)(P.k + bh * P.ntile * (DK * 8)), *vp = (const uint8_t *)(P.v + bh * P.ntile * (DK * 8));
    const uint8_t *rp = (const uint8_t *)(P.r + (size_t)by * (2 * n) * (DK * 8));
    const int *ke = P.ke + bh * P.ntile * 32, *re = P.re + (size_t)by * (2 * n) * 32;
    const float *vs = P.vs + bh * P.ntile * DK;
    const unsigned lo16 = lane * 16u;
    auto frag = [&](const uint8_t *base, size_t tile, int i) {   // fragment i of a tile
        return *(const half8 *)(base + (tile * (DK / 8) + i) * 1024 + lo16);
    };

    constexpr int HU = NU / 2;
    half8 kf[NU][2], rf[NU][2];
    int ek = 0, er = 0;   // row c's exponents of the key tile and the position block
    auto load_r = [&](int t, int u0) {   // half the fragments of tile t's second block
#pragma unroll
        for (int u = 0; u < HU; u++)
#pragma unroll
            for (int p = 0; p < 2; p++) rf[u0 + u][p] = frag(rp, (size_t)(t - bx + n), 2 * (u0 + u) + p);
    };
    // the rows' (q + bias_u), (q + bias_v), split, into LDS in B-operand order:
    // wave w forms half-steps w, w + NW, ... Loads return in order: the rows
    // first, then the first operands (the position block before the first
    // tile's, the first tile's keys), which land while the rows are prepared.
    {
        f4 xq[NUW][2], xu[NUW][2], xv[NUW][2];
#pragma unroll
        for (int i = 0; i < NUW; i++) {
            const int u = w + NW * i;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                xq[i][j] = xu[i][j] = xv[i][j] = f4{0.f, 0.f, 0.f, 0.f};
                if (u < NU && t0 + c < T) {
                    const int f = ho + 16 * u + 8 * hh + 4 * j;
                    xq[i][j] = *(const f4 *)(q + ((size_t)bz * T + t0 + c) * d + f);
                    xu[i][j] = *(const f4 *)(bu + f);
                    xv[i][j] = *(const f4 *)(bv + f);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ta < tb) {
            load_r(ta - 1, 0);
            load_r(ta - 1, HU);
            er = re[(size_t)(ta - 1 - bx + n) * 32 + c];
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int p = 0; p < 2; p++) kf[u][p] = frag(kp, ta, 2 * u + p);
            ek = ke[(size_t)ta * 32 + c];
        }
        __builtin_amdgcn_sched_barrier(0);
        float xa[NUW][8], xb[NUW][8];
#pragma unroll
        for (int i = 0; i < NUW; i++) {
            const int u = w + NW * i;
            float ma = 0.0f, mb = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                xa[i][j] = xq[i][j >> 2][j & 3] + xu[i][j >> 2][j & 3];
                xb[i][j] = xq[i][j >> 2][j & 3] + xv[i][j >> 2][j & 3];
                ma = fmaxf(ma, fabsf(xa[i][j]));
                mb = fmaxf(mb, fabsf(xb[i][j]));
            }
            if (u < NU) {
                X[(2 * u + hh) * 32 + c] = ma;
                X[(2 * NU + 2 * u + hh) * 32 + c] = mb;
            }
        }
        __syncthreads();
        float ma = 0.0f, mb = 0.0f;
#pragma unroll
        for (int i = 0; i < 2 * NU; i++) {
            ma = fmaxf(ma, X[i * 32 + c]);
            mb = fmaxf(mb, X[(2 * NU + i) * 32 + c]);
        }
        const int ea = row_exp(ma), eb = row_exp(mb);
#pragma unroll
        for (int i = 0; i < NUW; i++) {
            const int u = w + NW * i;
            if (u < NU) {
                half8 h, l;
                split8(xa[i], ea, h, l);
                Q[(2 * u) * 64 + lane] = h;
                Q[(2 * u + 1) * 64 + lane] = l;
                split8(xb[i], eb, h, l);
                Q[(2 * (NU + u)) * 64 + lane] = h;
                Q[(2 * (NU + u) + 1) * 64 + lane] = l;
            }
        }
        if (w == 0 && hh == 0) EQ[c] = -ea, EQ[32 + c] = -eb;   // negated: the unscale adds them
    }
    __syncthreads();
    const int eqa = EQ[c], eqb = EQ[32 + c];

    // position scores of block b (offsets' rows) -> the ring, as tile t's
    // second block: offset delta' of query c belongs to key 32 t + c + 1 + delta'
    int *es = (int *)ML + (2 * NW + w) * 32;
    // this lane's 16 rows' exponents, from one per lane through LDS (as 16-byte
    // loads of the rows they would cost the L1 path an eighth of its time)
    auto rows_e = [&](int e1, int (&o)[16]) {
        wave_lds_order();
        if (hh == 0) es[c] = e1;
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int4 v = *(const int4 *)(es + 8 * i + 4 * hh);
            o[4 * i] = v.x, o[4 * i + 1] = v.y, o[4 * i + 2] = v.z, o[4 * i + 3] = v.w;
        }
    };
    auto ring_put = [&](const f16v &bd, int er, int t) {
        const unsigned x = (unsigned)(32 * t + c + 1 + 4 * hh) * 32u;
        int ee[16];
        rows_e(er, ee);
#pragma unroll
        for (int e = 0; e < 16; e++)
            ring[((x + (8 * (e >> 2) + (e & 3)) * 32u) & 2047u) | (unsigned)c] = ldexpf(bd[e], eqb + ee[e]);
    };
    auto bd_step = [&](int u, const half8 &rh, const half8 &rl, f16v &bd) {
        const half8 qh = Q[(2 * (NU + u)) * 64 + lane], ql = Q[(2 * (NU + u) + 1) * 64 + lane];
        bd = mfma32(rh, qh, bd);
        bd = mfma32(rl, qh, bd);
        bd = mfma32(rh, ql, bd);
    };

    float m = -1e30f, l = 0.0f;
    f16v acc[NF];
#pragma unroll
    for (int i = 0; i < NF; i++) acc[i] = zero16();
    if (ta < tb) {
        // The operands of each product are loaded one product ahead, into the
        // registers that the product before has used up; the barriers keep the
        // compiler from moving the loads further (registers) or back (latency).
        // The block before the first tile's, as the tile before it would leave it
        {
            f16v bd = zero16();
#pragma unroll
            for (int u = 0; u < NU; u++) bd_step(u, rf[u][0], rf[u][1], bd);
            ring_put(bd, er, ta - 1);
        }
        for (int t = ta; t < tb; t++) {
            f16v s = zero16(), bd = zero16();
            load_r(t, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const half8 qh = Q[(2 * u) * 64 + lane], ql = Q[(2 * u + 1) * 64 + lane];
                s = mfma32(kf[u][0], qh, s);
                s = mfma32(kf[u][1], qh, s);
                s = mfma32(kf[u][0], ql, s);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_r(t, HU);
            er = re[(size_t)(t - bx + n) * 32 + c];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NU; u++) bd_step(u, rf[u][0], rf[u][1], bd);
            __builtin_amdgcn_sched_barrier(0);
            half8 vf[NF][2][2];
            float sc[NF];
#pragma unroll
            for (int i = 0; i < NF; i++) {
#pragma unroll
                for (int p = 0; p < 4; p++) vf[i][p >> 1][p & 1] = frag(vp, t, 4 * i + p);
                sc[i] = vs[(size_t)t * DK + 32 * i + c];
            }
            __builtin_amdgcn_sched_barrier(0);
            ring_put(bd, er, t);
            int ee[16];
            rows_e(ek, ee);   // (and orders the ring's writes before the reads)
            float sv[16];
            const float *rr = ring + 32 * (32 * (t & 1) + 4 * hh) + c;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                sv[e] = (ldexpf(s[e], eqa + ee[e]) + rr[32 * (8 * (e >> 2) + (e & 3))]) * kscale;
            }
            wave_lds_order();   // (the next tile's ring writes come after these reads)
            if (KT * t + KT > T) {
#pragma unroll
                for (int e = 0; e < 16; e++)
                    if (KT * t + 8 * (e >> 2) + 4 * hh + (e & 3) >= T) sv[e] = -INFINITY;
            }
            // online softmax. The maxima move only when some query of the wave
            // would exceed its maximum by more than 2^8 (base 2): the
            // probabilities stay <= 256, the context and the sum carry the same
            // maximum, and most tiles skip the rescale.
            float mx = sv[0];
#pragma unroll
            for (int e = 1; e < 16; e++) mx = fmaxf(mx, sv[e]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            if (__any(mx > m + 8.0f)) {
                const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= alpha;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float ae = __shfl(alpha, drow(e, hh));
#pragma unroll
                    for (int i = 0; i < NF; i++) acc[i][e] *= ae;
                }
            }
            // 2^6 times the probabilities (the sum carries the same factor)
            const float m6 = m - 6.0f;
            half8 ph[2], pl[2];
#pragma unroll
            for (int k2 = 0; k2 < 2; k2++) {
                float y[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    y[j] = __builtin_amdgcn_exp2f(sv[8 * k2 + j] - m6);
                    l += y[j];
                }
                split8u(y, ph[k2], pl[k2]);
            }
            // (past the last tile these are this one's again)
            const int tn = min(t + 1, tb - 1);
            ek = ke[(size_t)tn * 32 + c];
#pragma unroll
            for (int i = 0; i < NF; i++) {
                __builtin_amdgcn_sched_barrier(0);
                f16v tt = zero16();
#pragma unroll
                for (int k2 = 0; k2 < 2; k2++) {
                    tt = mfma32(ph[k2], vf[i][k2][0], tt);
                    tt = mfma32(ph[k2], vf[i][k2][1], tt);
                    tt = mfma32(pl[k2], vf[i][k2][0], tt);
                }
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][e] = fmaf(tt[e], sc[i], acc[i][e]);
                asm volatile("" : "+v"(acc[i]));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int p = 0; p < 4; p++) kf[2 * i + (p >> 1)][p & 1] = frag(kp, tn, 4 * i + p);
            }
        }
    }

    // the waves' contexts meet: each scaled to the common maximum, summed in wave order
    l += __shfl_xor(l, 32);
    if (hh == 0) ML[w * 32 + c] = m, ML[(NW + w) * 32 + c] = l;
    __syncthreads();   // (every wave is past its tiles: Q and the rings are free)
    float M = -1e30f, Ls = 0.0f;
#pragma unroll
    for (int i = 0; i < NW; i++) M = fmaxf(M, ML[i * 32 + c]);
#pragma unroll
    for (int i = 0; i < NW; i++) Ls = fmaf(ML[(NW + i) * 32 + c], __builtin_amdgcn_exp2f(ML[i * 32 + c] - M), Ls);
    const float fw = __builtin_amdgcn_exp2f(m - M);
    float *O = (float *)lds + w * 32 * L::OS;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float f = __shfl(fw, drow(e, hh));
#pragma unroll
        for (int i = 0; i < NF; i++) O[drow(e, hh) * L::OS + 32 * i + c] = acc[i][e] * f;
    }
    float *INV = X;
    if (w == 0 && hh == 0) INV[c] = 1.0f / (Ls * 0.015625f);
    __syncthreads();
    // thread = 8 features of one row, DK / 8 lanes per row
    constexpr int LPR = DK / 8, NV = 32 * LPR / (64 * NW);
    static_assert(NV * 64 * NW == 32 * LPR, "rows over threads");
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int idx = v * 64 * NW + tid;
        const int r = idx / LPR, sl = idx % LPR, t = t0 + r;
        float o[8];
        const float *op = (const float *)lds + r * L::OS + 8 * sl;
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = op[j];
#pragma unroll
        for (int i = 1; i < NW; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] += op[i * 32 * L::OS + j];
        const float inv = INV[r];
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] *= inv;
        if (DK == 128 && P.xp) {
            // the row's chunk (one head) as the output projection's prepared
            // input, split exactly as the products' preparation splits it
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) a = fmaxf(a, fabsf(o[j]));
#pragma unroll
            for (int x = 1; x < LPR; x <<= 1) a = fmaxf(a, __shfl_xor(a, x));
            const int sh = chunk_shift(a);
            half8 h, lo;
            split8(o, sh, h, lo);
            if (t < T) {
                const size_t mr = (size_t)bz * T + t;
                const int Kc = d / 128;
                uint8_t *xo = P.xp + ((((mr >> 5) * Kc + by) * 8 + (sl >> 1)) * 2 * 64 + (mr & 31) + 32 * (sl & 1)) * 16;
                *(half8 *)xo = h;
                *(half8 *)(xo + 1024) = lo;
                if (sl == 0) P.xpf[((mr >> 5) * Kc + by) * 32 + (mr & 31)] = ldexpf(1.0f, -sh);
            }
        } else if (t < T) {
            float *oc = ctx + ((size_t)bz * T + t) * d + ho + 8 * sl;
            *(f4 *)oc = f4{o[0], o[1], o[2], o[3]};
            *(f4 *)(oc + 4) = f4{o[4], o[5], o[6], o[7]};
        }
    }
    // the rows past M up to the 64-row padding: zeros (fold factor 1), as the
    // preparation pads; by the last block of the last segment
    if (DK == 128 && P.xp && bz == (int)gridDim.z - 1 && bx == (int)gridDim.x - 1) {
        const size_t Mr = (size_t)gridDim.z * T, Mp = (Mr + 63) / 64 * 64;
        const int Kc = d / 128;
        for (size_t i = tid; i < (Mp - Mr) * 32; i += 64 * NW) {
            const size_t mr = Mr + (i >> 5);
            const int sl = (int)(i & 31);
            *(uint4 *)(P.xp + ((((mr >> 5) * Kc + by) * 8 + (sl >> 2)) * 2 * 64 + 64 * ((sl >> 1) & 1) + (mr & 31) +
                               32 * (sl & 1)) * 16) = make_uint4(0, 0, 0, 0);
            if (sl == 0) P.xpf[((mr >> 5) * Kc + by) * 32 + (mr & 31)] = 1.0f;
        }
    }
}

// The splits, one workgroup per tile: [0, nk) K tiles, [nk, nk + nrb) rk blocks,
// the rest V tiles. Rows go through LDS so that both the reads (along features)
// and the writes (a tile's fragments) are contiguous.
struct SplitIn {
    const float *k, *rk, *v;
    unsigned nk, nrb;
    int T, d;
};

template <int DK>
__global__ __launch_bounds__(256) void k_attn_split(SplitIn S, Planes P) {
    constexpr int NU = DK / 16, TILE = NU * 2 * 64;   // fragments of 16 bytes
    __shared__ half8 st[TILE];
    const unsigned b = blockIdx.x;
    const int tid = threadIdx.x, T = S.T, d = S.d, H = d / DK;
    half8 *out;
    if (b < S.nk + S.nrb) {
        // rows: thread = row tid / 8, features DK/8 (tid % 8) .. of it
        constexpr int FPT = DK / 8;
        const bool isk = b < S.nk;
        const unsigned tile = isk ? b : b - S.nk, per = isk ? P.ntile : 2 * P.ntile;
        const int bh = (int)(tile / per), tt = (int)(tile % per), h = bh % H;
        const int r = tid >> 3, row = isk ? 32 * tt + r : T + 32 * (tt - P.ntile) + r;
        const bool live = row >= 0 && row < (isk ? T : 2 * T - 1);
        const float *x = (isk ? S.k + (size_t)(bh / H) * T * d : S.rk) + (size_t)(live ? row : 0) * d + h * DK + FPT * (tid & 7);
        float y[FPT], a = 0.0f;
#pragma unroll
        for (int j = 0; j < FPT; j += 4) {
            const f4 v = live ? *(const f4 *)(x + j) : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                y[j + e] = v[e];
                a = fmaxf(a, fabsf(v[e]));
            }
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) a = fmaxf(a, __shfl_xor(a, o));
        const int e = row_exp(a);
#pragma unroll
        for (int g = 0; g < FPT / 8; g++) {
            const int f8 = (FPT / 8) * (tid & 7) + g;   // group of 8 features: half-step f8 / 2, half f8 % 2
            float z[8];
#pragma unroll
            for (int j = 0; j < 8; j++) z[j] = y[8 * g + j];
            half8 hi, lo;
            split8(z, e, hi, lo);
            st[(2 * (f8 >> 1)) * 64 + r + 32 * (f8 & 1)] = hi;
            st[(2 * (f8 >> 1) + 1) * 64 + r + 32 * (f8 & 1)] = lo;
        }
        if ((tid & 7) == 0) (isk ? P.ke : P.re)[(size_t)tile * 32 + r] = -e;
        out = (isk ? P.k : P.r) + (size_t)tile * TILE;
    } else {
        // V: thread = a feature and the keys of one lane half hh (4hh .. 4hh+3 of
        // every 8): 16 keys, the two k-steps' 8 each; DK = 64: half the threads
        const unsigned tile = b - S.nk - S.nrb;
        const int bh = (int)(tile / P.ntile), tt = (int)(tile % P.ntile), h = bh % H;
        const int f = tid >> 1, hh = tid & 1;
        if (f < DK) {
            const float *x = S.v + ((size_t)(bh / H) * T + 32 * (size_t)tt) * d + h * DK + f;
            float y[2][8], a = 0.0f;
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int key = 16 * u + 8 * (j >> 2) + 4 * hh + (j & 3);
                    y[u][j] = 32 * tt + key < T ? x[(size_t)key * d] : 0.0f;
                    a = fmaxf(a, fabsf(y[u][j]));
                }
            a = fmaxf(a, __shfl_xor(a, 1));
            const int ex = min(max(row_exp(a), -100), 100);   // (the scale below stays a normal float)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                half8 hi, lo;
                split8(y[u], ex, hi, lo);
                st[((f >> 5) * 4 + 2 * u) * 64 + (f & 31) + 32 * hh] = hi;
                st[((f >> 5) * 4 + 2 * u + 1) * 64 + (f & 31) + 32 * hh] = lo;
            }
            if (hh == 0) P.vs[(size_t)tile * DK + f] = __int_as_float((127 - 6 - ex) << 23);
        }
        out = P.v + (size_t)tile * TILE;
    }
    __syncthreads();
#pragma unroll
    for (int i = tid; i < TILE; i += 256) out[i] = st[i];
}

size_t al256(size_t b) { return (b + 255) / 256 * 256; }

// the workspace: K planes and exponents, then rk's (offsets of query block bx and
// key tile t are block t - bx, and the one before it), then V's and scales
struct SplitWs {
    size_t kp, ke, rp, re, vs, total;
    int ntile;
    SplitWs(int T, int d, int H, int nseq) {
        ntile = (T + KT - 1) / KT;
        const size_t kt = (size_t)nseq * ntile, nr = 2 * (size_t)ntile;
        kp = al256(kt * KT * d * 4);
        ke = al256(kt * KT * H * sizeof(int));
        rp = al256(nr * KT * d * 4);
        re = al256(nr * KT * H * sizeof(int));
        vs = al256(kt * d * sizeof(float));
        total = 2 * kp + ke + rp + re + vs;
    }
};

template <int DK>
hipError_t launch_dk(const float *q, const float *k, const float *v, const float *rk, const float *bu,
                     const float *bv, float *ctx, int T, int d, int H, int nseq, void *ws, uint8_t *xp, float *xpf,
                     hipStream_t st) {
    if ((size_t)(2 * (size_t)T) * d >= 0x7fffffffu || !ws) return hipErrorInvalidValue;
    const SplitWs W(T, d, H, nseq);
    uint8_t *b = (uint8_t *)ws;
    Planes P{};
    P.k = (half8 *)b;
    P.v = (half8 *)(b + W.kp);
    P.ke = (int *)(b + 2 * W.kp);
    P.r = (half8 *)(b + 2 * W.kp + W.ke);
    P.re = (int *)(b + 2 * W.kp + W.ke + W.rp);
    P.vs = (float *)(b + 2 * W.kp + W.ke + W.rp + W.re);
    P.ntile = W.ntile;
    P.xp = xp, P.xpf = xpf;
    SplitIn S{};
    S.k = k, S.rk = rk, S.v = v;
    S.T = T, S.d = d;
    const size_t nk = (size_t)nseq * H * W.ntile, nrb = (size_t)H * 2 * W.ntile;
    if (2 * nk + nrb > 0x7fffffffu) return hipErrorInvalidValue;
    S.nk = (unsigned)nk, S.nrb = (unsigned)nrb;
    hipLaunchKernelGGL(k_attn_split<DK>, dim3((unsigned)(2 * nk + nrb)), dim3(256), 0, st, S, P);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    constexpr int bytes = AttnLds<DK>::BYTES;
    // set once per instantiation (thread-safe static initialisation)
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)k_attn<DK>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return attr;
    // exponentials are base 2: scores carry log2(e) / sqrt(DK)
    const float kscale = (1.0f / sqrtf((float)DK)) * 1.4426950408889634f;
    hipLaunchKernelGGL((k_attn<DK>), dim3(P.ntile, H, nseq), dim3(64 * NW), bytes, st, q, bu, bv, ctx, T, d, kscale,
                       P);
    return hipGetLastError();
}

}  // namespace

bool mh_attn_supported(int dk) { return dk == 64 || dk == 128; }

size_t mh_attn_ws_bytes(int T, int d, int H, int nseq, int left) {
    if (left >= 0 || T <= 0 || nseq <= 0 || H <= 0) return 0;   // (chunked windows split nothing)
    return SplitWs(T, d, H, nseq).total;
}

hipError_t mh_launch_relpos_attn(const float *q, const float *k, const float *v, const float *rk,
                                 const float *bias_u, const float *bias_v, float *ctx, int T, int d, int H,
                                 int left, int right, int nseq, void *ws, uint8_t *xp, float *xpf,
                                 hipStream_t st) {
    const int dk = d / H;
    if (left >= 0)
        return xp ? hipErrorInvalidValue
                  : mh_launch_relpos_attn_win(q, k, v, rk, bias_u, bias_v, ctx, T, d, H, left, right, nseq, st);
    if (dk == 128) return launch_dk<128>(q, k, v, rk, bias_u, bias_v, ctx, T, d, H, nseq, ws, xp, xpf, st);
    if (dk == 64 && !xp)
        return launch_dk<64>(q, k, v, rk, bias_u, bias_v, ctx, T, d, H, nseq, ws, nullptr, nullptr, st);
    return hipErrorInvalidValue;
}

bool mh_attn_preps_out(int d, int H, int left) { return left < 0 && H > 0 && d / H == 128; }
