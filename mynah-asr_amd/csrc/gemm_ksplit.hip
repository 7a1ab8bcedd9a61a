// gemm_ksplit.hip — the products of few rows (EXACT and INT8ACT numerics, on
// prepared input), K split over the waves of one workgroup.
//
// k_gemm gives a workgroup whole outputs, chunk after chunk: with few row
// bands that is a handful of workgroups, each one long dependent chain. Here
// the eight waves of a workgroup take the chunks of one output tile side by
// side, S at a time, and their results meet in LDS, where they are folded in
// chunk order from zero with the prepared input's fold factors: the
// operations, and so the bits, of k_gemm's fold in registers.
//
// Operands go straight from L2 to registers (each wave has chunks of its own,
// so LDS would bring no reuse). What bounds it: for one workgroup per CU,
// latency (a launch, one memory round trip and one exchange: 4.6 us at K =
// 1024 whatever the rows); for several, the 64 B/clk L1 path (a 32 x 32 tile
// reads 20 KB per chunk: about 1.9 us per workgroup and round of 8 chunks,
// where MFMA and VALU would take 0.9).
// Tried at the same sizes and slower or no faster: 32 x 64 and 64 x 64 tiles
// (half the L1 bytes, but one workgroup per CU: 1024 -> 1024 at 250 rows 4.9 ->
// 6.0 and 7.9 us, 4096 -> 1024 at 750 rows 24.6 -> 31.6 and 28.3), 16 waves
// (4096 -> 1024 at 64 rows 10.4 -> 10.1, at 750 rows 24.6 -> 30.0).
#include "product.h"

namespace {

// PC waves side by side over columns, S = 8 / PC over chunks; each wave 32 rows by
// WN groups of 32 columns.
template <int QT, int WN, int PC> struct KsTile {
    static constexpr int NW = 8, S = NW / PC, NT = 64 * NW;
    static constexpr int TR = 32, TC = 32 * WN * PC;
    static constexpr int TCS = TC + 8;    // LDS row stride: the two lane halves' rows (4 apart) fall in different banks
    // ksteps of operands in flight per wave: two for the 32 x 32 tile, so that
    // two workgroups share a CU (128 registers)
    static constexpr int PF = WN == 1 || QT == QT_F32 ? 2 : 4;
    static constexpr size_t LDS = (size_t)S * TR * TCS * 4 + (size_t)S * TR * 4;
};

template <int QT, int EPI, bool A1, int WN, int PC>
__global__ __launch_bounds__(512, (WN == 1 ? 4 : 2)) void k_gemm_ks(GemmJobs J, const uint8_t *__restrict__ xp,
                                                    const uint8_t *__restrict__ xm, const float *__restrict__ xpf, int M,
                                                    int act, int tilesM, int tilesN, int pr, PrepOut po) {
    using F = Fmt<QT>;
    using L = KsTile<QT, WN, PC>;
    constexpr int S = L::S, TR = L::TR, TC = L::TC, TCS = L::TCS, NT = L::NT, PF = L::PF;
    constexpr int TERMS = A1 ? 1 : 2;
    constexpr bool HALVES = A1 && QT == QT_Q5_K;   // (as in k_gemm)
    static_assert(EPI != EPI_PREP || (TC == 128 && !A1), "the prepared output is one chunk of 32 rows");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float *part = lds, *pfs = lds + S * TR * TCS;
    // The tiles of a launch as 8 rectangles of (row band, column tile), one per
    // XCD (workgroups are dealt to the XCDs round-robin): pr row parts by 8 / pr
    // column parts, so that the operand with more bytes is read by fewer L2s
    const int nt = J.n * tilesN, bid = blockIdx.x, xcd = bid & 7, loc = bid >> 3, pcn = 8 / pr;
    const int xr = xcd % pr, xc = xcd / pr;
    const int r0 = tilesM * xr / pr, r1 = tilesM * (xr + 1) / pr, q0 = nt * xc / pcn, q1 = nt * (xc + 1) / pcn;
    const int rh = r1 - r0;
    if (loc >= rh * (q1 - q0)) return;   // (whole workgroup: no barrier is left waiting)
    const int tm = r0 + loc % rh, tr = q0 + loc / rh;
    const int job = tr / tilesN, tn = tr - job * tilesN;
    const DevW W = job == 0 ? J.W[0] : (job == 1 ? J.W[1] : J.W[2]);
    float *__restrict__ y = job == 0 ? J.y[0] : (job == 1 ? J.y[1] : J.y[2]);
    const float *__restrict__ bias = job == 0 ? J.bias[0] : (job == 1 ? J.bias[1] : J.bias[2]);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hh = lane >> 5, col = lane & 31;
    const int pcI = wave % PC, s = wave / PC;
    const int Kc = W.Kp / 128;
    int gn[WN];
#pragma unroll
    for (int j = 0; j < WN; j++) gn[j] = (tn * PC + pcI) * WN + j;

    AK<1> a[PF];
    BK<QT, WN> b[PF];
    BH<QT, WN> hd;
    half8 xmv = {};
    float pf = 0.0f;
    auto load_k = [&](int c, int sl, AK<1> &aa, BK<QT, WN> &bb) {
        load_bk<QT, WN>(W, Kc, gn, c, sl, lane, bb);
#pragma unroll
        for (int kh = 0; kh < 2; kh++) {
            const uint8_t *p = xp + ((((size_t)tm * Kc + c) * HSTEPS + 2 * sl + kh) * TERMS * 64 + lane) * 16;
            aa.h[0][kh] = *(const half8 *)p;
            if constexpr (!A1) aa.l[0][kh] = *(const half8 *)(p + 1024);
        }
    };
    auto load_h = [&](int c) {
        load_bh<QT, WN>(W, Kc, gn, c, lane, hd);
        if constexpr (F::MINS) xmv = *(const half8 *)(xm + (((size_t)tm * Kc + c) * 64 + lane) * 16);
        if (pcI == 0 && lane < TR) pf = xpf[((size_t)tm * Kc + c) * 32 + col];
    };
    if (s < Kc) {
        load_h(s);
#pragma unroll
        for (int k = 0; k < PF; k++) load_k(s, k, a[k], b[k]);
    }

    // the fold: thread = VN vectors of V outputs in row-major order
    constexpr int OPT = TR * TC / NT, V = OPT < 4 ? OPT : 4, VN = OPT / V;
    static_assert(V * VN * NT == TR * TC, "outputs per thread");
    float total[VN][V];
#pragma unroll
    for (int v = 0; v < VN; v++)
#pragma unroll
        for (int j = 0; j < V; j++) total[v][j] = 0.0f;

    for (int cb = 0; cb < Kc; cb += S) {
        const int c = cb + s;
        f16v acc[1][WN];
        const float pfc = pf;
        if (c < Kc) {
            int half0[HALVES ? WN : 1][HALVES ? 16 : 1];
#pragma unroll
            for (int j = 0; j < WN; j++) acc[0][j] = zero16();
#pragma unroll
            for (int sl = 0; sl < KSTEPS; sl++) {
                kstep<QT, 1, WN, A1>(a[sl % PF], b[sl % PF], hd, sl, acc);
                if (sl + PF < KSTEPS) load_k(c, sl + PF, a[sl % PF], b[sl % PF]);
                // pin the order: the loads of later ksteps stay behind this one's
                // MFMAs, and its block factors' fmas ahead of the next one's (left
                // free, every kstep's products stay live and the tile spills)
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!fold_fmt<QT>() && QT != QT_F32)
#pragma unroll
                    for (int j = 0; j < WN; j++) asm volatile("" : "+v"(acc[0][j]));
                if constexpr (HALVES) {
                    if (sl == KSTEPS / 2 - 1)
#pragma unroll
                        for (int j = 0; j < WN; j++)
#pragma unroll
                            for (int e = 0; e < 16; e++) {
                                half0[j][e] = (int)acc[0][j][e];
                                acc[0][j][e] = 0.0f;
                            }
                }
            }
            if constexpr (HALVES) {
#pragma unroll
                for (int j = 0; j < WN; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[0][j][e] = (float)(half0[j][e] + (int)acc[0][j][e]);
            }
            if constexpr (fold_fmt<QT>()) {
#pragma unroll
                for (int j = 0; j < WN; j++) fold_finish<QT>(xmv, hd.h[j], acc[0][j]);
            }
            // the next chunk's first operands are in flight during the exchange
            if (c + S < Kc) {
                load_h(c + S);
#pragma unroll
                for (int k = 0; k < PF; k++) load_k(c + S, k, a[k], b[k]);
            }
        }
        if (cb > 0) __syncthreads();   // the round before is folded
        if (c < Kc) {
#pragma unroll
            for (int j = 0; j < WN; j++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    part[(s * TR + drow(e, hh)) * TCS + 32 * (WN * pcI + j) + col] = acc[0][j][e];
            if (pcI == 0 && lane < TR) pfs[s * TR + lane] = pfc;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < S; u++) {
            if (cb + u < Kc)
#pragma unroll
            for (int v = 0; v < VN; v++) {
                const int idx = v * NT + tid, row = idx / (TC / V), cv = V * (idx % (TC / V));
                const float f = pfs[u * TR + row];
                const float *p = part + (u * TR + row) * TCS + cv;
#pragma unroll
                for (int j = 0; j < V; j++) total[v][j] = __builtin_fmaf(f, p[j], total[v][j]);
            }
        }
    }

    if constexpr (EPI == EPI_PREP) {
        // SiLU, then the rows as one chunk of the second product's prepared
        // input, formed with k_prep's operations: 32 lanes hold a row (4 columns
        // each), lane l32 the elements of half-step l32 / 4, half (l32 / 2) % 2.
        // The 16 KiB block of this (row group, chunk) is contiguous in xp.
        __syncthreads();
        uint8_t *blk = (uint8_t *)lds, *xmb = blk + 16 * 1024;
        const int l32 = lane & 31, hu = l32 >> 2, h2 = (l32 >> 1) & 1;
#pragma unroll
        for (int v = 0; v < VN; v++) {
            const int row = (v * NT + tid) / 32;
            float xs[4], amax = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float t = total[v][j];
                const int n = TC * tn + 4 * l32 + j;
                if constexpr (QT == QT_F32) t = ldexpf(t, -wshift<QT>(W, n));
                if (bias && n < W.n) t = t + bias[n];
                xs[j] = silu_f(t);
                amax = fmaxf(amax, fabsf(xs[j]));
            }
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
            const int sh = chunk_shift(amax);
            _Float16 hv[4], lv[4];
            float s4 = 0.0f;   // (lanes 2q, 2q + 1 hold 8 elements: their sum in order)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                xs[j] = ldexpf(xs[j], sh);
                hv[j] = (_Float16)xs[j];
                lv[j] = (_Float16)(xs[j] - (float)hv[j]);
                s4 += xs[j];
            }
            uint8_t *o = blk + ((hu * 2) * 64 + row + 32 * h2) * 16 + 8 * (l32 & 1);
            __builtin_memcpy(o, hv, 8);
            __builtin_memcpy(o + 1024, lv, 8);
            if (l32 == 0) po.xpf[((size_t)tm * po.Kc + tn) * 32 + row] = ldexpf(1.0f, -sh);
            if (po.xsum) {
                const float even = __shfl_xor(s4, 1, 64);
                float s8 = even;
#pragma unroll
                for (int j = 0; j < 4; j++) s8 += xs[j];         // odd lanes: the 8 elements' sum
                const float s16 = s8 + __shfl_xor(s8, 2, 64);     // lanes 4u + 1, 4u + 3: half-step u
                const float s32 = __shfl_xor(s16, 4, 64) + s16;
                _Float16 *slot = (_Float16 *)(xmb + row * 16);    // hi parts; the lo parts 32 rows on
                if (po.xsum == 1) {
                    if ((l32 & 3) == 3) slot[hu] = xm_part(s16, 0), slot[hu + 32 * 8] = xm_part(s16, 1);
                } else if ((l32 & 7) == 7) {
                    slot[l32 >> 3] = xm_part(s32, 0), slot[(l32 >> 3) + 32 * 8] = xm_part(s32, 1);
                    slot[4 + (l32 >> 3)] = (_Float16)0.0f, slot[4 + (l32 >> 3) + 32 * 8] = (_Float16)0.0f;
                }
            }
        }
        __syncthreads();
        uint8_t *gx = po.xp + ((size_t)tm * po.Kc + tn) * 16 * 1024;
#pragma unroll
        for (int i = 0; i < 1024 / NT; i++) *(uint4 *)(gx + (i * NT + tid) * 16) = *(const uint4 *)(blk + (i * NT + tid) * 16);
        if (po.xsum && tid < 64)
            *(uint4 *)(po.xm + (((size_t)tm * po.Kc + tn) * 64 + tid) * 16) = *(const uint4 *)(xmb + tid * 16);
        return;
    }
    const bool vec = W.n % V == 0 && ((uintptr_t)y & (4 * V - 1)) == 0;
#pragma unroll
    for (int v = 0; v < VN; v++) {
        const int idx = v * NT + tid, m = TR * tm + idx / (TC / V), n = TC * tn + V * (idx % (TC / V));
        if (m >= M || n >= W.n) continue;
        float *yp = y + (size_t)m * W.n + n;
        float o[V];
#pragma unroll
        for (int j = 0; j < V; j++) {
            o[j] = total[v][j];
            const int nj = min(n + j, W.n - 1);
            if constexpr (QT == QT_F32) o[j] = ldexpf(o[j], -wshift<QT>(W, nj));
            if (bias) o[j] = o[j] + bias[nj];
        }
        if (vec) {
            typedef float fv __attribute__((ext_vector_type(V)));
            fv r = {};
            if (act_res(act)) r = *(const fv *)yp;
            fv w;
#pragma unroll
            for (int j = 0; j < V; j++) w[j] = epi_out(act, o[j], r[j]);
            *(fv *)yp = w;
        } else {
#pragma unroll
            for (int j = 0; j < V; j++)
                if (n + j < W.n) yp[j] = epi_out(act, o[j], act_res(act) ? yp[j] : 0.0f);
        }
    }
}

template <int QT, int EPI, bool A1, int WN, int PC>
hipError_t launch_ks(const GemmJobs &J, const uint8_t *xp, const float *xs16, const float *xpf, int M, int act,
                     const PrepOut &po, hipStream_t st) {
    using L = KsTile<QT, WN, PC>;
    const DevW &W = J.W[0];
    const float wbytes = w_bpe<QT>() * W.Np * W.Kp * J.n, abytes = (A1 ? 2.0f : 4.0f) * mh_mpad(M) * W.Kp;
    const int tilesM = (EPI == EPI_PREP ? mh_mpad(M) : M + L::TR - 1) / L::TR, tilesN = W.Np / L::TC, nt = J.n * tilesN;
    static const hipError_t attr = hipFuncSetAttribute((const void *)k_gemm_ks<QT, EPI, A1, WN, PC>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::LDS);
    if (attr != hipSuccess) return attr;
    // row parts of the XCD grid: the fewest bytes over the eight L2s, times the
    // fullest XCD's share of the tiles
    int pr = 1;
    size_t wgs = 0;
    float best = 0.0f;
    for (int p = 1; p <= 8; p *= 2) {
        const size_t rect = (size_t)((tilesM + p - 1) / p) * ((nt + 8 / p - 1) / (8 / p));
        const float cost = (wbytes * p + abytes * (8 / p)) * (8.0f * rect / ((float)tilesM * nt));
        if (p == 1 || cost < best) best = cost, pr = p, wgs = 8 * rect;
    }
    hipLaunchKernelGGL((k_gemm_ks<QT, EPI, A1, WN, PC>), dim3((unsigned)wgs), dim3(L::NT), L::LDS, st, J, xp,
                       (const uint8_t *)xs16, xpf, M, act, tilesM, tilesN, pr, po);
    return hipGetLastError();
}

template <int QT, bool A1>
hipError_t ks_t(const GemmJobs &J, const uint8_t *xp, const float *xs16, const float *xpf, int M, int act,
                const PrepOut *po, hipStream_t st) {
    if (po) {
        if constexpr (!A1) return launch_ks<QT, EPI_PREP, false, 2, 2>(J, xp, xs16, xpf, M, 1, *po, st);
        return hipErrorInvalidValue;
    }
    return launch_ks<QT, EPI_Y, A1, 1, 1>(J, xp, xs16, xpf, M, act, PrepOut{}, st);
}

template <int QT>
hipError_t ks_dispatch(const GemmJobs &J, const uint8_t *xp, const float *xs16, const float *xpf, int M, int act,
                       const PrepOut *po, bool a1, hipStream_t st) {
    if constexpr (QT == QT_F32 || QT == QT_INT8 || QT == QT_INT4) {
        if (a1) return hipErrorInvalidValue;
        return ks_t<QT, false>(J, xp, xs16, xpf, M, act, po, st);
    } else {
        if (a1) return ks_t<QT, true>(J, xp, xs16, xpf, M, act, po, st);
        return ks_t<QT, false>(J, xp, xs16, xpf, M, act, po, st);
    }
}

}  // namespace

// By the number of 32 x 32 output tiles, the chunks of K and the format. A CU
// runs tiles two at a time, so the time steps every 256 tiles; K of fewer than
// eight chunks leaves waves idle, and of ten leaves most of them idle every second
// round. Where an element costs the most instructions k_gemm's chains are longest:
// the super-block formats leave later than the others (with one term per element,
// INT8ACT, so do the rest from eight chunks on; so do f32 weights of 8 to 15 chunks
// when they are more than two XCDs' L2 or of a chunk count that is no power of
// two, where k_gemm waits for their planes). This form / k_gemm, us, Q8_0 and Q6_K:
//    256 -> 1024   251 rows (256 tiles)  3.7 / 4.5   4.0 / 5.2     763 (768)  6.2 / 4.9   6.7 / 5.5
//    512 -> 2048   251 rows (512 tiles)  5.2 / 6.6   5.6 / 7.7     379 (768)  7.0 / 6.9   7.5 / 8.0
//                  507 rows (1024)       8.2 / 7.2   8.9 / 8.1
//   1024 -> 1024   763 rows (768 tiles)  9.6 / 10.4  10.4 / 12.7  1019 (1024) 11.0 / 10.6 12.3 / 12.8
//   1280 -> 1280   507 rows (640 tiles)  0.90 / 1    0.85 / 1      660 (840)  1.03 / 1    0.99 / 1
//   2048 -> 512   2555 rows (1280)      21.4 / 23.0  24.2 / 29.9  2811 (1408) 24.1 / 23.6 27.2 / 30.2
//   4096 -> 1024  1275 rows (1280)      39.8 / 43.2  44.4 / 56.3  1403 (1408) 49.5 / 44.0 51.4 / 56.3
// The other formats of each kind lie within 8% of these ratios. f32 weights: 1024 ->
// 4096 at 251 rows (1024 tiles) 13.8 / 18.6, 1280 -> 1280 at 660 (840) 16.3 / 22.0,
// but 1024 -> 2048 at 507 (1024) 13.2 / 12.6, 1024 -> 1024 at 1019 (1024) 13.8 / 12.9.
// The prepared output (32 x 128 tiles, SiLU and split as the epilogue) wins while a
// CU has one such workgroup: the whole FFN 1024 -> 4096 at 125 rows (128) 25.3 /
// 30.1, at 253 rows (256) 28.2 / 32.9, at 317 rows (320) 41.1 / 38.1; 0.77 to 0.93
// of it in every format up to 256.
bool mh_use_gemm_ks(int qtype, const DevW &W, int M, int jobs, bool prep, bool a1) {
    const long rows = (M + 31) / 32, Kc = W.Kp / 128;
    if (prep) return mh_mpad(M) / 32 * (W.Np / 128) <= 256;
    const bool super_blocks = qtype == QT_Q2_K || qtype == QT_Q3_K || qtype == QT_Q4_K || qtype == QT_Q5_K || qtype == QT_Q6_K;
    const bool late = super_blocks || (a1 && Kc >= 8);
    const bool f32_late = qtype == QT_F32 && (Kc > 8 || 4L * W.Np * W.Kp * jobs > 9000000);
    const long most = Kc < 4   ? 256
                      : Kc < 8 ? (late ? 768 : 512)
                      : Kc < 16 ? (late || f32_late ? 1024 : Kc == 10 ? 640 : 768)
                                : (late ? 1408 : 1280);
    return rows * (W.Np / 32) * jobs <= most;
}

hipError_t mh_launch_gemm_ks(int qtype, const GemmJobs &J, const uint8_t *xp, const float *xs16, const float *xpf, int M,
                             int act, const PrepOut *po, bool a1, hipStream_t st) {
    MH_DISPATCH(ks_dispatch, qtype, J, xp, xs16, xpf, M, act, po, a1, st)
}
