// Backward of the union attention in fp32 on the matrix cores
// (v_mfma_f32_16x16x4_f32), for up to 16 query heads per KV head, sinks within
// block 0 and k <= 64.  The gradients are those of hba_attn_bwd.hip's header.
//
//   bwd_dq_f32:  the forward's row tiles (16 / G queries x G heads as the 16
//                columns): S^T = K . Q^T, dP^T = V . dO^T and
//                dQ^T += K^T . dS^T per unit of keys, in one pass online in
//                the softmax (dS needs only p and D = <dO, O>).  It also
//                leaves the prepared query rows, the LSE and D for:
//   bwd_dkv_f32: a wave takes 16 keys of a 64-key block and the (query, head)
//                pairs of a range of query rows that attend them, 16 per
//                tile: S = X . K^T, dP = dO . V^T, dV += P^T . dO,
//                dK += dS^T . X.
//   bwd_k_f32:   the ranges' sums added to dk and dv, and the QKNorm backward
//                of the key rows.
// dk and dv are the same bits from run to run, and with any workspace: a
// launch of bwd_dkv_f32 takes as many ranges as there are places for their sums
// beyond the workspace that hba_attn_bwd asks for, bwd_k_f32 adds these in order,
// and with fewer than two places each range is a launch that adds to dk and dv
// itself.  Atomic sums, in another order each time, took 993 us per training
// step at 2048 tokens, 14 / 2 heads, head dim 64, where these take 999; over 67
// shapes of 64 to 32768 tokens these take 0.86 to 1.05 of the atomics' time.
//
// Matrix cores bound all three products at 64 FLOP per SIMD and cycle; every
// operand comes from L1 / L2 in the layout it is used in (16 bytes per lane,
// or 64-byte runs for the transposed one), without LDS or barriers in the
// loops.  A training step of 14 / 2 heads at 2048 tokens and head dim 64 took
// 15.8 ms with one lane per key element on the VALU (dq 7.3, dk and dv 6.9,
// sinks 0.9).
//
// As in the forward, a masked product leaves 0 * y in its sums, which is a
// NaN where y is not finite: a wave whose sums are not finite takes its tile
// again with the masked products skipped one by one (`safe`).
#include <algorithm>

#include "hba_abi.h"
#include "hba_attn_f32.h"
#include "hba_attn_f32_tile.h"
#include "hba_common.h"
#include "hba_xcd.h"

namespace hba {
namespace af {

__device__ __forceinline__ float col_sum(float v) {   // over the 4 lanes of a column
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// 16-key units: with 32 keys a unit's operands, rows and accumulators pass the
// registers of two waves per SIMD at d = 64.
template <int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_dq_f32_kernel(
    const float *__restrict__ q, const float *__restrict__ kc, const float *__restrict__ kr,
    const float *__restrict__ v, const float *__restrict__ qgain, float eps, const float *__restrict__ cosT,
    const float *__restrict__ sinT, const int32_t *__restrict__ idx, const int32_t *__restrict__ cnt,
    const float *__restrict__ out, const float *__restrict__ dout, int n, int Hq, int Hkv, int S, int W, int kk,
    float scale, int ntiles, int Cn, int xmap, float *__restrict__ qc_ws, float *__restrict__ qr_ws,
    float *__restrict__ lse_ws, float *__restrict__ dd_ws, float *__restrict__ dq, float *__restrict__ dq_gain) {
    constexpr int KT = 16, NC = D / 16, NM = KT / 16;
    __shared__ float gsum[4][16];
    int combo, wt;
    xcd_map(blockIdx.x, Cn, ntiles, xmap, combo, wt);
    if (wt >= ntiles || combo >= Cn) return;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = Hq / Hkv, qpt = 16 / G;
    const int g = combo % Hkv;
    const int64_t b = combo / Hkv, bh = combo;
    const int64_t i0l = ((int64_t)wt * 4 + w) * qpt;
    const bool live = i0l < n;   // wave-uniform; an idle wave still meets the barrier
    const int i0 = live ? (int)i0l : 0;
    const int qs = l16 / G;
    const int i = i0 + qs;
    const bool ok = live && qs < qpt && i < n;
    const int ic = ok ? i : 0, h = g * G + (ok ? l16 % G : 0);
    float gain_term = 0.0f;
    if (live) {
        const int64_t row = ((b * n + ic) * Hq + h) * D + 4 * lg;
        const float *KC = kc + bh * n * D, *KR = kr + bh * n * D, *V = v + (b * n * Hkv + g) * D;
        const int64_t vs = (int64_t)Hkv * D;
        const float *cs = cosT + (int64_t)ic * D, *sn = sinT + (int64_t)ic * D;
        Units<KT> u;
        u.init(idx, cnt, bh * n + i0, n, S, W, kk, qpt, i0);
        f32x4 x[NC], dO[NC], O[NC], On[NC], kf[NM][NC], vf[NM][NC];
        float ms, r, dd = 0.0f;
        q_load<D>(q + row - 4 * lg, ok, qgain ? qgain + h : nullptr, eps, lg, x, ms, r);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            dO[c] = ok ? ld4(dout + row + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
            const f32x4 o = ok ? ld4(out + row + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) dd = fmaf(dO[c][e], o[e], dd);
        }
        dd = col_sum(dd);
        if (ok) {
#pragma unroll
            for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4 *>(qc_ws + row + 16 * c) = x[c];
        }
        q_rope<D>(x, cs, sn, lg);
        if (ok) {
#pragma unroll
            for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4 *>(qr_ws + row + 16 * c) = x[c];
        }
        auto load_kv = [&]() {
            const float *kp = (u.ph == 2 ? KR : KC) + (int64_t)(u.kb + l16) * D + 4 * lg;
            const float *vp = V + (int64_t)(u.kb + l16) * vs + 4 * lg;
#pragma unroll
            for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    kf[mt][c] = ld4(kp + 16 * mt * D + 16 * c);
                    vf[mt][c] = ld4(vp + 16 * mt * vs + 16 * c);
                }
        };
        float m, l, mn_;   // mn_: the maximum that On (the NoPE part) is relative to
        for (int safe = 0;; safe = 1) {
            q_load<D>(q + row - 4 * lg, ok, qgain ? qgain + h : nullptr, eps, lg, x, ms, r);
#pragma unroll
            for (int c = 0; c < NC; ++c) O[c] = On[c] = f32x4{0.f, 0.f, 0.f, 0.f};
            m = mn_ = -INFINITY;
            l = 0.0f;
            bool roped = false;
            auto to_window = [&]() {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    On[c] = O[c];
                    O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                mn_ = m;
                roped = true;
            };
            u.restart();
            bool more = u.next(lane, qs);
            if (more) load_kv();
            while (more) {
                // the same keys transposed: element 16 c + l16 of keys 4 lg + e
                float kt[NM][4][NC];
                const float *tp = (u.ph == 2 ? KR : KC) + (int64_t)(u.kb + 4 * lg) * D + l16;
#pragma unroll
                for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int c = 0; c < NC; ++c) kt[mt][e][c] = tp[(16 * mt + e) * D + 16 * c];
                if (u.ph == 2 && !roped) {
                    q_rope<D>(x, cs, sn, lg);
                    to_window();
                }
                int lo, hi;
                u.range(i, ok, lo, hi);
                const float mul = (float)(u.ph == 1 ? u.mult : 1);
                const bool full = __all(!ok || (lo <= 0 && hi >= KT - 1 && mul == 1.0f)) && !safe;
                f32x4 Sa[NM], dP[NM];
                bool act[NM];   // wave-uniform: the group holds a key of some column
#pragma unroll
                for (int mt = 0; mt < NM; ++mt) {
                    act[mt] = full || __any(lo <= 16 * mt + 15 && hi >= 16 * mt && lo <= hi);
                    Sa[mt] = dP[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (act[mt]) {
#pragma unroll
                        for (int c = 0; c < NC; ++c)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                Sa[mt] = mma4(kf[mt][c][e], x[c][e], Sa[mt]);
                                dP[mt] = mma4(vf[mt][c][e], dO[c][e], dP[mt]);
                            }
                    }
                }
                more = u.next(lane, qs);
                if (more) load_kv();
                // online softmax of the column; p = dS = 0 outside its keys
                float tmax = -INFINITY;
#pragma unroll
                for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int j = 16 * mt + 4 * lg + e;
                        Sa[mt][e] = (full || (j >= lo && j <= hi)) ? Sa[mt][e] * scale : -INFINITY;
                        tmax = fmaxf(tmax, Sa[mt][e]);
                    }
                tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
                tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
                const float mx = fmaxf(m, tmax);
                const float sh = (mx == -INFINITY) ? 0.0f : mx;
                const float alpha = expf(m - sh);
                m = mx;
                l *= alpha;
#pragma unroll
                for (int c = 0; c < NC; ++c) O[c] *= alpha;
#pragma unroll
                for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int j = 16 * mt + 4 * lg + e;
                        const float p = expf(Sa[mt][e] - sh) * mul;
                        l += p;
                        Sa[mt][e] = (full || (j >= lo && j <= hi)) ? p * (dP[mt][e] - dd) : 0.0f;
                    }
                if (!safe) {
#pragma unroll
                    for (int mt = 0; mt < NM; ++mt)
                        if (act[mt]) {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
#pragma unroll
                                for (int c = 0; c < NC; ++c) O[c] = mma4(kt[mt][e][c], Sa[mt][e], O[c]);
                        }
                } else {
                    // the same sums without the masked products: key j of this
                    // column, elements 16 c + 4 lg + e
#pragma unroll
                    for (int mt = 0; mt < NM; ++mt)
#pragma nounroll
                        for (int tg = 0; tg < 4; ++tg)
#pragma unroll
                            for (int te = 0; te < 4; ++te) {
                                const int j = 16 * mt + 4 * tg + te;
                                const float ds = __shfl(Sa[mt][te], 16 * tg + l16, 64);
#pragma unroll
                                for (int c = 0; c < NC; ++c)
#pragma unroll
                                    for (int e = 0; e < 4; ++e) {
                                        const float y = __shfl(kt[mt][te][c], 16 * tg + 4 * lg + e, 64);
                                        if (j >= lo && j <= hi) O[c][e] = fmaf(ds, y, O[c][e]);
                                    }
                            }
                }
            }
            if (!roped) to_window();
            l = col_sum(l);
            bool fin = l < INFINITY;
#pragma unroll
            for (int c = 0; c < NC; ++c) fin = fin && finite4(O[c]) && finite4(On[c]);
            if (safe || __all(!ok || fin)) break;
        }
        if (ok && lg == 0) {
            const int64_t o = (b * Hq + h) * n + i;
            lse_ws[o] = m + logf(l);
            dd_ws[o] = dd;
        }
        // rope^T of the window part, then the QKNorm backward
        const float fr = scale / l, fn = (mn_ == -INFINITY) ? 0.0f : expf(mn_ - m) * fr;
        f32x4 y[NC], zs[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) zs[c] = (O[c] * fr) * ld4(sn + 16 * c + 4 * lg);
        float yx = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const f32x4 z = (c < NC / 2) ? zs[c + NC / 2] : -zs[c - NC / 2];
            y[c] = On[c] * fn + (O[c] * fr) * ld4(cs + 16 * c + 4 * lg) + z;
            if (qgain) {
                x[c] = ld4(q + row + 16 * c);
#pragma unroll
                for (int e = 0; e < 4; ++e) yx = fmaf(y[c][e], x[c][e], yx);
            }
        }
        if (qgain) {
            const float gn = qgain[h];
            yx = col_sum(yx);
            const float corr = (ms >= eps) ? gn * yx / ((float)D * r * r * r) : 0.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c) y[c] = (gn / r) * y[c] - x[c] * corr;
            if (ok) gain_term = yx / r;
        }
        if (ok) {
#pragma unroll
            for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4_a4 *>(dq + row + 16 * c) = y[c];
        }
    }
    // the gain gradient: one atomic per head and workgroup (the adds of all
    // workgroups meet on Hq floats)
    if (qgain && dq_gain) {
        if (lg == 0) gsum[w][l16] = gain_term;
        __syncthreads();
        if ((int)threadIdx.x < G) {
            float t = 0.0f;
            for (int w4 = 0; w4 < 4; ++w4)
                for (int qq = 0; qq < qpt; ++qq) t += gsum[w4][qq * G + threadIdx.x];
            unsafeAtomicAdd(&dq_gain[g * G + threadIdx.x], t);
        }
    }
}

// Workgroup (b, g, range of R query rows, 64-key block); the block index nb
// stands for the sink keys of block 0, which every row from j on attends.  A
// launch takes the nr ranges from split0 on.  Slot ((b, g), block, range) of
// `part` is [4 waves][dk, dv][D / 16][64 lanes] f32x4 (lane (l16, lg), e: key 4
// lg + e of the wave's 16, element 16 c + l16); `used` says per slot and wave
// whether it was written.  DIRECT (nr = 1) adds the sums to dk and dv, the
// sinks' to `part`, a slot per (b, g).
// About 32 ranges per sequence balance the blocks' rows (a block that many
// queries picked, a range that a window only touches): at 2048 tokens, 14 / 2
// heads, ranges of 256 rows took 424 us, 128 303, 64 263; at 4096 256 853, 128
// 790.  Past 64K tokens ranges stay at 2048 rows, so that the list fits LDS.
constexpr int F32_RMIN = 64, F32_RMAX = 2048;

template <int D, bool DIRECT>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_dkv_f32_kernel(
    const float *__restrict__ kc, const float *__restrict__ kr, const float *__restrict__ v,
    const float *__restrict__ cosT, const float *__restrict__ sinT, const int32_t *__restrict__ idx,
    const int32_t *__restrict__ cnt, const float *__restrict__ dout, int n, int Hq, int Hkv, int S, int W, int kk,
    float scale, int R, int split0, int nr, int nblk, const float *__restrict__ qc_ws,
    const float *__restrict__ qr_ws, const float *__restrict__ lse_ws, const float *__restrict__ dd_ws,
    float *__restrict__ part, int *__restrict__ used, float *__restrict__ dk, float *__restrict__ dv) {
    constexpr int NC = D / 16;
    __shared__ int rows[F32_RMAX];
    __shared__ int wcount[4];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = n / 64, G = Hq / Hkv;
    const int bx = (int)(blockIdx.x % nblk), sp = (int)((blockIdx.x / nblk) % nr);
    const int64_t bg = blockIdx.x / ((int64_t)nblk * nr), b = bg / Hkv;
    const int64_t slot = (DIRECT ? bg : (bg * nblk + bx) * nr + sp) * 4 + w;
    const int g = (int)(bg % Hkv);
    const bool sinks = bx == nb;
    const int blk = sinks ? 0 : bx;
    const int r0 = (split0 + sp) * R, r1 = min(n, r0 + R);

    // the range's rows that picked the block, ascending
    int nrt = 0;
    if (!sinks && blk >= 1) {
        for (int rb = r0; rb < r1; rb += 256) {
            const int i = rb + tid;
            bool picked = false;
            if (i < r1) {
                const int nc = min(max(cnt[bg * n + i], 0), kk);
                const int32_t *sl = idx + (bg * n + i) * kk;
                for (int t = 0; t < nc; ++t) picked |= sl[t] == blk;
            }
            const uint64_t bal = __ballot(picked);
            if (lane == 0) wcount[w] = __popcll(bal);
            __syncthreads();
            int base = nrt;
            for (int t = 0; t < 4; ++t) {
                if (t < w) base += wcount[t];
                nrt += wcount[t];
            }
            if (picked) rows[base + __popcll(bal & ((1ull << lane) - 1ull))] = i;
            __syncthreads();
        }
    }
    // from here on each wave is alone
    const int j0 = 64 * blk + 16 * w, j = j0 + l16;
    const int wa = max(j0, r0), wb = sinks ? -1 : min(min(n, j0 + 16 + W - 1), r1);   // window rows [wa, wb)
    const bool any = sinks ? (16 * w < S && r1 > j0) : (wb > wa || nrt > 0);
    if (!DIRECT && lane == 0) used[slot] = any;
    if (!any && (!DIRECT || split0 > 0)) return;
    const uint32_t magic = 0xffffffffu / (uint32_t)G + 1u;   // G > 1: u / G = umulhi(u, magic) for u < 2^16
    const int64_t qb = b * n * Hq * D;
    f32x4 kf[NC], vf[NC], gk[NC], gv[NC];
    auto load_k = [&](const float *src) {
#pragma unroll
        for (int c = 0; c < NC; ++c) kf[c] = ld4(src + (bg * n + j) * D + 16 * c + 4 * lg);
    };
#pragma unroll
    for (int c = 0; c < NC; ++c) vf[c] = ld4(v + ((b * n + j) * Hkv + g) * D + 16 * c + 4 * lg);

    // the pairs (row_of(u / G), head u % G), u < total, against the wave's
    // keys.  mode 0: window rows, 1: sink keys, 2: rows that attend them all
    auto run = [&](int total, auto row_of, int mode, const float *qx, bool safe) {
        f32x4 xa[NC], da[NC];
        int rh, row;
        float lse, dd;
        auto load = [&](int t) {
            const int uu = min(16 * t + l16, total - 1);
            const int r = (G == 1) ? uu : (int)__umulhi((uint32_t)uu, magic);
            const int h = g * G + uu - r * G;
            row = row_of(r);
            rh = row * Hq + h;
            const int64_t ro = qb + (int64_t)rh * D + 4 * lg;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                xa[c] = ld4(qx + ro + 16 * c);
                da[c] = ld4(dout + ro + 16 * c);
            }
            const int64_t so = (b * Hq + h) * n + row;
            lse = lse_ws[so];
            dd = dd_ws[so];
        };
        const int nt = (total + 15) / 16;
        load(0);
        for (int t = 0; t < nt; ++t) {
            // the pairs 4 lg + e of the accumulators' rows, and their rows
            // transposed: elements 16 c + l16
            float xb[4][NC], ob[4][NC], lseb[4], ddb[4];
            bool valid[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int src = 4 * lg + e;
                const int64_t ro = qb + (int64_t)__shfl(rh, src, 64) * D + l16;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    xb[e][c] = qx[ro + 16 * c];
                    ob[e][c] = dout[ro + 16 * c];
                }
                lseb[e] = __shfl(lse, src, 64);
                ddb[e] = __shfl(dd, src, 64);
                const int ri = __shfl(row, src, 64);
                const bool in = (mode == 0) ? (j >= S && ri >= j && ri - j < W) : (mode == 1) ? (j < S && ri >= j) : true;
                valid[e] = in && 16 * t + src < total;
            }
            f32x4 Sa = {0.f, 0.f, 0.f, 0.f}, dP = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    Sa = mma4(xa[c][e], kf[c][e], Sa);
                    dP = mma4(da[c][e], vf[c][e], dP);
                }
            if (t + 1 < nt) load(t + 1);
            float p[4], ds[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                p[e] = valid[e] ? expf(Sa[e] * scale - lseb[e]) : 0.0f;
                ds[e] = valid[e] ? p[e] * (dP[e] - ddb[e]) * scale : 0.0f;
            }
            if (!safe) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        gv[c] = mma4(p[e], ob[e][c], gv[c]);
                        gk[c] = mma4(ds[e], xb[e][c], gk[c]);
                    }
            } else {
                // the same sums without the masked products: pair 4 tg + te
                // against keys 4 lg + e
#pragma nounroll
                for (int tg = 0; tg < 4; ++tg)
#pragma unroll
                    for (int te = 0; te < 4; ++te)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int src = 16 * tg + 4 * lg + e;
                            const float pp = __shfl(p[te], src, 64), dd2 = __shfl(ds[te], src, 64);
                            const int vv = __shfl((int)valid[te], src, 64);
#pragma unroll
                            for (int c = 0; c < NC; ++c) {
                                const float o = __shfl(ob[te][c], 16 * tg + l16, 64);
                                const float xx = __shfl(xb[te][c], 16 * tg + l16, 64);
                                if (vv) {
                                    gv[c][e] = fmaf(pp, o, gv[c][e]);
                                    gk[c][e] = fmaf(dd2, xx, gk[c][e]);
                                }
                            }
                        }
            }
        }
    };
    for (int safe = 0;; safe = 1) {
#pragma unroll
        for (int c = 0; c < NC; ++c) gk[c] = gv[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (DIRECT && !any) break;
        if (sinks) {
            load_k(kc);
            const int ra = max(r0, j0);
            run((r1 - ra) * G, [&](int r) { return ra + r; }, 1, qc_ws, safe);
        }
        if (wb > wa) {
            load_k(kr);
            run((wb - wa) * G, [&](int r) { return wa + r; }, 0, qr_ws, safe);
            // rope^T at the keys' positions; d and d +- D/2 sit in one lane
            f32x4 zs[NC];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float *cp = cosT + (int64_t)(j0 + 4 * lg + e) * D + l16;
                const float *sp = sinT + (int64_t)(j0 + 4 * lg + e) * D + l16;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    zs[c][e] = gk[c][e] * sp[16 * c];
                    gk[c][e] *= cp[16 * c];
                }
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) gk[c] += (c < NC / 2) ? zs[(c + NC / 2) % NC] : -zs[(c + NC / 2) % NC];
        }
        if (nrt > 0) {
            load_k(kc);
            run(nrt * G, [&](int r) { return rows[r]; }, 2, qc_ws, safe);
        }
        bool fin = true;
#pragma unroll
        for (int c = 0; c < NC; ++c) fin = fin && finite4(gk[c]) && finite4(gv[c]);
        if (safe || __all(fin)) break;
    }
    const bool plus = DIRECT && split0 > 0;
    if (!DIRECT || sinks) {
        float *pp = part + slot * (2 * 16 * D) + 4 * lane;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            f32x4 *pk = reinterpret_cast<f32x4 *>(pp + 256 * c), *pv = reinterpret_cast<f32x4 *>(pp + 256 * (NC + c));
            *pk = plus ? *pk + gk[c] : gk[c];
            *pv = plus ? *pv + gv[c] : gv[c];
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t o = ((b * n + j0 + 4 * lg + e) * Hkv + g) * D + l16;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            dk[o + 16 * c] = plus ? dk[o + 16 * c] + gk[c][e] : gk[c][e];
            dv[o + 16 * c] = plus ? dv[o + 16 * c] + gv[c][e] : gv[c][e];
        }
    }
}

// dk and dv of 16 keys of one (b, g), a wave a quarter of their elements.  With
// `part`, its nr ranges' sums are added to those of the earlier launches (in dk
// and dv, the sinks' in `sink`; none if this is the first).  After the last
// launch of ranges the sinks' sums are added to block 0 and the key rows taken
// through the QKNorm backward, with one gain atomic per workgroup.  Bound by the
// latency of its reads, U places of which are in flight: 2048 tokens, 2 KV heads,
// 32 ranges 15 us, with a wave per 16 keys and 4 places 23.
template <int D>
__global__ __launch_bounds__(256) void bwd_k_f32_kernel(const float *__restrict__ part, const int *__restrict__ used,
                                                        float *__restrict__ sink, int nr, int nblk, int S, bool first,
                                                        bool last, const float *__restrict__ k,
                                                        const float *__restrict__ kgain, float eps, int n, int Hkv,
                                                        float *__restrict__ dk, float *__restrict__ dv,
                                                        float *__restrict__ dk_gain) {
    constexpr int NC = D / 16, C = NC / 4, U = 16 / C;   // C: 16-element groups per wave
    __shared__ float red[4][2][16];
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = n / 64, kg = (int)(blockIdx.x & 3), blk = (int)((blockIdx.x >> 2) % nb);
    const int64_t bg = (blockIdx.x >> 2) / nb, b = bg / Hkv;
    const int g = (int)(bg % Hkv);
    const int64_t row = (b * n + 64 * (int64_t)blk + 16 * kg + 4 * lg) * Hkv + g, rs = (int64_t)Hkv * D;
    const int64_t o = row * D + 16 * C * w + l16;   // element 16 c of key e: o + e rs + 16 c
    const int fo = 256 * C * w + 4 * lane;          // this wave's first f32x4 of a slot's dk part
    f32x4 gk[C], gv[C];
    auto add = [&](int bx) {
        const int64_t s0 = (bg * nblk + bx) * nr;
        for (int c0 = 0; c0 < nr; c0 += 64) {
            const bool u = c0 + lane < nr && used[(s0 + c0 + lane) * 4 + kg] != 0;
            for (uint64_t m = __ballot(u); m;) {   // U slots' loads in flight
                f32x4 x[U][2 * C];
                bool has[U];
                int i = 0;
#pragma unroll
                for (int t = 0; t < U; ++t) {
                    has[t] = m != 0;
                    i = m ? __builtin_ctzll(m) : i;   // none left: the last one again, unused
                    m &= m - 1;
                    const float *pp = part + ((s0 + c0 + i) * 4 + kg) * (2 * 16 * D) + fo;
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        x[t][c] = ld4(pp + 256 * c);
                        x[t][C + c] = ld4(pp + 256 * (NC + c));
                    }
                }
#pragma unroll
                for (int t = 0; t < U; ++t)
                    if (has[t]) {
#pragma unroll
                        for (int c = 0; c < C; ++c) {
                            gk[c] += x[t][c];
                            gv[c] += x[t][C + c];
                        }
                    }
            }
        }
    };
    f32x4 *sp = reinterpret_cast<f32x4 *>(sink + (bg * 4 + kg) * (2 * 16 * D) + fo);
    const bool sinks = blk == 0 && S > 16 * kg;
    if (part && sinks) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            gk[c] = first ? f32x4{0.f, 0.f, 0.f, 0.f} : sp[64 * c];
            gv[c] = first ? f32x4{0.f, 0.f, 0.f, 0.f} : sp[64 * (NC + c)];
        }
        add(nb);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            sp[64 * c] = gk[c];
            sp[64 * (NC + c)] = gv[c];
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            gk[c][e] = first ? 0.0f : dk[o + e * rs + 16 * c];
            gv[c][e] = first ? 0.0f : dv[o + e * rs + 16 * c];
        }
    if (part) add(blk);
    if (last && sinks) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            gk[c] += sp[64 * c];
            gv[c] += sp[64 * (NC + c)];
        }
    }
    if (last && kgain) {   // uniform
        const float gn = kgain[g];
        float x[4][C], gs = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float ss = 0.0f, yx = 0.0f;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                x[e][c] = k[o + e * rs + 16 * c];
                ss = fmaf(x[e][c], x[e][c], ss);
                yx = fmaf(gk[c][e], x[e][c], yx);
            }
#pragma unroll
            for (int d = 1; d < 16; d *= 2) {   // over the key's 16 lanes
                ss += __shfl_xor(ss, d, 64);
                yx += __shfl_xor(yx, d, 64);
            }
            if (l16 == 0) {
                red[w][0][4 * lg + e] = ss;
                red[w][1][4 * lg + e] = yx;
            }
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 4 * lg + e;
            const float ss = (red[0][0][j] + red[1][0][j]) + (red[2][0][j] + red[3][0][j]);
            const float yx = (red[0][1][j] + red[1][1][j]) + (red[2][1][j] + red[3][1][j]);
            const float ms = ss / (float)D;
            const float r = sqrtf(fmaxf(ms, eps));
            const float corr = (ms >= eps) ? gn * yx / ((float)D * r * r * r) : 0.0f;
#pragma unroll
            for (int c = 0; c < C; ++c) gk[c][e] = (gn / r) * gk[c][e] - x[e][c] * corr;
            gs += yx / r;
        }
        gs = col_sum(gs);
        if (dk_gain && threadIdx.x == 0) unsafeAtomicAdd(&dk_gain[g], gs);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dk[o + e * rs + 16 * c] = gk[c][e];
            dv[o + e * rs + 16 * c] = gv[c][e];
        }
}

// Ranges of query rows (R rows each, nsplit in all) and how many of them a
// launch of bwd_dkv_f32 takes if the workspace has a place for each.  Up to 32
// ranges, and no more than make F32_WGS workgroups (16 rounds of the 512 that
// run at once): a range costs each block a place's write and read (8192 tokens,
// 8 heads: 1415 us with 32 ranges, summed by atomics, 1298 with 8 in order).  All
// of them in a launch if they are within F32_PLACES blocks (32 KB each at d = 64),
// since each launch ends with its longest blocks (32768 tokens, 14 / 2 heads: 13.6
// ms, 14.7 with two launches of 8 ranges).  A range of as many blocks fills the chip
// by itself and takes no place.
constexpr int64_t F32_WGS = 8192, F32_PLACES = 16384;
struct Plan {
    int64_t R, nsplit, nr;
};
static Plan bwd_plan(int64_t Cn, int64_t n) {
    Plan p;
    p.R = F32_RMIN;
    while ((n / p.R > 32 || Cn * (n / 64) * (n / p.R) > F32_WGS) && p.R < F32_RMAX) p.R *= 2;
    p.nsplit = (n + p.R - 1) / p.R;
    const int64_t per = Cn * (n / 64 + 1);
    p.nr = std::min(p.nsplit, (F32_PLACES + per - 1) / per);
    return p;
}
// one range's places: sums and flags
static size_t range_bytes(int64_t Cn, int64_t n, int64_t d) {
    return (size_t)(4 * Cn * (n / 64 + 1)) * (size_t)(2 * 16 * d + 1) * 4;
}

}  // namespace af

size_t attn_bwd_f32_part_bytes(int64_t B, int64_t n, int64_t Hkv, int64_t d) {
    const int64_t nr = af::bwd_plan(B * Hkv, n).nr;
    return nr < 2 ? 0 : (size_t)nr * af::range_bytes(B * Hkv, n, d);
}

template <int D>
int launch_attn_bwd_f32(const float *q, const float *k, const float *v, const float *kc, const float *kr,
                        const float *qgain, const float *kgain, float eps, const float *cosT, const float *sinT,
                        const int32_t *idx, const int32_t *cnt, const float *out, const float *dout, int64_t B,
                        int64_t n, int64_t Hq, int64_t Hkv, int64_t S, int64_t W, int64_t k_blocks, float scale,
                        float *qc_ws, float *qr_ws, float *lse_ws, float *dd_ws, float *sink, float *part,
                        size_t part_bytes, float *dq, float *dk, float *dv, float *dq_gain, float *dk_gain,
                        hipStream_t s) {
    const int64_t qpt = 16 / (Hq / Hkv), ntiles = ((n + qpt - 1) / qpt + 3) / 4, Cn = B * Hkv, nb = n / 64;
    int64_t grid;
    const int xmap = xcd_pick(Cn, ntiles, grid);
    const af::Plan p = af::bwd_plan(Cn, n);
    const int64_t places = std::min<int64_t>(p.nr, (int64_t)(part_bytes / af::range_bytes(Cn, n, D)));
    const int64_t per = places < 2 ? 1 : places;   // ranges per launch
    const int64_t nblk = nb + (S > 0);
    if (grid > 0x7fffffffLL || Cn * nblk * std::max<int64_t>(per, 4) > 0x7fffffffLL || n > 0x3fffffffLL || n * Hq > 0x7fffffffLL)
        return HBA_ERR_UNSUPPORTED;
    if (places < 2) part = nullptr;
    int *used = part ? reinterpret_cast<int *>(part + 4 * Cn * nblk * per * (2 * 16 * D)) : nullptr;
    const int Wc = (int)std::min<int64_t>(W, n);   // past n a longer window changes nothing
    hipLaunchKernelGGL(af::bwd_dq_f32_kernel<D>, dim3((unsigned)grid), dim3(256), 0, s, q, kc, kr, v, qgain, eps, cosT,
                       sinT, idx, cnt, out, dout, (int)n, (int)Hq, (int)Hkv, (int)S, Wc, (int)k_blocks, scale,
                       (int)ntiles, (int)Cn, xmap, qc_ws, qr_ws, lse_ws, dd_ws, dq, dq_gain);
    const auto dkv = part ? af::bwd_dkv_f32_kernel<D, false> : af::bwd_dkv_f32_kernel<D, true>;
    for (int64_t r0 = 0; r0 < p.nsplit; r0 += per) {
        const int64_t nr = std::min(per, p.nsplit - r0);
        const bool last = r0 + nr == p.nsplit;
        hipLaunchKernelGGL(dkv, dim3((unsigned)(Cn * nblk * nr)), dim3(256), 0, s, kc, kr, v, cosT, sinT, idx, cnt,
                           dout, (int)n, (int)Hq, (int)Hkv, (int)S, Wc, (int)k_blocks, scale, (int)p.R, (int)r0,
                           (int)nr, (int)nblk, qc_ws, qr_ws, lse_ws, dd_ws, part ? part : sink, used, dk, dv);
        if (part || (last && (kgain || S > 0)))
            hipLaunchKernelGGL(af::bwd_k_f32_kernel<D>, dim3((unsigned)(4 * Cn * nb)), dim3(256), 0, s, part, used, sink,
                               (int)nr, (int)nblk, (int)S, part && r0 == 0, last, k, kgain, eps, (int)n, (int)Hkv, dk,
                               dv, dk_gain);
    }
    return HBA_OK;
}
#define HBA_INST(D)                                                                                                \
    template int launch_attn_bwd_f32<D>(const float *, const float *, const float *, const float *, const float *, \
                                        const float *, const float *, float, const float *, const float *,         \
                                        const int32_t *, const int32_t *, const float *, const float *, int64_t,   \
                                        int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, float, float *,      \
                                        float *, float *, float *, float *, float *, size_t, float *, float *,     \
                                        float *, float *, float *, hipStream_t);
HBA_INST(64)
HBA_INST(128)
#undef HBA_INST

}  // namespace hba
