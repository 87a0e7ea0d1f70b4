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
//                dK += dS^T . X.  The ranges' sums meet in dk and dv by fp32
//                atomics.
//   bwd_k_f32:   the QKNorm backward of the key rows, in place.
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
    float *__restrict__ lse_ws, float *__restrict__ dd_ws, float *__restrict__ dq, float *__restrict__ dk,
    float *__restrict__ dv, float *__restrict__ dq_gain) {
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
        // bwd_dkv_f32 adds into the key rows of these positions next
        for (int r = i0; r <= u.ilast; ++r)
            for (int t = lane; t < D; t += 64) {
                dk[((b * n + r) * Hkv + g) * D + t] = 0.0f;
                dv[((b * n + r) * Hkv + g) * D + t] = 0.0f;
            }
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
            for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4 *>(dq + row + 16 * c) = y[c];
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
// stands for the sink keys of block 0, which every row from j on attends.
// About 32 ranges per sequence balance the blocks' rows (a block that many
// queries picked, a range that a window only touches): at 2048 tokens, 14 / 2
// heads, ranges of 256 rows took 424 us, 128 303, 64 263; at 4096 256 853, 128
// 790.  Past 64K tokens ranges stay at 2048 rows, so that the list fits LDS.
constexpr int F32_RMIN = 64, F32_RMAX = 2048;

template <int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_dkv_f32_kernel(
    const float *__restrict__ kc, const float *__restrict__ kr, const float *__restrict__ v,
    const float *__restrict__ cosT, const float *__restrict__ sinT, const int32_t *__restrict__ idx,
    const int32_t *__restrict__ cnt, const float *__restrict__ dout, int n, int Hq, int Hkv, int S, int W, int kk,
    float scale, int R, int nsplit, int nblk, const float *__restrict__ qc_ws, const float *__restrict__ qr_ws,
    const float *__restrict__ lse_ws, const float *__restrict__ dd_ws, float *__restrict__ dk,
    float *__restrict__ dv) {
    constexpr int NC = D / 16;
    __shared__ int rows[F32_RMAX];
    __shared__ int wcount[4];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = n / 64, G = Hq / Hkv;
    const int bx = (int)(blockIdx.x % nblk), split = (int)((blockIdx.x / nblk) % nsplit);
    const int64_t bg = blockIdx.x / ((int64_t)nblk * nsplit), b = bg / Hkv;
    const int g = (int)(bg % Hkv);
    const bool sinks = bx == nb;
    const int blk = sinks ? 0 : bx;
    const int r0 = split * R, r1 = min(n, r0 + R);

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
    if (sinks && 16 * w >= S) return;
    const int j0 = 64 * blk + 16 * w, j = j0 + l16;
    const int wa = max(j0, r0), wb = sinks ? -1 : min(min(n, j0 + 16 + W - 1), r1);   // window rows [wa, wb)
    if (!sinks && wb <= wa && nrt == 0) return;
    if (sinks && r1 <= j0) return;
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
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (sinks && j0 + 4 * lg + e >= S) continue;
        const int64_t o = ((b * n + j0 + 4 * lg + e) * Hkv + g) * D + l16;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            unsafeAtomicAdd(dk + o + 16 * c, gk[c][e]);
            unsafeAtomicAdd(dv + o + 16 * c, gv[c][e]);
        }
    }
}

// The QKNorm backward of key rows, in place on dk: a workgroup takes a 64-key
// block of one (b, g), lanes over d; one gain atomic per workgroup.
template <int D>
__global__ __launch_bounds__(256) void bwd_k_f32_kernel(const float *__restrict__ k, const float *__restrict__ kgain,
                                                        float eps, int64_t n, int Hkv, float *__restrict__ dk,
                                                        float *__restrict__ dk_gain) {
    constexpr int E = D / 64;
    __shared__ float gsum[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t bg = blockIdx.x / (n / 64), b = bg / Hkv;
    const int g = (int)(bg % Hkv);
    const float gn = kgain[g];
    float gs = 0.0f;
    for (int rr = 0; rr < 16; ++rr) {
        const int64_t j = (blockIdx.x % (n / 64)) * 64 + 16 * w + rr;
        const int64_t o = ((b * n + j) * Hkv + g) * D + lane;
        float x[E], y[E], ss = 0.0f, yx = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            x[e] = k[o + 64 * e];
            y[e] = dk[o + 64 * e];
            ss = fmaf(x[e], x[e], ss);
            yx = fmaf(y[e], x[e], yx);
        }
        const float ms = wave_sum(ss) / (float)D;
        yx = wave_sum(yx);
        const float r = sqrtf(fmaxf(ms, eps));
        const float corr = (ms >= eps) ? gn * yx / ((float)D * r * r * r) : 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) dk[o + 64 * e] = (gn / r) * y[e] - x[e] * corr;
        gs += yx / r;
    }
    if (dk_gain) {
        if (lane == 0) gsum[w] = gs;
        __syncthreads();
        if (threadIdx.x == 0) unsafeAtomicAdd(&dk_gain[g], (gsum[0] + gsum[1]) + (gsum[2] + gsum[3]));
    }
}

}  // namespace af

template <int D>
int launch_attn_bwd_f32(const float *q, const float *k, const float *v, const float *kc, const float *kr,
                        const float *qgain, const float *kgain, float eps, const float *cosT, const float *sinT,
                        const int32_t *idx, const int32_t *cnt, const float *out, const float *dout, int64_t B,
                        int64_t n, int64_t Hq, int64_t Hkv, int64_t S, int64_t W, int64_t k_blocks, float scale,
                        float *qc_ws, float *qr_ws, float *lse_ws, float *dd_ws, float *dq, float *dk, float *dv,
                        float *dq_gain, float *dk_gain, hipStream_t s) {
    const int64_t qpt = 16 / (Hq / Hkv), ntiles = ((n + qpt - 1) / qpt + 3) / 4, Cn = B * Hkv;
    int64_t grid;
    const int xmap = xcd_pick(Cn, ntiles, grid);
    int64_t R = af::F32_RMIN;
    while (n / R > 32 && R < af::F32_RMAX) R *= 2;
    const int64_t nsplit = (n + R - 1) / R, nblk = n / 64 + (S > 0), grid2 = Cn * nsplit * nblk;
    if (grid > 0x7fffffffLL || grid2 > 0x7fffffffLL || n > 0x3fffffffLL || n * Hq > 0x7fffffffLL)
        return HBA_ERR_UNSUPPORTED;
    const int Wc = (int)std::min<int64_t>(W, n);   // past n a longer window changes nothing
    hipLaunchKernelGGL(af::bwd_dq_f32_kernel<D>, dim3((unsigned)grid), dim3(256), 0, s, q, kc, kr, v, qgain, eps, cosT,
                       sinT, idx, cnt, out, dout, (int)n, (int)Hq, (int)Hkv, (int)S, Wc, (int)k_blocks, scale,
                       (int)ntiles, (int)Cn, xmap, qc_ws, qr_ws, lse_ws, dd_ws, dq, dk, dv, dq_gain);
    hipLaunchKernelGGL(af::bwd_dkv_f32_kernel<D>, dim3((unsigned)grid2), dim3(256), 0, s, kc, kr, v, cosT, sinT, idx,
                       cnt, dout, (int)n, (int)Hq, (int)Hkv, (int)S, Wc, (int)k_blocks, scale, (int)R, (int)nsplit,
                       (int)nblk, qc_ws, qr_ws, lse_ws, dd_ws, dk, dv);
    if (kgain)
        hipLaunchKernelGGL(af::bwd_k_f32_kernel<D>, dim3((unsigned)(Cn * (n / 64))), dim3(256), 0, s, k, kgain, eps, n,
                           (int)Hkv, dk, dk_gain);
    return HBA_OK;
}
#define HBA_INST(D)                                                                                                \
    template int launch_attn_bwd_f32<D>(const float *, const float *, const float *, const float *, const float *, \
                                        const float *, const float *, float, const float *, const float *,         \
                                        const int32_t *, const int32_t *, const float *, const float *, int64_t,   \
                                        int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, float, float *,      \
                                        float *, float *, float *, float *, float *, float *, float *, float *,    \
                                        hipStream_t);
HBA_INST(64)
HBA_INST(128)
#undef HBA_INST

}  // namespace hba
