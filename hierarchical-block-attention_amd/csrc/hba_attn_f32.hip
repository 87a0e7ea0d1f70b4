// Union attention in fp32 on the matrix cores (v_mfma_f32_16x16x4_f32: fp32
// products and sums, 64 FLOP per SIMD and cycle).
//
// A wave takes a row tile: the G heads of 16 / G consecutive queries of one
// KV head are the 16 columns of S^T = K . Q^T (the columns that share window
// keys and routed blocks; more than 16 heads go as chunks of at most 16).  It
// walks the keys its columns attend in units of KT keys: the sinks, each
// block of the union of its queries' picks, then the window.  A lane holds
// column l16 = lane % 16 and, of a 16-key group, keys 4 lg + e (lg = lane /
// 16): the accumulator layout, which is also the operand layout of the next
// product when its step e contracts the keys {4 lg + e}.  The contraction
// over d takes the elements in the order 16 c + 4 lg + e, so that every
// operand load is 16 bytes per lane.
//
// No LDS: a unit's K and V fragments are each read once per wave, 32 KB for
// 4096 cycles of products per SIMD, half of what L1 delivers.
//
// Keys outside a column's union are masked in the probabilities, which leaves
// 0 * v in its sums.  Where v or k is not finite that is a NaN the column
// must not see, so a wave whose results are not finite takes its tile again
// with the masked products skipped one by one (`safe`).
#include <algorithm>

#include "hba_abi.h"
#include "hba_attn_f32.h"
#include "hba_attn_f32_tile.h"
#include "hba_common.h"
#include "hba_xcd.h"

namespace hba {
namespace af {

// The forward.  64-key units at d = 64 and 32-key ones at d = 128: a unit's K
// and V fragments are 128 VGPRs, so that two waves share a SIMD and each
// one's loads run half a unit ahead of their products.
template <int D>
__global__ __launch_bounds__(256, 2) void attn_f32_kernel(
    const float *__restrict__ q, int64_t qsb, int64_t qsn, int64_t qsh, const float *__restrict__ qgain, float eps,
    const float *__restrict__ kc, const float *__restrict__ kr, const float *__restrict__ vt,
    const float *__restrict__ cosT, const float *__restrict__ sinT, const int32_t *__restrict__ idx,
    const int32_t *__restrict__ cnt, int n, int Hq, int Hkv, int hc, int gw, int S, int W, int kk, float scale,
    int ntiles, int Cn, int xmap, float *__restrict__ out, int64_t osb, int64_t osn, int64_t osh) {
    constexpr int KT = (D == 64) ? 64 : 32, NC = D / 16, NM = KT / 16;
    int combo, wt;
    xcd_map(blockIdx.x, Cn, ntiles, xmap, combo, wt);
    if (wt >= ntiles || combo >= Cn) return;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = Hq / Hkv, qpt = 16 / gw;
    const int ch = combo % hc, g = (combo / hc) % Hkv;
    const int64_t b = combo / (hc * Hkv);
    const int64_t i0l = ((int64_t)wt * 4 + w) * qpt;
    if (i0l >= n) return;
    const int i0 = (int)i0l;
    const int64_t bh = b * Hkv + g;
    const int qs = l16 / gw, hh = ch * gw + l16 % gw;
    const int i = i0 + qs;
    const bool ok = qs < qpt && i < n && hh < G;
    const int h = g * G + (ok ? hh : 0);
    const float *KC = kc + bh * n * D, *KR = kr + bh * n * D, *VT = vt + bh * n * D;

    Units<KT> u;
    u.init(idx, cnt, bh * n + i0, n, S, W, kk, qpt, i0);
    f32x4 x[NC], O[NC], kf[NM][NC], vf[NC][NM];
    float m = -INFINITY, l = 0.0f;
    auto load_k = [&]() {
        const float *kp = (u.ph == 2 ? KR : KC) + (int64_t)(u.kb + l16) * D + 4 * lg;
#pragma unroll
        for (int mt = 0; mt < NM; ++mt)
#pragma unroll
            for (int c = 0; c < NC; ++c) kf[mt][c] = ld4(kp + 16 * mt * D + 16 * c);
    };
    for (int safe = 0;; safe = 1) {
        float ms, r;
        q_load<D>(q + b * qsb + (int64_t)(ok ? i : 0) * qsn + (int64_t)h * qsh, ok, qgain ? qgain + h : nullptr, eps, lg,
                  x, ms, r);
#pragma unroll
        for (int c = 0; c < NC; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        m = -INFINITY;
        l = 0.0f;
        bool roped = false;
        u.restart();
        bool more = u.next(lane, qs);
        if (more) load_k();
        while (more) {
            const float *vp = VT + (int64_t)l16 * n + u.kb + 4 * lg;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int mt = 0; mt < NM; ++mt) vf[c][mt] = ld4(vp + (int64_t)16 * c * n + 16 * mt);
            if (u.ph == 2 && !roped) {
                q_rope<D>(x, cosT + (int64_t)(ok ? i : 0) * D, sinT + (int64_t)(ok ? i : 0) * D, lg);
                roped = true;
            }
            int lo, hi;
            u.range(i, ok, lo, hi);
            const float mul = (float)(u.ph == 1 ? u.mult : 1);
            const bool full = __all(!ok || (lo <= 0 && hi >= KT - 1 && mul == 1.0f)) && !safe;
            f32x4 Sa[NM];
            bool act[NM];   // wave-uniform: the group holds a key of some column
#pragma unroll
            for (int mt = 0; mt < NM; ++mt) {
                act[mt] = full || __any(lo <= 16 * mt + 15 && hi >= 16 * mt && lo <= hi);
                Sa[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (act[mt]) {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int e = 0; e < 4; ++e) Sa[mt] = mma4(kf[mt][c][e], x[c][e], Sa[mt]);
                }
            }
            more = u.next(lane, qs);
            if (more) load_k();
            // online softmax of the column; p = 0 outside its keys
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
            const float mn = fmaxf(m, tmax);
            const float sh = (mn == -INFINITY) ? 0.0f : mn;
            const float alpha = expf(m - sh);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int c = 0; c < NC; ++c) O[c] *= alpha;
#pragma unroll
            for (int mt = 0; mt < NM; ++mt)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    Sa[mt][e] = expf(Sa[mt][e] - sh) * mul;
                    l += Sa[mt][e];
                }
            if (!safe) {
#pragma unroll
                for (int mt = 0; mt < NM; ++mt)
                    if (act[mt]) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
#pragma unroll
                            for (int c = 0; c < NC; ++c) O[c] = mma4(vf[c][mt][e], Sa[mt][e], O[c]);
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
                            const float p = __shfl(Sa[mt][te], 16 * tg + l16, 64);
#pragma unroll
                            for (int c = 0; c < NC; ++c)
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const float v = __shfl(vf[c][mt][te], 16 * tg + 4 * lg + e, 64);
                                    if (j >= lo && j <= hi) O[c][e] = fmaf(p, v, O[c][e]);
                                }
                        }
            }
        }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        bool fin = l < INFINITY;
#pragma unroll
        for (int c = 0; c < NC; ++c) fin = fin && finite4(O[c]);
        if (safe || __all(!ok || fin)) break;
    }
    if (!ok) return;
    const float inv = 1.0f / l;
    float *orow = out + b * osb + (int64_t)i * osn + (int64_t)h * osh + 4 * lg;
#pragma unroll
    for (int c = 0; c < NC; ++c) *reinterpret_cast<f32x4 *>(orow + 16 * c) = O[c] * inv;
}

}  // namespace af

template <int D>
int launch_attn_f32(const void *q, const int64_t *qs, const float *qgain, float eps, const void *kc, const void *kr,
                    const void *vt, const float *cosT, const float *sinT, const int32_t *idx, const int32_t *cnt,
                    int64_t B, int64_t n, int64_t Hq, int64_t Hkv, int64_t S, int64_t W, int64_t k, float scale,
                    void *out, const int64_t *os, hipStream_t s) {
    const int64_t G = Hq / Hkv, hc = (G + 15) / 16, gw = (G + hc - 1) / hc, qpt = 16 / gw;
    const int64_t ntiles = ((n + qpt - 1) / qpt + 3) / 4;   // workgroups of 4 row tiles
    const int64_t Cn = B * Hkv * hc;
    int64_t grid;
    const int xmap = xcd_pick(Cn, ntiles, grid);
    if (grid > 0x7fffffffLL || n > 0x3fffffffLL || qpt * k > 0x3fffffffLL) return HBA_ERR_UNSUPPORTED;
    // past n neither a longer window nor more sinks change anything
    const int Wc = (int)std::min<int64_t>(W, n), Sc = (int)std::min<int64_t>(S, n);
    hipLaunchKernelGGL(af::attn_f32_kernel<D>, dim3((unsigned)grid), dim3(256), 0, s, (const float *)q, qs[0], qs[1],
                       qs[2], qgain, eps, (const float *)kc, (const float *)kr, (const float *)vt, cosT, sinT, idx, cnt,
                       (int)n, (int)Hq, (int)Hkv, (int)hc, (int)gw, Sc, Wc, (int)k, scale, (int)ntiles, (int)Cn, xmap,
                       (float *)out, os[0], os[1], os[2]);
    return HBA_OK;
}
template int launch_attn_f32<64>(const void *, const int64_t *, const float *, float, const void *, const void *,
                                 const void *, const float *, const float *, const int32_t *, const int32_t *, int64_t,
                                 int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, float, void *, const int64_t *,
                                 hipStream_t);
template int launch_attn_f32<128>(const void *, const int64_t *, const float *, float, const void *, const void *,
                                  const void *, const float *, const float *, const int32_t *, const int32_t *, int64_t,
                                  int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, float, void *, const int64_t *,
                                  hipStream_t);

}  // namespace hba
