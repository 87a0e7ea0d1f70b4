// The row tiles of the fp32 union attention's kernels (forward and query
// gradient): the walk over a tile's keys and the query row in the layout of
// v_mfma_f32_16x16x4_f32.
#pragma once

#include "hba_common.h"

namespace hba {
namespace af {

__device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// the backward's callers may pass rows off 16-byte boundaries
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
__device__ __forceinline__ f32x4 ld4(const float *p) { return *reinterpret_cast<const f32x4_a4 *>(p); }
__device__ __forceinline__ bool finite4(f32x4 v) {
    return fabsf(v[0]) < INFINITY && fabsf(v[1]) < INFINITY && fabsf(v[2]) < INFINITY && fabsf(v[3]) < INFINITY;
}

// The units of a row tile (queries i0 .. ilast, each with kk picks), in
// order: sinks, routed blocks, window.  All members but pick, pq and mult are
// wave-uniform.
template <int KT>
struct Units {
    const int32_t *ix, *ct;   // picks and counts of query i0
    int nb, S, W, kk, qpt, i0, ilast, nchunk;
    int ph, sub, chunk, kb;   // phase (0 sinks, 1 routed, 2 window), KT step within a block, pick chunk, first key
    uint64_t rem;             // picks of the chunk that are still to be taken
    int pick, pq;             // this lane's pick of the chunk (-1: none) and its query
    int mult;                 // routed: how often this lane's column picked the block

    __device__ __forceinline__ void init(const int32_t *idx, const int32_t *cnt, int64_t row0, int n, int S_, int W_,
                                         int kk_, int qpt_, int i0_) {
        ix = idx + row0 * kk_;
        ct = cnt + row0;
        nb = n / 64;
        S = S_;
        W = W_;
        kk = kk_;
        i0 = i0_;
        ilast = min(i0_ + qpt_, n) - 1;
        qpt = ilast - i0 + 1;
        nchunk = (qpt * kk + 63) / 64;
        restart();
    }
    __device__ __forceinline__ void restart() {
        ph = 0;
        kb = -KT;
        sub = 64;
        chunk = -1;
        rem = 0;
        mult = 0;
    }
    __device__ __forceinline__ void load_chunk(int c, int lane, int &p, int &q) const {
        const int e = 64 * c + lane;
        q = e / kk;
        p = -1;
        if (q < qpt && e - q * kk < ct[q]) {
            const int v = ix[e];
            if (v >= 1 && v < nb) p = v;   // block 0 is never routed (sinks, window)
        }
    }
    // the next unit: its first key kb and, if routed, mult; false past the last
    __device__ __forceinline__ bool next(int lane, int qs) {
        if (ph == 0) {
            kb += KT;
            if (kb < min(S, ilast + 1)) return true;
            ph = 1;
        }
        if (ph == 1) {
            sub += KT;
            if (sub < 64) {
                kb += KT;
                return true;
            }
            for (;;) {
                while (rem == 0 && ++chunk < nchunk) {
                    load_chunk(chunk, lane, pick, pq);
                    rem = __ballot(pick > 0);
                }
                if (rem == 0) break;
                const int blk = __builtin_amdgcn_readlane(pick, __builtin_ctzll(rem));
                const uint64_t same = __ballot(pick == blk);
                rem &= ~same;
                bool seen = false;   // taken with an earlier chunk
                mult = 0;
                for (int q = 0; q < qpt; ++q) {
                    const int c = __popcll(__ballot(pick == blk && pq == q));
                    if (qs == q) mult = c;
                }
                for (int c = 0; c < nchunk; ++c) {
                    if (c == chunk || nchunk == 1) continue;
                    int p2, q2;
                    load_chunk(c, lane, p2, q2);
                    const uint64_t b2 = __ballot(p2 == blk);
                    if (b2 == 0) continue;
                    if (c < chunk) seen = true;
                    for (int q = 0; q < qpt; ++q) {
                        const int t = __popcll(__ballot(p2 == blk && q2 == q));
                        if (qs == q) mult += t;
                    }
                }
                if (seen || 64 * blk + 63 < S) continue;   // a block of sinks only counts there
                kb = 64 * blk;
                sub = 0;
                return true;
            }
            ph = 2;
            const int w0 = max(S, i0 - W + 1);
            kb = (w0 / KT) * KT - KT;
        }
        kb += KT;
        return kb <= ilast;
    }
    // the keys (from kb) of the current unit that column (query i) attends;
    // none unless ok
    __device__ __forceinline__ void range(int i, bool ok, int &lo, int &hi) const {
        if (ph == 0) {
            lo = 0;
            hi = min(S - 1, i) - kb;
        } else if (ph == 1) {
            lo = S - kb;
            hi = mult > 0 ? KT - 1 : -1;
        } else {
            lo = max(S, i - W + 1) - kb;
            hi = i - kb;
        }
        if (!ok) hi = -1;
    }
};

// One column's query row (elements 16 c + 4 lg + e), QKNorm'd in fp32
// (attention.py:88-94); the sum of squares over the column's four lanes.
// Invalid columns are zero.
template <int D>
__device__ __forceinline__ void q_load(const float *row, bool ok, const float *gain, float eps, int lg,
                                       f32x4 (&x)[D / 16], float &ms, float &r) {
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
        x[c] = ok ? ld4(row + 16 * c + 4 * lg) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(x[c][e], x[c][e], ss);
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    ms = ss / (float)D;
    r = sqrtf(ms < eps ? eps : ms);
    if (gain) {
        const float gn = *gain;
#pragma unroll
        for (int c = 0; c < D / 16; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[c][e] = (x[c][e] / r) * gn;
    }
}

// apply_rope (attention.py:40-44) on the row's elements; d and d +- D/2 sit
// in the same lane.
template <int D>
__device__ __forceinline__ void q_rope(f32x4 (&x)[D / 16], const float *cs, const float *sn, int lg) {
    constexpr int NC = D / 16;
    f32x4 y[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 16 * c + 4 * lg + e;
            const float rot = (c < NC / 2) ? -x[c + (NC / 2) % NC][e] : x[(c + NC / 2) % NC][e];
            y[c][e] = x[c][e] * cs[t] + rot * sn[t];
        }
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = y[c];
}

}  // namespace af
}  // namespace hba
