// Launchers of the fp32 union attention on the fp32 matrix cores: the forward
// (launch_attn_f32; any query heads per KV head, sinks, k and window) and the
// backward's query and key gradients (G <= 16, S <= 64, k <= 64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hba {

template <int D>
int launch_attn_f32(const void *q, const int64_t *qs, const float *qgain, float eps, const void *kc, const void *kr,
                    const void *vt, const float *cosT, const float *sinT, const int32_t *idx, const int32_t *cnt,
                    int64_t B, int64_t n, int64_t Hq, int64_t Hkv, int64_t S, int64_t W, int64_t k, float scale,
                    void *out, const int64_t *os, hipStream_t s);

// qc_ws, qr_ws [B, n, Hq, d]; lse_ws, dd_ws [B, Hq, n]; sink [B, Hkv, 2, 64, d];
// part: part_bytes more for the row ranges' sums of dk and dv, of which the
// launches use up to attn_bwd_f32_part_bytes; the gain gradients are added to.
size_t attn_bwd_f32_part_bytes(int64_t B, int64_t n, int64_t Hkv, int64_t d);
template <int D>
int launch_attn_bwd_f32(const float *q, const float *k, const float *v, const float *kc, const float *kr,
                        const float *qgain, const float *kgain, float eps, const float *cosT, const float *sinT,
                        const int32_t *idx, const int32_t *cnt, const float *out, const float *dout, int64_t B,
                        int64_t n, int64_t Hq, int64_t Hkv, int64_t S, int64_t W, int64_t k_blocks, float scale,
                        float *qc_ws, float *qr_ws, float *lse_ws, float *dd_ws, float *sink, float *part,
                        size_t part_bytes, float *dq, float *dk, float *dv, float *dq_gain, float *dk_gain,
                        hipStream_t s);

}  // namespace hba
