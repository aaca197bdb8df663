// Device helpers of the decoder-layer kernels (layer.hip, attn.hip): the per-head q / k norm + NEOX RoPE
// of head size 128. Include after `#pragma clang fp contract(off)`:
// these expressions must round exactly as ggml-cpu forms them (no fused multiply-adds unless written as fmaf).
#pragma once

#include "mx_device.h"

namespace mx {

// The NEOX angle of pair `lane` of a head of 128 at position p: the chain p * theta_scale ... (lane factors) as
// k_rope_neox forms it. Every lane runs the chain to the start of each group of eight pairs and keeps its own group's,
// then its remaining factors: 77 operations in a row instead of the 126 of a select after every product.
__device__ __forceinline__ void rope_angle(int64_t p, float theta_scale, float freq_scale, int lane, float &c, float &s) {
    float chain = (float)p, theta = chain;
#pragma unroll
    for (int j = 1; j <= 56; j++) {
        chain *= theta_scale;
        if (j % 8 == 0) theta = (lane >> 3) >= j / 8 ? chain : theta;
    }
#pragma unroll
    for (int j = 0; j < 7; j++) {
        const float next = theta * theta_scale;
        theta = j < (lane & 7) ? next : theta;
    }
    const float t = freq_scale * theta;
    c = cosf(t);
    s = sinf(t);
}

// One head of 128 (lane l holds channels l and l + 64, the NEOX pair l): rms_norm then mul by w; the arithmetic of
// k_rms_norm.
__device__ __forceinline__ void qk_norm(float x0, float x1, float w0, float w1, float eps, float &y0, float &y1) {
    double ss = (double)(x0 * x0) + (double)(x1 * x1);
    ss = wave_sum_d(ss);
    const float mean = (float)(ss / 128.0);
    const float scale = 1.0f / sqrtf(mean + eps);
    y0 = (x0 * scale) * w0;
    y1 = (x1 * scale) * w1;
}

// ... then RoPE at position p; the arithmetic of k_rms_norm and k_rope_neox.
__device__ __forceinline__ void qk_norm_rope(float x0, float x1, float w0, float w1, int64_t p, float eps,
                                             float theta_scale, float freq_scale, int lane, float &o0, float &o1) {
    float y0, y1, c, s;
    qk_norm(x0, x1, w0, w1, eps, y0, y1);
    rope_angle(p, theta_scale, freq_scale, lane, c, s);
    o0 = y0 * c - y1 * s;
    o1 = y0 * s + y1 * c;
}

}  // namespace mx
