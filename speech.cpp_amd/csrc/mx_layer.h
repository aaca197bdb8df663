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

// One wave's sums of head h, row i over a split's positions, in fp32 and over the positions that the row sees alone
// (qs [D], ps [64]: LDS of its own). The second form of the attention kernels of several rows, where values are infinities
// or NaN, so small rather than fast.
template <int D>
__device__ __forceinline__ void fa_row_alone(const FaArgs &a, int64_t split, int64_t h, int64_t i, int lane, float *qs,
                                             float *ps) {
    typedef _Float16 half8 __attribute__((ext_vector_type(8)));
    constexpr int DL = D / 64, NV = 16;  // channels per lane; value rows in flight
    auto own = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    const int64_t hk = h / a.gqa, j0 = split * a.split_len, j1 = min(a.n_kv, j0 + a.split_len);
    const uint8_t *kb = (const uint8_t *)a.k + hk * a.k_nb2, *vb = (const uint8_t *)a.v + hk * a.v_nb2;
    const uint16_t *mrow = a.mask ? (const uint16_t *)((const uint8_t *)a.mask + i * a.m_nb1) : nullptr;
    const float *q = (const float *)((const uint8_t *)a.q + i * a.q_nb1 + h * a.q_nb2);
    own();
#pragma unroll
    for (int c = 0; c < DL; c++) qs[64 * c + lane] = h2f(f2h(q[64 * c + lane]));
    own();
    float M = -INFINITY, S = 0.0f, acc[DL] = {};
    for (int64_t base = j0; base < j1; base += 64) {
        const int64_t j = base + lane;
        const float m = j < j1 ? (mrow ? h2f(mrow[j]) : 0.0f) : -INFINITY;
        float s = -INFINITY;
        if (m != -INFINITY) {
            const half8 *kr = (const half8 *)(kb + j * a.k_nb1);
            float dot = 0.0f;
#pragma unroll 4
            for (int c = 0; c < D / 8; c++) {
                const half8 w = kr[c];
#pragma unroll
                for (int e = 0; e < 8; e++) dot = fmaf((float)w[e], qs[8 * c + e], dot);
            }
            s = dot * a.scale + m;
        }
        const float mc = wave_max_f(s);
        if (mc == -INFINITY && !__any(s != s)) continue;  // uniform: nothing of the chunk is seen
        const float Mn = fmaxf(M, mc), r = M == Mn ? 1.0f : expf(M - Mn), p = expf(s - Mn);
        S = S * r + wave_sum_f(s == -INFINITY ? 0.0f : p);
        M = Mn;
        own();
        ps[lane] = s == -INFINITY ? -1.0f : p;
        own();
#pragma unroll
        for (int c = 0; c < DL; c++) acc[c] *= r;
#pragma unroll 1
        for (int t0 = 0; t0 < 64; t0 += NV) {
            _Float16 v[NV][DL];
#pragma unroll
            for (int t = 0; t < NV; t++)
#pragma unroll
                for (int c = 0; c < DL; c++)
                    v[t][c] = ((const _Float16 *)(vb + min(base + t0 + t, j1 - 1) * a.v_nb1))[64 * c + lane];
#pragma unroll
            for (int t = 0; t < NV; t++) {
                const float pt = ps[t0 + t];
#pragma unroll
                for (int c = 0; c < DL; c++) acc[c] = pt < 0.0f ? acc[c] : fmaf(pt, (float)v[t][c], acc[c]);
            }
        }
    }
    const float inv = a.nsplit > 1 ? 1.0f : (S == 0.0f ? 0.0f : 1.0f / S);
    float *part = a.part + ((i * a.n_head + h) * a.nsplit + split) * (D + 2);
    float *o = a.nsplit > 1 ? part + 2 : a.dst + (i * a.n_head + h) * D;
#pragma unroll
    for (int c = 0; c < DL; c++) o[64 * c + lane] = acc[c] * inv;
    if (a.nsplit > 1 && lane == 0) {
        part[0] = M;
        part[1] = S;
    }
}

}  // namespace mx
