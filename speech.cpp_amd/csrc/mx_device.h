// Device-side helpers for libmx's gfx950 kernels: fp16 conversion, wave64 reductions and the activation quantizers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mx.h"

namespace mx {

// fp16 bits <-> fp32. v_cvt_f16_f32 rounds to nearest even and keeps binary16 subnormals (the default FP mode of a
// HIP kernel), which is IEEE conversion as ggml_compute_fp32_to_fp16 performs it.
__device__ __forceinline__ float h2f(uint16_t h) {
    _Float16 v;
    __builtin_memcpy(&v, &h, 2);
    return (float)v;
}
__device__ __forceinline__ uint16_t f2h(float f) {
    _Float16 v = (_Float16)f;
    uint16_t h;
    __builtin_memcpy(&h, &v, 2);
    return h;
}

// Cross-lane exchanges on DPP (a modifier of the consuming VALU op: no LDS round trip). Each control reads, for lane
// i: XOR1 / XOR2 lane i^1 / i^2 of its quad; HALF_MIRROR lane 7-i of its eight; MIRROR lane 15-i of its row of 16;
// BCAST15 lane 15 of the row below (written into rows 1 and 3 with row mask 0xA); BCAST31 lane 31 (rows 2 and 3, row
// mask 0xC). Lanes of rows outside the row mask get `old`.
namespace dpp {
constexpr int XOR1 = 0xB1, XOR2 = 0x4E, HALF_MIRROR = 0x141, MIRROR = 0x140, BCAST15 = 0x142, BCAST31 = 0x143;
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int dpp_i(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROW_MASK, 0xF, false);
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_f(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, ROW_MASK, 0xF,
                                                      false));
}

// Sum over aligned groups of WIDTH lanes (16, 32 or 64). Exact in the group's last lane (lane % WIDTH == WIDTH - 1);
// for WIDTH 16 in every lane.
template <int WIDTH>
__device__ __forceinline__ float sum_lanes(float v) {
    static_assert(WIDTH == 16 || WIDTH == 32 || WIDTH == 64, "group of 16, 32 or 64 lanes");
    v += dpp_f<dpp::XOR1>(0.0f, v);
    v += dpp_f<dpp::XOR2>(0.0f, v);
    v += dpp_f<dpp::HALF_MIRROR>(0.0f, v);
    v += dpp_f<dpp::MIRROR>(0.0f, v);
    if (WIDTH >= 32) v += dpp_f<dpp::BCAST15, 0xA>(0.0f, v);
    if (WIDTH >= 64) v += dpp_f<dpp::BCAST31, 0xC>(0.0f, v);
    return v;
}

// The butterfly x_i + x_(i ^ 32), then ^ 16, 8, 4, 2, 1, in every lane, without an LDS round trip: the halves and the rows
// of 16 are exchanged by permlane swaps; after the step over 8 the values repeat every 8 lanes (then every 4), so that
// rotations of a row by 8 and 4 read lanes i ^ 8 and one equal to lane i ^ 4.
namespace lanes {
constexpr int ROR8 = 0x128, ROR4 = 0x124;
__device__ __forceinline__ void swap32(uint32_t v, uint32_t &lo, uint32_t &hi) {  // both halves' values in every lane
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    lo = r[0];
    hi = r[1];
}
__device__ __forceinline__ void swap16(uint32_t v, uint32_t &lo, uint32_t &hi) {  // both rows' of a pair of rows
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    lo = r[0];
    hi = r[1];
}
}  // namespace lanes

__device__ __forceinline__ double wave_sum_d(double v) {
    auto w = [](double x, int i) { return (uint32_t)(__builtin_bit_cast(uint64_t, x) >> (32 * i)); };
    auto d = [](uint32_t lo, uint32_t hi) { return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo); };
    uint32_t a0, b0, a1, b1;
    lanes::swap32(w(v, 0), a0, b0);
    lanes::swap32(w(v, 1), a1, b1);
    v = d(a0, a1) + d(b0, b1);
    lanes::swap16(w(v, 0), a0, b0);
    lanes::swap16(w(v, 1), a1, b1);
    v = d(a0, a1) + d(b0, b1);
#define MX_STEP(CTRL) v += d((uint32_t)dpp_i<CTRL>(0, (int)w(v, 0)), (uint32_t)dpp_i<CTRL>(0, (int)w(v, 1)))
    MX_STEP(lanes::ROR8);
    MX_STEP(lanes::ROR4);
    MX_STEP(dpp::XOR2);
    MX_STEP(dpp::XOR1);
#undef MX_STEP
    return v;
}
__device__ __forceinline__ float wave_sum_f(float v) {
    uint32_t a, b;
    lanes::swap32(__float_as_uint(v), a, b);
    v = __uint_as_float(a) + __uint_as_float(b);
    lanes::swap16(__float_as_uint(v), a, b);
    v = __uint_as_float(a) + __uint_as_float(b);
    v += dpp_f<lanes::ROR8>(0.0f, v);
    v += dpp_f<lanes::ROR4>(0.0f, v);
    v += dpp_f<dpp::XOR2>(0.0f, v);
    v += dpp_f<dpp::XOR1>(0.0f, v);
    return v;
}
__device__ __forceinline__ float wave_max_f(float v) {
    uint32_t a, b;
    lanes::swap32(__float_as_uint(v), a, b);
    v = fmaxf(__uint_as_float(a), __uint_as_float(b));
    lanes::swap16(__float_as_uint(v), a, b);
    v = fmaxf(__uint_as_float(a), __uint_as_float(b));
    v = fmaxf(v, dpp_f<lanes::ROR8>(0.0f, v));
    v = fmaxf(v, dpp_f<lanes::ROR4>(0.0f, v));
    v = fmaxf(v, dpp_f<dpp::XOR2>(0.0f, v));
    v = fmaxf(v, dpp_f<dpp::XOR1>(0.0f, v));
    return v;
}

// ------------------------------------------------------------------------------------------------------------------
// Buffer-to-LDS copies and their waits (the prefill GEMMs' and the MoE product's operand rings).
// ------------------------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// The LDS address of a pointer into the workgroup's shared memory.
__device__ __forceinline__ uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(const lds_void *)p; }

// A buffer descriptor for raw dword loads: base, no stride, `bytes` records (reads past them return zeros), format
// word as the buffer-resource builtin makes it for these loads.
__device__ __forceinline__ v4u buf_rsrc(const void *base, uint32_t bytes) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    return v4u{(uint32_t)b, (uint32_t)(b >> 32), bytes, 0x00020000u};
}

// Buffer-to-LDS copies (each lane's 16 or 4 bytes land at m0 + 16 or 4 x lane), issued through asm: issued as the
// builtin, the compiler counts them as LDS stores that every later LDS read may alias, and waits for all of them
// (the next stages' too) before the first fragment read of a stage. Their waits are counted by the caller (wait_vm).
__device__ __forceinline__ void dma16_lds(v4u r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(r), "s"(soff)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4_lds(v4u r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(r), "s"(soff)
                 : "memory", "m0");
}

// Waits until at most n vector memory ops of this wave are outstanding. The memory clobber keeps the compiler from
// moving loads and stores across it, so the LDS reads that follow see the copies it waited for.
template <int n>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}

// The low bytes of four ints.
__device__ __forceinline__ int pack4(int a, int b, int c, int d) {
    const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0c0c0400u);
    return (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// ------------------------------------------------------------------------------------------------------------------
// Correctly rounded quotients for the quantizers, without the scaling steps of a general division (Markstein's corrected
// quotient: q = a r, q + r (a - b q)). The Q8_0 / Q8_1 quantizer has no branch to a general division either: its code,
// even when never reached, costs a decode step 25 us in 680, its instructions being fetched in 140 short kernels
// (quant256_wave keeps one, for a scale whose reciprocal may be subnormal). The divisor's mantissa is divided by and the
// exponent put back, which is exact while the quotient is normal or overflows. v_rcp_f32's last bit is the chip's own, so
// that a correct rounding is a matter of measurement: the tests quantize blocks of every mantissa.
// ------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ bool mid_range(float v) {  // |v| in [2^-60, 2^60)
    return (__float_as_uint(v) & 0x7FFFFFFFu) - (67u << 23) < (120u << 23);
}
__device__ __forceinline__ float div127(float a) {  // a / 127, a finite
    const float r = 1.0f / 127.0f, q = a * r;
    return fmaf(fmaf(-127.0f, q, a), r, q);
}
__device__ __forceinline__ float recip_mid(float d) {  // 1 / d, d in mid_range
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}
__device__ __forceinline__ float recip_to126(float d) {  // 1 / d, 0 < |d| <= 2^126
    return __builtin_amdgcn_ldexpf(recip_mid(__builtin_amdgcn_frexp_mantf(d)), -__builtin_amdgcn_frexp_expf(d));
}
__device__ __forceinline__ float quot127(float d) {  // 127 / d, d finite and not 0
    const float m = __builtin_amdgcn_frexp_mantf(d), r = recip_mid(m), q = 127.0f * r;
    return __builtin_amdgcn_ldexpf(fmaf(fmaf(-m, q, 127.0f), r, q), -__builtin_amdgcn_frexp_expf(d));
}
__device__ __forceinline__ bool zero_or_inf(float v) { return __builtin_amdgcn_classf(v, 0x264); }
// (int)roundf(x * y) for |x y| < 2^17: half away from zero by adding the largest float below a half before truncating
// (checked over every such float); the product rounds first.
__device__ __forceinline__ int round_product(float x, float y) {
#pragma clang fp contract(off)
    const float v = x * y;
    return (int)(v + copysignf(0x1.fffffep-2f, v));
}

// ------------------------------------------------------------------------------------------------------------------
// 32-block quantizer (Q8_0 / Q8_1 activations). Eight consecutive lanes hold one block, four floats each (lane j of
// the eight holds elements 4j..4j+3).
//   REF (ggml-quants.c quantize_row_q8_{0,1}_ref): d = amax/127, id = d ? 1/d : 0, q = roundf(x*id).
//   X86 (ggml-cpu x86 quantize_row_q8_{0,1}):       d = amax/127, id = amax ? 127/amax : 0, q = rint(x*id).
// The divisions are correctly rounded (the corrected quotients above), the products single roundings.
// Returns the four quants packed in an int; *d gets fp32 d (unrounded), *sum the block's quant sum (all 8 lanes).
// ------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ int quant32_lane(float4 v, int rounding, float *d_out, int *sum_out) {
    float a = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    a = fmaxf(a, dpp_f<dpp::XOR1>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::XOR2>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::HALF_MIRROR>(0.0f, a));  // every lane of the eight now holds the block's amax
    const float d = a == INFINITY ? a : div127(a);
    int q0, q1, q2, q3;
    if (rounding == MX_ROUND_X86) {
        const float id = zero_or_inf(a) ? 0.0f : quot127(a);
        q0 = (int)rintf(v.x * id);
        q1 = (int)rintf(v.y * id);
        q2 = (int)rintf(v.z * id);
        q3 = (int)rintf(v.w * id);
    } else {
        const float id = zero_or_inf(d) ? 0.0f : recip_to126(d);
        q0 = round_product(v.x, id);
        q1 = round_product(v.y, id);
        q2 = round_product(v.z, id);
        q3 = round_product(v.w, id);
    }
    int s = q0 + q1 + q2 + q3;
    s += dpp_i<dpp::XOR1>(0, s);
    s += dpp_i<dpp::XOR2>(0, s);
    s += dpp_i<dpp::HALF_MIRROR>(0, s);
    *d_out = d;
    *sum_out = s;
    return pack4(q0, q1, q2, q3);
}

// ------------------------------------------------------------------------------------------------------------------
// 256-block quantizer (Q8_K activations of Q4_K / Q6_K weights), ggml-quants.c quantize_row_q8_K_ref. One wave holds
// one block, four floats per lane (lane l holds elements 4l..4l+3).
//   max = the element of largest |x|, the first one on ties; iscale = -127/max; q = min(127, rint(iscale*x));
//   d = 1/iscale; bsums[j] = sum of q[16j..16j+15]. An all-zero block gives d = 0, q = 0 and bsums 0.
// Returns packed quants; *d the block's d; *bsum the sum over this lane's group of four lanes (16 elements).
// ------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ int quant256_wave(float4 v, int lane, float *d_out, int *bsum_out) {
    const float e[4] = {v.x, v.y, v.z, v.w};
    const float ax = fabsf(v.x), ay = fabsf(v.y), az = fabsf(v.z), aw = fabsf(v.w);
    // amax: the largest |x| (fmaxf passes NaNs over, as ggml's strict '>' scan does), reduced within rows of 16, then
    // across rows into lane 63
    float a = fmaxf(fmaxf(ax, ay), fmaxf(az, aw));
    a = fmaxf(a, dpp_f<dpp::XOR1>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::XOR2>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::HALF_MIRROR>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::MIRROR>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::BCAST15, 0xA>(0.0f, a));
    a = fmaxf(a, dpp_f<dpp::BCAST31, 0xC>(0.0f, a));
    const float amax = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(a), 63));
    if (amax == 0.0f) {
        *d_out = 0.0f;
        *bsum_out = 0;
        return 0;
    }
    // max: the element of the first index (4 lane + j) whose |x| is amax -- the lowest lane holding one, its lowest j
    const uint64_t m0 = __ballot(ax == amax), m1 = __ballot(ay == amax), m2 = __ballot(az == amax),
                   m3 = __ballot(aw == amax);
    const int L = __builtin_ctzll(m0 | m1 | m2 | m3);
    const int c = ((m0 >> L) & 1) ? 0 : (((m1 >> L) & 1) ? 1 : (((m2 >> L) & 1) ? 2 : 3));
    const float mine = c == 0 ? v.x : (c == 1 ? v.y : (c == 2 ? v.z : v.w));
    const float maxv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), L));
    const float iscale = zero_or_inf(maxv) ? -127.0f * __builtin_amdgcn_rcpf(maxv) : -quot127(maxv);
    int q[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int t = (int)rintf(iscale * e[j]);
        q[j] = t < 127 ? t : 127;
    }
    int s = q[0] + q[1] + q[2] + q[3];
    s += dpp_i<dpp::XOR1>(0, s);
    s += dpp_i<dpp::XOR2>(0, s);
    *d_out = mid_range(iscale) ? recip_mid(iscale) : 1.0f / iscale;  // (1 / iscale may be subnormal; uniform)
    *bsum_out = s;
    return pack4(q[0], q[1], q[2], q[3]);
}

}  // namespace mx
