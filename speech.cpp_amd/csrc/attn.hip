// FLASH_ATTN_EXT of several query rows (a prompt block, a drafted run) on the fp16 matrix cores.
//
// The (row, head) pairs that read one kv head are the columns of the products: a workgroup takes 32 of them, and its
// eight waves take turns at 32-position steps of the cache, each with a running softmax of its own that is merged at
// the end. Nothing is shared between the waves until then, so there is no barrier in the loop: every wave copies its
// steps' keys, values and mask into LDS of its own, the next keys and mask as soon as the current scores are formed,
// the next values as soon as the current ones are used. With few pairs the positions are also split over workgroups
// (partials merged by k_fa_merge).
//
// Per step: S^T = K Q^T (v_mfma_f32_32x32x16_f16; a lane ends up with 16 positions of one pair, so the row maximum and
// sum are register reductions and one exchange), softmax in fp32, O^T += V^T P^T with V read transposed from LDS
// (ds_read_b64_tr_b16). A weight is multiplied in as the sum of two fp16 values, hi + lo, scaled by 2^13 so that lo keeps
// full precision: 23 bits together, where the weight itself, an exponential rounded to 24, is good to about as many.
// The running maximum is a reference that moves only when a score passes it by more than 2 (weights then stay below e^2,
// 2^16 in fp16), so the accumulators are rarely rescaled; a larger margin would cost the large weights' exponents bits.
// Error against double precision over 64 shapes of 2 to 512 rows, relative to the one-row kernels': 0.50 of it on
// (geometric) average; with exact scores, few positions: 7.3e-8 against 7.7e-8.
//
// What bounds it: the VALU, at about 14 issue slots a score against 6 of the matrix cores (two waves per SIMD). 512 rows
// at 1024 positions before them, 16 heads on 8 of 128: 21 us, 25 with the q / k norms, RoPE and stores before it, where
// one workgroup per row (k_fa_gqa) takes 366 (an earlier form 16-21 us; on four waves and a two-slot ring 29.6, q not
// staged through LDS and the rescale inside the loop 25.5).
#include "mx_common.h"
#include "mx_device.h"

// s = dot * scale + mask with two roundings, as ggml-cpu and the one-row kernels form it
#pragma clang fp contract(off)

#include "mx_layer.h"

namespace mx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

constexpr int FM_P = 32, FM_STEP = 32, FM_W = 8;  // pairs of a workgroup, positions of a step, waves

template <int D>
struct FmLds {
    static constexpr int RB = 2 * D, CH = D / 8;  // bytes and 16-byte chunks of a K / V row
    static constexpr int K = 0, V = FM_STEP * RB, M = 2 * FM_STEP * RB, SLOT = M + FM_P * 64;  // mask: 64 bytes a pair
    static constexpr int RPC = 64 / CH, OPK = FM_STEP / RPC, OPM = FM_P / 16;  // rows of a copy; copies
    static constexpr int RING = FM_W * SLOT;
    static constexpr int OS = D + 4;  // floats between pairs of the waves' merged sums
    static constexpr int STAT = FM_W * FM_P * 8, OUT = STAT + FM_W * FM_P * OS * 4;
    static constexpr int Q = RING, END = Q + FM_P * RB;  // the pairs' q rows in fp16, laid out as a key tile
    static constexpr int SIZE = END > OUT ? END : OUT;
    static_assert(SIZE <= 160 * 1024 && OUT + FM_W * (D + 64) * 4 <= SIZE, "LDS");
};

// Chunk c of K row r lies at c ^ fm_swk(r), of V row r at c ^ fm_swv(r): the rows of a key fragment read (16 at one
// chunk), and the eight rows by two chunks of a transposed value read, cover all banks.
template <int D>
__device__ __forceinline__ int fm_swk(int r) {
    return D == 128 ? r & 15 : (r >> 1) & 7;
}
template <int D>
__device__ __forceinline__ int fm_swv(int r) {
    return D == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3);
}

// Over lanes l and l ^ 32.
__device__ __forceinline__ float half_max(float v) {
    uint32_t a, b;
    lanes::swap32(__float_as_uint(v), a, b);
    return fmaxf(__uint_as_float(a), __uint_as_float(b));
}
__device__ __forceinline__ float half_sum(float v) {
    uint32_t a, b;
    lanes::swap32(__float_as_uint(v), a, b);
    return __uint_as_float(a) + __uint_as_float(b);
}

// fp16 of a times s and of b times s, in two instructions (left to the compiler: two products and a conversion)
__device__ __forceinline__ v2h fm_halves(float a, float b, float s) {
    v2h h;
    asm("v_fma_mixlo_f16 %0, %1, %3, 0\n\tv_fma_mixhi_f16 %0, %2, %3, 0" : "=&v"(h) : "v"(a), "v"(b), "s"(s));
    return h;
}

template <int D, bool MASK>
__global__ __launch_bounds__(64 * FM_W) void k_fa_mfma(FaArgs a) {
    using L = FmLds<D>;
    constexpr int DT = D / 32, KB = D / 16, OPS_K = L::OPK + (MASK ? L::OPM : 0), OPS_V = L::OPK;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t hk = blockIdx.x, split = blockIdx.z;
    const uint32_t p0 = blockIdx.y * FM_P, gqa = (uint32_t)a.gqa, np = (uint32_t)a.n_q * gqa;
    const int64_t j0 = split * a.split_len, j1 = min(a.n_kv, j0 + a.split_len);
    const int len = (int)(j1 - j0), nst = (len + FM_STEP - 1) / FM_STEP;  // a split is never empty
    auto row_of = [&](uint32_t p) -> uint32_t { return min(p, np - 1) / gqa; };

    // copies: descriptors end with the split's last position: past it they read zeros
    const v4u rk = buf_rsrc((const uint8_t *)a.k + hk * a.k_nb2 + j0 * a.k_nb1, (uint32_t)((len - 1) * a.k_nb1 + 2 * D));
    const v4u rv = buf_rsrc((const uint8_t *)a.v + hk * a.v_nb2 + j0 * a.v_nb1, (uint32_t)((len - 1) * a.v_nb1 + 2 * D));
    const uint32_t i0 = __builtin_amdgcn_readfirstlane(row_of(p0)), mnb = (uint32_t)a.m_nb1;
    // (to the end of the 16 bytes that hold the last position: a piece that the descriptor cuts would read as zeros)
    const uint32_t mend = __builtin_amdgcn_readfirstlane((row_of(p0 + FM_P - 1) - i0) * mnb) +
                          (((uint32_t)(a.n_kv - j0) * 2 + 15) & ~15u);
    const v4u rm = buf_rsrc((const uint8_t *)a.mask + i0 * a.m_nb1 + j0 * 2, mend);
    uint32_t vk[L::OPK], vv[L::OPK], vm[L::OPM];
#pragma unroll
    for (int o = 0; o < L::OPK; o++) {
        const int r = L::RPC * o + lane / L::CH, c = lane % L::CH;
        vk[o] = (uint32_t)r * (uint32_t)a.k_nb1 + 16u * (uint32_t)(c ^ fm_swk<D>(r));
        vv[o] = (uint32_t)r * (uint32_t)a.v_nb1 + 16u * (uint32_t)(c ^ fm_swv<D>(r));
    }
#pragma unroll
    for (int o = 0; o < L::OPM; o++) {  // 16 pairs of four 16-byte chunks; chunk c of pair p at c ^ (p / 4) % 4
        const int p = 16 * o + lane / 4, c = (lane & 3) ^ ((p >> 2) & 3);
        vm[o] = MASK ? (row_of(p0 + p) - i0) * mnb + 16u * (uint32_t)c : 0u;
    }
    const uint32_t base = lds_addr(smem) + (uint32_t)(wave * L::SLOT);
    auto issue_k = [&](int st) __attribute__((always_inline)) {  // a step's keys and mask
        const uint32_t sk = (uint32_t)(st * FM_STEP) * (uint32_t)a.k_nb1;
#pragma unroll
        for (int o = 0; o < L::OPK; o++) dma16_lds(rk, base + L::K + 1024u * o, vk[o], sk);
        if constexpr (MASK)
#pragma unroll
            for (int o = 0; o < L::OPM; o++) dma16_lds(rm, base + L::M + 1024u * o, vm[o], (uint32_t)(st * FM_STEP * 2));
    };
    auto issue_v = [&](int st) __attribute__((always_inline)) {
        const uint32_t sv = (uint32_t)(st * FM_STEP) * (uint32_t)a.v_nb1;
#pragma unroll
        for (int o = 0; o < L::OPK; o++) dma16_lds(rv, base + L::V + 1024u * o, vv[o], sv);
    };
    // this wave's LDS reads have returned: what they read may be copied over
    auto reads_done = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

    if (wave < nst) {
        issue_k(wave);
        issue_v(wave);
    }
    // the pairs' q rows, rounded to fp16 as ggml converts q to K's type: one 8-channel chunk per thread, through LDS (each
    // lane reading its fragments from its own row costs 64 lines a load). Loads return in order, so a wave that waits for
    // its q has its first step's copies too.
    if (tid < FM_P * L::CH) {
        const int pr = tid / L::CH, c = tid % L::CH;
        const uint32_t pc = min(p0 + (uint32_t)pr, np - 1), qi = pc / gqa;
        const int64_t qh = hk * a.gqa + (pc - qi * gqa);
        const float *q = (const float *)((const uint8_t *)a.q + qi * a.q_nb1 + qh * a.q_nb2) + 8 * c;
        const v4f u = *(const v4f *)q, w = *(const v4f *)(q + 4);
        *(v8h *)(smem + L::Q + pr * L::RB + 16 * (c ^ fm_swk<D>(pr))) =
            v8h{(_Float16)u[0], (_Float16)u[1], (_Float16)u[2], (_Float16)u[3],
                (_Float16)w[0], (_Float16)w[1], (_Float16)w[2], (_Float16)w[3]};
    }
    // fragment addresses within a slot
    uint32_t ko[KB], vo[DT][4], mo[4];
#pragma unroll
    for (int kb = 0; kb < KB; kb++) ko[kb] = (uint32_t)(L::K + fr * L::RB + 16 * ((2 * kb + fh) ^ fm_swk<D>(fr)));
    // B fragments of S^T: column (pair) fr, k = 16 kb + 8 fh ..
    v8h qf[KB];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int kb = 0; kb < KB; kb++) qf[kb] = *(const v8h *)(smem + L::Q + ko[kb]);
    // a transposed read gives lane l of each 16 the four rows (4 fh ..) of value channel l; rows 8 u + 4 fh .. + 3
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int r = 8 * u + 4 * fh + ((lane & 15) >> 2), c = 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
            vo[dt][u] = (uint32_t)(L::V + r * L::RB + 16 * (c ^ fm_swv<D>(r)) + 8 * (lane & 1));
        }
#pragma unroll
    for (int u = 0; u < 4; u++) mo[u] = (uint32_t)(L::M + fr * 64 + 16 * (u ^ ((fr >> 2) & 3)) + 8 * fh);

    v16f zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.0f;
    v16f O[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) O[dt] = zero;
    float Mr = -INFINITY, l = 0.0f;  // the reference exponent and this lane's half of the row's sum
    constexpr float LOG2E = 1.44269504f, LN2 = 0.693147181f;
    constexpr float PSCALE = 0x1p13f;  // of the weights on their way to fp16: at most e^2, so below fp16's largest

    const uint8_t *sl = smem + wave * L::SLOT;
    v16f S;                 // register r of lane l: position 8 (r / 4) + 4 fh + r % 4 of the step, pair fr
    float Mn = -INFINITY;   // the reference that the scores of S ask for
    float sc = 1.0f;        // s = S * sc
    bool plain = false;     // no score of S is hidden
    bool formed = false;    // S holds the current step's scores
    int st = wave;
    for (;;) {  // (the accumulators are rescaled outside the loop that accumulates, so that it works on them in place)
        bool rescale = false;
        for (; st < nst; st += FM_W, formed = false) {
            const bool more = st + FM_W < nst;  // uniform
            if (!formed) {
                wait_vm<OPS_V>();  // the keys and mask have landed (the values, issued after them, may not)
                const bool tail = (st + 1) * FM_STEP > len;  // uniform
                v2u mw[4];
                bool add = tail || !(a.scale > 0.0f);  // scores to mask, or not to be compared before they are scaled
                bool hidden = false;                   // every position of the step is masked off for every pair
                if constexpr (MASK) {
                    uint32_t any = 0, all = 0xFC00FC00u;
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        mw[u] = *(const v2u *)(sl + mo[u]);
                        any |= mw[u].x | mw[u].y;
                        all = mw[u].x == 0xFC00FC00u && mw[u].y == 0xFC00FC00u ? all : 0u;
                    }
                    hidden = __all(all != 0);
                    add = add || __any(any != 0);
                }
                S = zero;
                if (!hidden)
#pragma unroll
                    for (int kb = 0; kb < KB; kb++)
                        S = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const v8h *)(sl + ko[kb]), qf[kb], S, 0, 0, 0);
                reads_done();
                if (more) issue_k(st + FM_W);
                if (hidden) {
                    if (more) issue_v(st + FM_W);  // (over values that nothing reads; a copy still on its way lands first)
                    continue;
                }
                sc = a.scale;
                if (add) {
                    sc = 1.0f;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float s = S[r] * a.scale;
                        if constexpr (MASK) {
                            const uint32_t w = (r & 2) ? mw[r >> 2].y : mw[r >> 2].x;
                            const float m = h2f((uint16_t)((r & 1) ? w >> 16 : w & 0xFFFF));
                            s = m == -INFINITY ? -INFINITY : s + m;
                        }
                        if (tail && st * FM_STEP + 8 * (r >> 2) + 4 * fh + (r & 3) >= len) s = -INFINITY;
                        S[r] = s;
                    }
                }
                float mc = fmaxf(S[0], S[1]), ml = fminf(S[0], S[1]);
#pragma unroll
                for (int r = 2; r < 16; r += 2) {
                    mc = fmaxf(fmaxf(mc, S[r]), S[r + 1]);
                    ml = fminf(fminf(ml, S[r]), S[r + 1]);
                }
                plain = !__any(ml == -INFINITY);
                mc = half_max(mc) * sc;
                const bool need = mc > Mr + 2.0f;  // (always from Mr = -inf, once a score is finite)
                Mn = need ? mc : Mr;
                formed = true;
                if (__any(need)) {
                    rescale = true;
                    break;
                }
            }
            // p = exp(s - Mr): 2^(t log2 e) corrected by the rounding of its exponent (the residual in natural units)
            float p[16];
            if (plain) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float t = fmaf(S[r], sc, -Mr), y = t * LOG2E, x = __builtin_amdgcn_exp2f(y);
                    p[r] = fmaf(x, fmaf(-y, LN2, t), x);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float t = fmaf(S[r], sc, -Mr), y = t * LOG2E, x = __builtin_amdgcn_exp2f(y);
                    p[r] = S[r] == -INFINITY ? 0.0f : fmaf(x, fmaf(-y, LN2, t), x);
                }
            }
            l += (((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]))) +
                 (((p[8] + p[9]) + (p[10] + p[11])) + ((p[12] + p[13]) + (p[14] + p[15])));
            v8h hi[2], lo[2];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const v2h h = fm_halves(p[r], p[r + 1], PSCALE);
                hi[r >> 3][r & 7] = h[0];
                hi[r >> 3][(r & 7) + 1] = h[1];
                lo[r >> 3][r & 7] = (_Float16)fmaf(p[r], PSCALE, -(float)h[0]);
                lo[r >> 3][(r & 7) + 1] = (_Float16)fmaf(p[r + 1], PSCALE, -(float)h[1]);
            }
            if (more) wait_vm<OPS_K>();  // the values have landed (the next keys, issued after them, may not)
            else wait_vm<0>();
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int u = 0; u < 2; u++) {  // positions 16 u ..: k of lane half fh: rows 16 u + 4 fh .., 16 u + 8 + 4 fh ..
                    typedef __attribute__((address_space(3))) v4s lds4;
                    const v4s x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(lds_void *)(sl + vo[dt][2 * u]));
                    const v4s x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(lds_void *)(sl + vo[dt][2 * u + 1]));
                    const v8h vf = __builtin_bit_cast(v8h, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
                    O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, hi[u], O[dt], 0, 0, 0);
                    O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, lo[u], O[dt], 0, 0, 0);
                }
            reads_done();
            if (more) issue_v(st + FM_W);
        }
        if (!rescale) break;
        const float f = Mr == -INFINITY ? 0.0f : expf(Mr - Mn);
        l *= f;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) O[dt][r] *= f;
        Mr = Mn;
    }
    wait_vm<0>();  // (a last step that was hidden leaves its values' copies in flight)
    l = half_sum(l);

    // merge the waves: sums brought to the largest reference, added in wave order
    __syncthreads();  // every wave is done with its ring, and none has a copy in flight
    float *st_m = (float *)smem, *st_l = st_m + FM_W * FM_P, *os = (float *)(smem + L::STAT);
    if (fh == 0) st_m[wave * FM_P + fr] = Mr;
    __syncthreads();
    float Mt = st_m[fr];
#pragma unroll
    for (int w = 1; w < FM_W; w++) Mt = fmaxf(Mt, st_m[w * FM_P + fr]);
    const float f = Mr == -INFINITY ? 0.0f : expf(Mr - Mt);
    if (fh == 0) st_l[wave * FM_P + fr] = l * f;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int u = 0; u < 4; u++) {  // channels 32 dt + 8 u + 4 fh .. + 3
            v4f x;
#pragma unroll
            for (int c = 0; c < 4; c++) x[c] = O[dt][4 * u + c] * (f * (1.0f / PSCALE));
            *(v4f *)(os + (wave * FM_P + fr) * L::OS + 32 * dt + 8 * u + 4 * fh) = x;
        }
    __syncthreads();
    constexpr int TP = 64 * FM_W / (D / 4);  // pairs in a round of the threads, four channels each
    const int d4 = 4 * (tid % (D / 4));
    bool odd = false;  // a sum that is not finite
#pragma unroll
    for (int pr = tid / (D / 4); pr < FM_P; pr += TP) {
        const uint32_t p = p0 + (uint32_t)pr, i = p / gqa;
        if (p >= np) break;
        float M = -INFINITY, Ls = 0.0f;
        v4f x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < FM_W; w++) {
            M = fmaxf(M, st_m[w * FM_P + pr]);
            Ls += st_l[w * FM_P + pr];
            x += *(const v4f *)(os + (w * FM_P + pr) * L::OS + d4);
        }
#pragma unroll
        for (int c = 0; c < 4; c++) odd |= !(fabsf(x[c]) < INFINITY);
        const int64_t row = i * a.n_head + hk * a.gqa + (p - i * gqa);
        if (a.nsplit == 1) {
            const float inv = Ls == 0.0f ? 0.0f : 1.0f / Ls;
            *(v4f *)(a.dst + row * D + d4) = x * inv;
        } else {
            float *part = a.part + (row * a.nsplit + split) * (D + 2);
#pragma unroll
            for (int c = 0; c < 4; c++) part[2 + d4 + c] = x[c];
            if (d4 == 0) {
                part[0] = M;
                part[1] = Ls;
            }
        }
    }
    // An infinity or a NaN among the values reaches pairs that do not see its position (0 times it is NaN), and as NaN
    // those that see an infinity (times the halves of its weight). Then this wave forms its pairs' sums again, one by one
    // over the positions that each sees.
    if (!__any(odd)) return;
    wait_vm<0>();  // the stores above come first
    constexpr int PW = 64 / (D / 4);  // pairs of a wave in a round
    float *qs = (float *)(smem + L::OUT) + wave * (D + 64);
#pragma unroll 1
    for (int e = 0; e < FM_P / FM_W; e++) {
        const uint32_t p = p0 + (uint32_t)(e / PW * TP + wave * PW + e % PW), i = p / gqa;
        if (p < np) fa_row_alone<D>(a, split, hk * a.gqa + (p - i * gqa), i, lane, qs, qs + D);
    }
}

// Whether the kernel can take these tensors: 16-byte aligned q rows (read as float4) and mask rows (copied in 16-byte
// pieces), and a split's positions within 32-bit offsets.
bool fa_mfma_supported(const FaArgs &a) {
    auto al = [](const void *p, int64_t nb) { return ((uintptr_t)p & 15) == 0 && nb % 16 == 0; };
    const int64_t lim = (int64_t)1 << 31;
    return a.n_q > 1 && a.n_kv > 0 && (a.D == 64 || a.D == 128) && al(a.q, a.q_nb1) && al(a.q, a.q_nb2) &&
           (!a.mask || (al(a.mask, a.m_nb1) && a.m_nb1 >= 0 && FM_P * a.m_nb1 + 2 * a.n_kv < lim)) && a.k_nb1 >= 0 &&
           a.v_nb1 >= 0 && a.k_nb1 < lim && a.v_nb1 < lim && (a.n_kv + FM_STEP) * a.k_nb1 < lim &&
           (a.n_kv + FM_STEP) * a.v_nb1 < lim && ((uintptr_t)a.dst & 15) == 0 &&
           (a.n_q * a.gqa + FM_P - 1) / FM_P <= 65535;
}

// Splits of the positions: toward 256 workgroups (one to a CU), each of at least FM_W steps; none where the merge's launch
// costs more than further turns (us, one split / one turn a split: 5 rows at 320 positions, 16 heads on 8 of 128 8.6 /
// 10.0, 16 of 64 6.8 / 9.1; at 1088 12.0 / 10.3 in splits of two turns).
void fa_mfma_split(FaArgs &a) {
    const int64_t units = a.n_head / a.gqa * ((a.n_q * a.gqa + FM_P - 1) / FM_P), turn = FM_W * FM_STEP;
    const int64_t turns = (a.n_kv + turn - 1) / turn;
    int64_t want = units >= 160 || turns <= (a.D == 64 ? 3 : 2) ? 1 : 256 / units;
    want = want > turns ? turns : (want > 64 ? 64 : want);  // the merge holds one split per lane
    const int64_t per = (turns + want - 1) / want;
    a.nsplit = (int)((turns + per - 1) / per);
    a.split_len = per * turn;
}

template <int D, bool MASK>
static hipError_t fa_mfma_launch(const FaArgs &a, hipStream_t s) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)k_fa_mfma<D, MASK>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, FmLds<D>::SIZE);
    if (attr != hipSuccess) return attr;
    const dim3 grid((unsigned)(a.n_head / a.gqa), (unsigned)((a.n_q * a.gqa + FM_P - 1) / FM_P), (unsigned)a.nsplit);
    hipLaunchKernelGGL((k_fa_mfma<D, MASK>), grid, dim3(64 * FM_W), FmLds<D>::SIZE, s, a);
    return hipGetLastError();
}

hipError_t launch_fa_mfma(const FaArgs &a, hipStream_t s) {
    if (a.n_q == 0 || a.n_head == 0) return hipSuccess;
    const hipError_t e = a.D == 128 ? (a.mask ? fa_mfma_launch<128, true>(a, s) : fa_mfma_launch<128, false>(a, s))
                                    : (a.mask ? fa_mfma_launch<64, true>(a, s) : fa_mfma_launch<64, false>(a, s));
    if (e != hipSuccess || a.nsplit == 1) return e;
    return launch_fa_merge(a, s);
}

}  // namespace mx
