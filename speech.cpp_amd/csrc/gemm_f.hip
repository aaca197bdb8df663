// Prefill products (M > 8) on F16 / F32 weights: Y[m, n] = sum_k x[m, k] * w[n, k] on the matrix cores, both operands
// row-major with K contiguous (ggml's layout).
//
// ggml-cpu pairs F16 weights with activations rounded to fp16 (k_f16_act writes those rows once, into scratch) and F32
// weights with the activations as they are; products and sums are fp32, as the mat-vec on these types forms them:
// v_mfma_f32_32x32x16_f16 multiplies fp16 exactly, v_mfma_f32_16x16x4_f32 in fp32.
//
// A workgroup computes a BM x BN tile with KG * WGM * WGN waves. K advances in stages of KG slices of 128 bytes per row
// (64 halves, 32 floats); slice g of a stage belongs to the g-th group of WGM x WGN waves, so that with few tiles the
// waves of a tile share its K and their sums are added in group order at the end, in LDS (no second launch). Every wave
// copies its share of each stage into an NS-slot ring with buffer-to-LDS copies, NS - 1 stages ahead. Rows past M or N
// read as zeros (the descriptors end with the tile's last row); past K the fragments are zeroed in registers.
#include "mx_common.h"
#include "mx_device.h"

#include <algorithm>
#include <type_traits>

namespace mx {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int FG_ROW = 128;  // bytes of a row in one slice

struct FgProblem {
    const uint8_t *w;
    int64_t N;
    float *y;
    int64_t ldy;  // floats between consecutive m rows of y
};
// Up to four weights sharing the activations, or one weight (prob[0]) over batch slices. A slice's tiles are the grid's
// first dimension: split after split, problem after problem, the problem's tiles with n fastest; the slices are its second
// (the pass's and the reduce's third). Split s covers the stages [s per, (s + 1) per) and, with nsplit > 1, writes partial
// sums to ws ([slice][nsplit][M][ntot], problem p from column col0[p]), which k_fg_reduce adds in split order.
struct FgArgs {
    FgProblem prob[4];
    int nprob, nsplit;
    int64_t M, K;
    const uint8_t *x;
    int64_t x_nb;  // bytes between activation rows
    int64_t ntot, col0[4];
    float *ws;
    int batched;      // several slices (what follows is read only then)
    uint32_t z0, ne2, r2, r3;  // the launch's first slice; slices along axis 2, and to a matrix of the weight
    int64_t x_b2, x_b3, w_b2, w_b3, y_b2, y_b3;  // bytes between slices (the fp16 rows: x_b2, the launch's one after another)
};

// A launch's slice `rel` along the batch axes.
struct FgSlice {
    uint32_t i2, i3;
};
__device__ __forceinline__ uint32_t fg_uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ FgSlice fg_slice(const FgArgs &a, uint32_t rel) {
    const uint32_t z = a.z0 + rel, i3 = z / a.ne2;
    return FgSlice{fg_uniform(z - i3 * a.ne2), fg_uniform(i3)};
}

// x rows (f32) -> fp16 rows [M][K], round to nearest even, as ggml_cpu_fp32_to_fp16 makes src1 of F16 weights.
__global__ __launch_bounds__(256) void k_f16_act(const float *x, int64_t x_stride, int64_t K, uint16_t *xh, FgArgs a) {
    if (a.batched) {
        const FgSlice z = fg_slice(a, blockIdx.z);
        x = (const float *)((const uint8_t *)x + z.i2 * a.x_b2 + z.i3 * a.x_b3);
        xh += (int64_t)blockIdx.z * a.M * K;
    }
    const int64_t m = blockIdx.x, e = ((int64_t)blockIdx.y * 256 + threadIdx.x) * 8;
    if (e >= K) return;
    const float4 u = *(const float4 *)(x + m * x_stride + e), v = *(const float4 *)(x + m * x_stride + e + 4);
    v8h h = {(_Float16)u.x, (_Float16)u.y, (_Float16)u.z, (_Float16)u.w,
             (_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    *(v8h *)(xh + m * K + e) = h;
}

template <class T>
__device__ __forceinline__ T fg_pick(int i, T v0, T v1, T v2, T v3) {
    return i == 0 ? v0 : (i == 1 ? v1 : (i == 2 ? v2 : v3));
}

// 16-byte chunk c of row r lies at chunk c ^ fg_swz(r): eight consecutive rows of one fragment read fall on different
// banks, in rows of 128 bytes (two to a round of the banks) and of 256 (XF).
template <bool WIDE = false>
__device__ __forceinline__ int fg_swz(int r) {
    return (WIDE ? r : r >> 1) & 7;
}

// WT, the tile, the waves over M and N, the K groups, the ring's slots; XF: F16 weights whose activations are read as
// floats and rounded on the way from LDS to the matrix cores, by every wave that uses them (no pass before the product).
template <int WT_, int BM_, int BN_, int WGM_, int WGN_, int KG_, int NS_, bool XF_ = false>
struct FgCfg {
    static constexpr int WT = WT_, BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, KG = KG_, NS = NS_;
    static constexpr bool H = WT == MX_TYPE_F16, XF = XF_;
    static constexpr int NW = KG * WGM * WGN, WM = BM / WGM, WN = BN / WGN;
    static constexpr int T = H ? 32 : 16;  // rows and columns of one MFMA tile
    static constexpr int TM = WM / T, TN = WN / T, NR = H ? 16 : 4;  // tiles of a wave; registers of a tile
    static constexpr int ES = H ? 2 : 4, KS = FG_ROW / ES;           // weight element size, K per slice
    static constexpr int AROW = XF ? 2 * FG_ROW : FG_ROW;            // bytes of an activation row in a slice
    static constexpr int SA = BM * AROW, SB = BN * FG_ROW, SLICE = SA + SB, STAGE = KG * SLICE, LDS = NS * STAGE;
    // copies of 1 KB (64 lanes x 16 bytes) of a slice's activations and weights; per wave and stage
    static constexpr int CA = SA / 1024, CB = SB / 1024, OPS = KG * (CA + CB) / NW;
    // Sums of sums: see the kernel. Three levels where the accumulators are few.
    static constexpr bool MID = TM * TN * NR <= 32;
    static_assert(NW <= 8 && KG * (CA + CB) % NW == 0 && WM % T == 0 && WN % T == 0, "tile");
    static_assert(LDS <= 160 * 1024 && (NS == 2 || NS == 3), "LDS, and the waits of a stage");
    static_assert((KG - 1) * WGM * WGN * TM * TN * NR * 256 <= LDS, "the groups' sums fit the ring");
};

template <class C>
__global__ __launch_bounds__(64 * C::NW) void k_gemm_f(FgArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t lds = lds_addr(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t MT = (a.M + C::BM - 1) / C::BM;
    int64_t per = 0;  // tiles of one split
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (i < a.nprob) per += (a.prob[i].N + C::BN - 1) / C::BN * MT;
    int64_t t = blockIdx.x;
    const int split = (int)(t / per);
    t -= split * per;
    int pi = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const int64_t ti = (a.prob[i].N + C::BN - 1) / C::BN * MT;
        if (pi == i && i + 1 < a.nprob && t >= ti) {
            t -= ti;
            pi = i + 1;
        }
    }
    const uint8_t *w = fg_pick(pi, a.prob[0].w, a.prob[1].w, a.prob[2].w, a.prob[3].w), *x = a.x;
    const int64_t N = fg_pick(pi, a.prob[0].N, a.prob[1].N, a.prob[2].N, a.prob[3].N);
    FgSlice z = {0, 0};
    if (a.batched) {
        z = fg_slice(a, blockIdx.y);
        w += fg_uniform(z.i2 / a.r2) * a.w_b2 + fg_uniform(z.i3 / a.r3) * a.w_b3;
        x += C::H && !C::XF ? blockIdx.y * a.x_b2 : z.i2 * a.x_b2 + z.i3 * a.x_b3;
    }
    const int64_t ntp = (N + C::BN - 1) / C::BN;
    // (the divisions run on the vector unit: their uniform results go back to scalar registers for the copies' operands)
    const int mt = __builtin_amdgcn_readfirstlane((int)(t / ntp)), nt = __builtin_amdgcn_readfirstlane((int)(t % ntp));
    const int64_t m0 = (int64_t)mt * C::BM, n0 = (int64_t)nt * C::BN;
    const int nslice = (int)((a.K + C::KS - 1) / C::KS), nst_all = (nslice + C::KG - 1) / C::KG;
    const int sper = (nst_all + a.nsplit - 1) / a.nsplit;
    const int st0 = __builtin_amdgcn_readfirstlane(split * sper);
    const int nst = __builtin_amdgcn_readfirstlane(min(nst_all - split * sper, sper));

    // This wave's copies of a stage: copy q = wave OPS + j of the stage's KG x (CA + CB), each slice's activations first;
    // a weight copy is 8 rows of 128 bytes, an activation copy 8 rows of 128 or 4 of 256 bytes.
    const int64_t row_b = a.K * C::ES, row_a = C::XF || !C::H ? a.K * 4 : a.K * 2;
    const v4u ra = buf_rsrc(x + m0 * a.x_nb, (uint32_t)((min<int64_t>(C::BM, a.M - m0) - 1) * a.x_nb + row_a));
    const v4u rb = buf_rsrc(w + n0 * row_b, (uint32_t)(min<int64_t>(C::BN, N - n0) * row_b));
    uint32_t voff[C::OPS];
#pragma unroll
    for (int j = 0; j < C::OPS; j++) {
        const int q = wave * C::OPS + j, gq = q / (C::CA + C::CB), c = q % (C::CA + C::CB);
        constexpr int LA = C::AROW / 16;  // lanes to an activation row
        if (c < C::CA) {                  // (uniform)
            const int r = (64 / LA) * c + lane / LA;
            voff[j] = (uint32_t)r * (uint32_t)a.x_nb + (uint32_t)(gq * C::AROW) + 16u * (uint32_t)((lane % LA) ^ fg_swz<C::XF>(r));
        } else {
            const int r = 8 * (c - C::CA) + (lane >> 3);
            voff[j] = (uint32_t)r * (uint32_t)row_b + (uint32_t)(gq * FG_ROW) + 16u * (uint32_t)((lane & 7) ^ fg_swz(r));
        }
    }
    auto issue = [&](int slot, int st) __attribute__((always_inline)) {  // stage st (of the whole K) into a slot
#pragma unroll
        for (int j = 0; j < C::OPS; j++) {
            const int q = wave * C::OPS + j;
            const bool isa = q % (C::CA + C::CB) < C::CA;
            const v4u rs = isa ? ra : rb;
            const uint32_t step = isa ? C::KG * C::AROW : C::KG * FG_ROW;
            dma16_lds(rs, lds + (uint32_t)(slot * C::STAGE + q * 1024), voff[j], (uint32_t)st * step);
        }
    };
#pragma unroll
    for (int s = 0; s < C::NS - 1; s++)
        if (s < nst) issue(s, st0 + s);

    const int g = wave / (C::WGM * C::WGN), wq = wave % (C::WGM * C::WGN);
    const int wm = (wq / C::WGN) * C::WM, wn = (wq % C::WGN) * C::WN;
    // fragments: F16 lane l: row l % 32, chunk 2 kb + l / 32 (8 halves); F32 lane l: row l % 16, chunk 4 kb + l / 16 (4
    // floats, one to each of four MFMAs: both operands take k in the same permuted order)
    constexpr int NK = C::H ? 4 : 2;  // fragment steps of a slice
    const int fr = lane % C::T, fh = lane / C::T;
    uint32_t aoff[C::TM][NK], boff[C::TN][NK];
#pragma unroll
    for (int kb = 0; kb < NK; kb++) {
        const int c = (C::H ? 2 : 4) * kb + fh;
#pragma unroll
        for (int i = 0; i < C::TM; i++) {
            const int r = wm + C::T * i + fr;
            aoff[i][kb] = (uint32_t)(g * C::SLICE + r * C::AROW + 16 * ((C::XF ? 2 * c : c) ^ fg_swz<C::XF>(r)));
        }
#pragma unroll
        for (int j = 0; j < C::TN; j++) {
            const int r = wn + C::T * j + fr;
            boff[j][kb] = (uint32_t)(g * C::SLICE + C::SA + r * FG_ROW + 16 * (c ^ fg_swz(r)));
        }
    }
    // One running fp32 sum over K would round once per MFMA; the error of a chain of n additions grows as its square
    // root, so the sums are formed in two or three levels (n = a b c additions as chains of a, b and c): two slices of
    // MFMAs, the sums of those, and the sums of four of those where registers allow. Relative to the sum in double
    // precision, K = 2048 / 6144: one chain 2.9e-7 / 5.0e-7; two levels 1.1e-7 / 1.5e-7; three 9.6e-8 / 1.1e-7; the
    // mat-vec's order 1.2e-7 / 1.8e-7.
    constexpr int NR = C::NR, NA = C::H ? 1 : 4;  // NA: F32's four MFMAs of a chunk sum apart
    typedef typename std::conditional<C::H, v16f, v4f>::type acc_t;
    acc_t acc[NA][C::TM][C::TN], mid[C::TM][C::TN], top[C::TM][C::TN];
    acc_t zero;
#pragma unroll
    for (int r = 0; r < NR; r++) zero[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < C::TM; i++)
#pragma unroll
        for (int j = 0; j < C::TN; j++) mid[i][j] = top[i][j] = zero;

    // stage s into the inner sums, started anew when `first`
    auto stage = [&](int s, auto first_c) __attribute__((always_inline)) {
        constexpr bool first = decltype(first_c)::value;
        // this wave's copies of stage s have landed, then every wave's, and every wave has read the slot that the next
        // copies overwrite (the bare barrier: __syncthreads would wait for the copies in flight too)
        const int rem = nst - 1 - s;
        if (rem >= C::NS - 2) wait_vm<(C::NS - 2) * C::OPS>();
        else wait_vm<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + C::NS - 1 < nst) issue((s + C::NS - 1) % C::NS, st0 + s + C::NS - 1);
        const int k0 = ((st0 + s) * C::KG + g) * C::KS;  // this group's slice
        if (k0 >= a.K) {                                 // wave-uniform: the last stage may lack slices
            if (first)
#pragma unroll
                for (int e = 0; e < NA; e++)
#pragma unroll
                    for (int i = 0; i < C::TM; i++)
#pragma unroll
                        for (int j = 0; j < C::TN; j++) acc[e][i][j] = zero;
            return;
        }
        const uint8_t *sl = smem + (s % C::NS) * C::STAGE;
        v4f af[NK][C::TM], bf[NK][C::TN];
#pragma unroll
        for (int kb = 0; kb < NK; kb++) {
#pragma unroll
            for (int i = 0; i < C::TM; i++) {
                if constexpr (C::XF) {  // chunks 2 c and 2 c + 1 (the swizzle leaves bit 0 of an even chunk's pair apart)
                    const v4f u = *(const v4f *)(sl + aoff[i][kb]), v = *(const v4f *)(sl + (aoff[i][kb] ^ 16u));
                    const v8h h = {(_Float16)u[0], (_Float16)u[1], (_Float16)u[2], (_Float16)u[3],
                                   (_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                    af[kb][i] = __builtin_bit_cast(v4f, h);
                } else {
                    af[kb][i] = *(const v4f *)(sl + aoff[i][kb]);
                }
            }
#pragma unroll
            for (int j = 0; j < C::TN; j++) bf[kb][j] = *(const v4f *)(sl + boff[j][kb]);
        }
        if (k0 + C::KS > a.K) {  // uniform: the tail of K; chunks past it hold the next row's bytes
            const v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < NK; kb++) {
                const bool in = k0 + ((C::H ? 2 : 4) * kb + fh) * (16 / C::ES) < a.K;
#pragma unroll
                for (int i = 0; i < C::TM; i++) af[kb][i] = in ? af[kb][i] : z;
#pragma unroll
                for (int j = 0; j < C::TN; j++) bf[kb][j] = in ? bf[kb][j] : z;
            }
        }
#pragma unroll
        for (int kb = 0; kb < NK; kb++) {
            if constexpr (C::H) {
#pragma unroll
                for (int i = 0; i < C::TM; i++)
#pragma unroll
                    for (int j = 0; j < C::TN; j++)
                        acc[0][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(v8h, af[kb][i]), __builtin_bit_cast(v8h, bf[kb][j]),
                            first && kb == 0 ? zero : acc[0][i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int i = 0; i < C::TM; i++)
#pragma unroll
                        for (int j = 0; j < C::TN; j++)
                            acc[e][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                af[kb][i][e], bf[kb][j][e], first && kb == 0 ? zero : acc[e][i][j], 0, 0, 0);
            }
        }
    };
    int flushes = 0;
    for (int s = 0; s < nst; s += 2) {
        stage(s, std::true_type{});
        if (s + 1 < nst) stage(s + 1, std::false_type{});
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int j = 0; j < C::TN; j++)
#pragma unroll
                for (int r = 0; r < NR; r++)
                    mid[i][j][r] += C::H ? acc[0][i][j][r]
                                         : (acc[0][i][j][r] + acc[NA > 1 ? 1 : 0][i][j][r]) +
                                               (acc[NA > 1 ? 2 : 0][i][j][r] + acc[NA > 1 ? 3 : 0][i][j][r]);
        if (C::MID && (++flushes & 3) == 0) {
#pragma unroll
            for (int i = 0; i < C::TM; i++)
#pragma unroll
                for (int j = 0; j < C::TN; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++) {
                        top[i][j][r] += mid[i][j][r];
                        mid[i][j][r] = 0.0f;
                    }
        }
    }
    if (C::MID)
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int j = 0; j < C::TN; j++)
#pragma unroll
                for (int r = 0; r < NR; r++) mid[i][j][r] += top[i][j][r];

    if constexpr (C::KG > 1) {  // groups 1 .. leave their sums in LDS, group 0 adds them in group order
        __syncthreads();        // (also: no copy is in flight, every wave is done with the ring)
        constexpr int GW = C::WGM * C::WGN, WB = C::TM * C::TN * NR * 64;  // floats per wave
        float *part = (float *)smem;
        if (g > 0) {
#pragma unroll
            for (int i = 0; i < C::TM; i++)
#pragma unroll
                for (int j = 0; j < C::TN; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++)
                        part[((g - 1) * GW + wq) * WB + ((i * C::TN + j) * NR + r) * 64 + lane] = mid[i][j][r];
        }
        __syncthreads();
        if (g > 0) return;
#pragma unroll
        for (int gg = 0; gg < C::KG - 1; gg++)
#pragma unroll
            for (int i = 0; i < C::TM; i++)
#pragma unroll
                for (int j = 0; j < C::TN; j++)
#pragma unroll
                    for (int r = 0; r < NR; r++)
                        mid[i][j][r] += part[(gg * GW + wq) * WB + ((i * C::TN + j) * NR + r) * 64 + lane];
    }

    float *y = fg_pick(pi, a.prob[0].y, a.prob[1].y, a.prob[2].y, a.prob[3].y);
    int64_t ldy = fg_pick(pi, a.prob[0].ldy, a.prob[1].ldy, a.prob[2].ldy, a.prob[3].ldy);
    if (a.nsplit > 1) {  // this split's partial sums
        y = a.ws + ((int64_t)blockIdx.y * a.nsplit + split) * a.M * a.ntot + fg_pick(pi, a.col0[0], a.col0[1], a.col0[2], a.col0[3]);
        ldy = a.ntot;
    } else if (a.batched) {
        y = (float *)((uint8_t *)y + z.i2 * a.y_b2 + z.i3 * a.y_b3);
    }
    // accumulators: 32 x 32 lane l, register r: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32; 16 x 16: row
    // 4 (l / 16) + r, column l % 16
#pragma unroll
    for (int i = 0; i < C::TM; i++)
#pragma unroll
        for (int j = 0; j < C::TN; j++) {
            const int64_t n = n0 + wn + C::T * j + fr;
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const int64_t m = m0 + wm + C::T * i + (C::H ? 8 * (r >> 2) + 4 * fh + (r & 3) : 4 * fh + r);
                if (m < a.M) y[m * ldy + n] = mid[i][j][r];
            }
        }
}

// y[m][col] = the nsplit partials of (m, col) added in split order; one thread per column.
__global__ __launch_bounds__(256) void k_fg_reduce(FgArgs a) {
    const int64_t m = blockIdx.x, c = (int64_t)blockIdx.y * 256 + threadIdx.x;
    if (c >= a.ntot) return;
    const int64_t plane = a.M * a.ntot;
    const float *ws = a.ws + (int64_t)blockIdx.z * a.nsplit * plane + m * a.ntot + c;
    float sum = ws[0];
    for (int s = 1; s < a.nsplit; s++) sum += ws[s * plane];
    int pi = 0;
#pragma unroll
    for (int i = 1; i < 4; i++) pi += i < a.nprob && c >= a.col0[i];
    float *y = fg_pick(pi, a.prob[0].y, a.prob[1].y, a.prob[2].y, a.prob[3].y);
    if (a.batched) {
        const FgSlice z = fg_slice(a, blockIdx.z);
        y = (float *)((uint8_t *)y + z.i2 * a.y_b2 + z.i3 * a.y_b3);
    }
    const int64_t ldy = fg_pick(pi, a.prob[0].ldy, a.prob[1].ldy, a.prob[2].ldy, a.prob[3].ldy);
    y[m * ldy + (c - fg_pick(pi, a.col0[0], a.col0[1], a.col0[2], a.col0[3]))] = sum;
}

// ------------------------------------------------------------------------------------------------------------------
// Host side.
// ------------------------------------------------------------------------------------------------------------------
namespace {
struct FgPlan {
    int tile = 0, bm = 0, bn = 0, nsplit = 1;
    bool pass = false;  // F16: the activations are rounded to fp16 rows in scratch first
    int64_t ntot = 0, grid = 0, rows = 0, slices = 0;  // of one launch: workgroups per slice, rows, slices
};

// Tiles (BM x BN, K groups) and K splits over workgroups, by the tiles the product has. Measured on MI355X with weights
// in the caches (us, pass and reduce included):
//   F16, N = 12288, K = 2048: M = 512 on 128 x 128 39.6, 64 x 128 49.7; M = 133 64 x 128 24.7, 64 x 64 28.4; M = 33
//     64 x 64 16.3, 64 x 128 20.8; M = 28 32 x 64 13.2, 64 x 64 16.3, 32 x 32 18.5
//   F16, N = 2048, K = 2048: M = 512 64 x 64 18.9, 32 x 64 22.2, 128 x 128 30.0; M = 133 32 x 64 11.2, 64 x 64 15.0;
//     M = 64 32 x 32 9.4, 32 x 64 11.1; splitting K there gains nothing (M = 512 in two 21.5)
//   F16, N = 2048, K = 6144: M = 512 64 x 64 in two splits 34.4, in one 39.6; M = 133 64 x 64 in four 20.1, 32 x 64 in
//     one 25.7; M = 28 32 x 32 in four 12.1, in one 20.1
//   F32, K = 2048, N = 64, M = 256: 16 x 16 7.4, 32 x 32 18.8; K = 3008, N = 1200, M = 396: 32 x 32 40.8, 16 x 16 70.0
//     (16 x 16: 98 KB, one workgroup per CU, eight waves that share K in stages of 256). Where K is one stage, a second round
//     of them costs more than the larger tile: K = 128, N = 512, 16 slices of M = 9 7.6, 32 x 32 5.2
// The mat-vec that these products ran on before takes 8 columns (fewer for K > 2048) at a time: F16 512 x 12288 x 2048
// 2,604 us, F32 256 x 64 x 2048 356 us.
// Batch slices share a launch, and their tiles count together. A launch for each slice against one for all, and the
// mat-vec, which takes every slice of eight columns: F16, N = 512, K = 128: 16 slices of M = 9 64.8 / 5.6 / 6.9 us, 256 of
// M = 64 1,236 / 31.5 / 201; F32, N = 64, K = 2048, 256 slices of M = 16 2,067 / 48.2 / 202.
FgPlan fg_plan_rows(const GemmFArgs &g, int64_t M) {
    FgPlan pl;
    const int type = g.type;
    const int64_t K = g.K;
    for (int i = 0; i < g.nprob; i++) pl.ntot += g.N[i];
    auto tiles = [&](int bm, int bn) {  // of every slice
        int64_t t = 0;
        for (int i = 0; i < g.nprob; i++) t += (g.N[i] + bn - 1) / bn;
        return t * ((M + bm - 1) / bm) * g.nbatch;
    };
    static constexpr int T16[][3] = {{128, 128, 1}, {64, 128, 1}, {64, 64, 2}, {32, 64, 4}, {32, 32, 4}};
    static constexpr int T32[][3] = {{32, 32, 2}, {16, 16, 8}};
    int64_t want = 1;
    if (type == MX_TYPE_F16) {
        const int64_t t64 = tiles(64, 64), long_k = K >= 4096;
        if (M <= 32) pl.tile = tiles(32, 64) >= 128 ? 3 : 4;
        else if (tiles(128, 128) >= 256) pl.tile = 0;
        else if (long_k && t64 <= 256) pl.tile = 2;
        else if (tiles(64, 128) >= 256) pl.tile = 1;
        else if (t64 >= 192) pl.tile = 2;
        else pl.tile = tiles(32, 64) >= 128 ? 3 : 4;
        const int64_t t32 = tiles(32, 32);
        if (pl.tile == 2 && long_k && t64 > 0) want = std::min<int64_t>(4, 512 / t64);
        if (pl.tile == 4 && t32 > 0 && t32 <= 128) want = std::min<int64_t>(256 / t32, K / 1536);
    } else {
        pl.tile = tiles(16, 16) <= (K > 256 ? 512 : 256);
    }
    const auto &t = type == MX_TYPE_F16 ? T16[pl.tile] : T32[pl.tile];
    pl.bm = t[0];
    pl.bn = t[1];
    pl.pass = type == MX_TYPE_F16 && pl.tile < 3;
    const int64_t ks = t[2] * (type == MX_TYPE_F16 ? 64 : 32), nst = (K + ks - 1) / ks;  // stages
    want = std::max<int64_t>(1, std::min(want, nst));
    const int64_t per = (nst + want - 1) / want;  // stages of a split; none is left empty
    pl.nsplit = (int)((nst + per - 1) / per);
    pl.grid = tiles(pl.bm, pl.bn) / g.nbatch * pl.nsplit;
    pl.rows = M;
    return pl;
}

// Bytes of scratch for `slices` slices of a launch: the fp16 rows, and the partial sums.
size_t fg_act_bytes(const FgPlan &pl, int64_t K, int64_t slices) {
    return pl.pass ? ((size_t)slices * (size_t)pl.rows * (size_t)K * 2 + 255) / 256 * 256 : 0;
}
size_t fg_bytes(const FgPlan &pl, int64_t K, int64_t slices) {
    return fg_act_bytes(pl, K, slices) +
           (pl.nsplit > 1 ? (size_t)slices * (size_t)pl.nsplit * (size_t)pl.rows * (size_t)pl.ntot * 4 : 0);
}

// ... with the rows and the slices of one launch: a grid dimension of fewer than 2^32 threads (HIP's limit; the pass and
// the reduce have 256 a row), and scratch for as many slices as stay within 64 MB. grid = 0: no launch can have it.
FgPlan fg_plan(const GemmFArgs &g) {
    constexpr int64_t ROWS = (int64_t)1 << 22, THREADS = (int64_t)1 << 32, WG = 512, WORK = (int64_t)64 << 20;
    FgPlan pl = fg_plan_rows(g, std::min(g.M, ROWS));
    while (pl.grid * WG >= THREADS && pl.rows > 32) pl = fg_plan_rows(g, (pl.rows / 2 + 31) / 32 * 32);
    if (pl.grid * WG >= THREADS) pl.grid = 0;
    const size_t one = fg_bytes(pl, g.K, 1);
    pl.slices = one ? std::max<int64_t>(1, std::min<int64_t>(g.nbatch, WORK / (int64_t)one)) : g.nbatch;
    return pl;
}

template <class C>
hipError_t fg_launch(int64_t grid, unsigned slices, const FgArgs &a, hipStream_t s) {
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)k_gemm_f<C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(k_gemm_f<C>, dim3((unsigned)grid, slices), dim3(64 * C::NW), C::LDS, s, a);
    return hipGetLastError();
}

// The rows m0 .. m0 + M (at most pl.rows) of the slices z0 .. z0 + slices.
hipError_t fg_run(const GemmFArgs &g, const FgPlan &pl, int64_t m0, int64_t M, int64_t z0, unsigned slices,
                  void *scratch, hipStream_t s) {
    FgArgs a{};
    int64_t tiles = 0;
    for (int i = 0; i < g.nprob; i++) {
        a.prob[i] = FgProblem{(const uint8_t *)g.w[i], g.N[i], g.y[i] + m0 * g.ldy[i], g.ldy[i]};
        a.col0[i] = i == 0 ? 0 : a.col0[i - 1] + g.N[i - 1];
        tiles += (g.N[i] + pl.bn - 1) / pl.bn;
    }
    tiles *= (M + pl.bm - 1) / pl.bm;
    if (tiles == 0) return hipSuccess;
    a.nprob = g.nprob;
    a.nsplit = pl.nsplit;
    a.M = M;
    a.K = g.K;
    a.x = (const uint8_t *)g.x + m0 * g.x_nb;
    a.x_nb = g.x_nb;
    a.ntot = pl.ntot;
    a.ws = (float *)((uint8_t *)scratch + fg_act_bytes(pl, g.K, slices));
    if (g.nbatch > 1) {
        a.batched = 1;
        a.z0 = (uint32_t)z0;
        a.ne2 = (uint32_t)g.ne2;
        a.r2 = (uint32_t)g.r2;
        a.r3 = (uint32_t)g.r3;
        a.x_b2 = g.x_b2;
        a.x_b3 = g.x_b3;
        a.w_b2 = g.w_b2;
        a.w_b3 = g.w_b3;
        a.y_b2 = g.y_b2;
        a.y_b3 = g.y_b3;
    }
    if (pl.pass) {
        hipLaunchKernelGGL(k_f16_act, dim3((unsigned)M, (unsigned)((g.K + 2047) / 2048), slices), dim3(256), 0, s,
                           (const float *)a.x, g.x_nb / 4, g.K, (uint16_t *)scratch, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        a.x = (const uint8_t *)scratch;
        a.x_nb = 2 * g.K;
        a.x_b2 = 2 * g.K * M;
    }
    const int64_t grid = tiles * pl.nsplit;
    hipError_t e;
    if (g.type == MX_TYPE_F16) {
        switch (pl.tile) {
            case 0: e = fg_launch<FgCfg<MX_TYPE_F16, 128, 128, 2, 2, 1, 2>>(grid, slices, a, s); break;
            case 1: e = fg_launch<FgCfg<MX_TYPE_F16, 64, 128, 2, 2, 1, 3>>(grid, slices, a, s); break;
            case 2: e = fg_launch<FgCfg<MX_TYPE_F16, 64, 64, 2, 2, 2, 2>>(grid, slices, a, s); break;
            case 3: e = fg_launch<FgCfg<MX_TYPE_F16, 32, 64, 1, 2, 4, 2, true>>(grid, slices, a, s); break;
            default: e = fg_launch<FgCfg<MX_TYPE_F16, 32, 32, 1, 1, 4, 3, true>>(grid, slices, a, s); break;
        }
    } else {
        e = pl.tile == 0 ? fg_launch<FgCfg<MX_TYPE_F32, 32, 32, 2, 2, 2, 3>>(grid, slices, a, s)
                         : fg_launch<FgCfg<MX_TYPE_F32, 16, 16, 1, 1, 8, 3>>(grid, slices, a, s);
    }
    if (e != hipSuccess || pl.nsplit == 1) return e;
    hipLaunchKernelGGL(k_fg_reduce, dim3((unsigned)M, (unsigned)((pl.ntot + 255) / 256), slices), dim3(256), 0, s, a);
    return hipGetLastError();
}
}  // namespace

bool gemm_f_supported(const GemmFArgs &g) {
    if ((g.type != MX_TYPE_F16 && g.type != MX_TYPE_F32) || (g.nprob > 1 && g.nbatch > 1)) return false;
    // a tile's rows within the descriptors' 32-bit offsets
    if (g.x_nb < 0 || g.x_nb >= ((int64_t)1 << 24) || g.K >= ((int64_t)1 << 22) || g.M >= ((int64_t)1 << 31)) return false;
    const FgPlan pl = fg_plan(g);
    return pl.grid > 0 && (pl.nsplit == 1 || pl.ntot <= 256 * 65535);
}

size_t gemm_f_scratch_bytes(const GemmFArgs &g) {
    const FgPlan pl = fg_plan(g);
    return fg_bytes(pl, g.K, pl.slices);
}

hipError_t launch_gemm_f(const GemmFArgs &g, void *scratch, hipStream_t s) {
    const FgPlan pl = fg_plan(g);
    for (int64_t z0 = 0; z0 < g.nbatch; z0 += pl.slices)
        for (int64_t m0 = 0; m0 < g.M; m0 += pl.rows) {
            const hipError_t e = fg_run(g, pl, m0, std::min(pl.rows, g.M - m0), z0,
                                        (unsigned)std::min(pl.slices, g.nbatch - z0), scratch, s);
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

}  // namespace mx
