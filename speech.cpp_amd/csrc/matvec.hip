// Small-M quantized products (decode M = 1, draft verification M <= 5): y[n, m] = W[n, :] . quant(x[:, m]).
//
// One launch does everything: the workgroup first quantizes its NC activation columns into LDS (the ggml CPU src1
// conversion, bit for bit), then streams weight rows with 16-byte loads from the planar layout and reduces each row
// over LPR lanes. HBM-bound by design: each weight byte is read once per launch.
#include "mx_common.h"
#include "mx_device.h"
#include "mx_dot.h"

#include <algorithm>
#include <cstdlib>

namespace mx {

__device__ __forceinline__ MatvecProblem pick_problem(const MatvecArgs &a, int i) {
    // Uniform selection keeps the kernel-argument struct out of private memory.
    return i == 0 ? a.prob[0] : (i == 1 ? a.prob[1] : (i == 2 ? a.prob[2] : a.prob[3]));
}

// The two shapes of a workgroup. Narrow: four waves, one set of rows. Wide, from two columns on: eight waves (Q5_K four: its
// dots take more registers than eight waves leave) that go on to further rows with the columns they have quantized, which
// every workgroup does for itself. Wide costs registers, so where the columns are soon quantized narrow is faster; mv_wide
// picks, mv_narrow says which narrow kernels there are.
template <int TYPE, bool WIDE>
__host__ __device__ constexpr int mv_waves() { return WIDE && TYPE != MX_TYPE_Q5_K ? 8 : 4; }
template <int TYPE, int NC, bool FUSED>
constexpr bool mv_narrow() {
    return NC == 1 || (TYPE == MX_TYPE_Q5_K && NC <= 4) || ((TYPE == MX_TYPE_Q4_K || TYPE == MX_TYPE_Q6_K) && (!FUSED || NC <= 5));
}
// The elements of a column that a workgroup handles at once (a PIECE) are 256 a wave, a float4 a thread. Every thread
// loads the first XPRE float4s of each column (elements PIECE i + 4 tid) ahead of the weights.
template <int NC>
__host__ __device__ constexpr int xpre() { return NC == 1 ? 4 : (NC == 2 ? 2 : 1); }

// Quantizes one piece, at `base`, of one activation column (v = elements base + 4 tid .. + 3) into LDS:
// Q8_0 weights take 32-blocks (d rounded to fp16 and back, as the CPU dot reads it), K-quants Q8_K 256-blocks with
// their 16-element sums (Q4_K: quants in unit order and sums of 32, as its dot reads them). Every wave of the
// workgroup calls it with the same `base`.
template <int TYPE>
__device__ __forceinline__ void quantize_piece(float4 v, int base, int K, int rounding, int8_t *xq, float *xd,
                                               int *xbs) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int e = base + 4 * tid;
    if constexpr (TYPE == MX_TYPE_Q8_0) {
        float d;
        int sum;
        const int q = quant32_lane(v, rounding, &d, &sum);
        if (e < K) {  // K % 32 == 0: the eight lanes of a block agree
            *(int *)(xq + e) = q;
            if ((tid & 7) == 0) xd[e / 32] = h2f(f2h(d));
        }
    } else {
        if (base + 256 * (tid >> 6) < K) {  // a whole wave per super-block
            float d;
            int bs;
            const int q = quant256_wave(v, lane, &d, &bs);
            if (lane == 0) xd[e / 256] = d;
            if constexpr (TYPE == MX_TYPE_Q4_K) {  // unit order, and sums of 32
                *(int *)(xq + q4u_xq_offset(e, K)) = q;
                const int bs32 = bs + dpp_i<dpp::HALF_MIRROR>(0, bs);  // lanes 8j..8j+7: quants 32j..32j+31
                if ((lane & 7) == 0) xbs[e / 32] = bs32;
            } else {
                *(int *)(xq + e) = q;
                if ((lane & 3) == 0) xbs[e / 16] = bs;
            }
        }
    }
}

__device__ __forceinline__ float4 load_x4(const float *xc, int e, int K) {
    const float4 v = *(const float4 *)(xc + (e < K ? e : K - 4));
    return e < K ? v : make_float4(0.f, 0.f, 0.f, 0.f);
}

// The fused prologue: each column x becomes silu(x) * glu_b (ggml_vec_swiglu_f32's scalar form) when glu_b is set,
// then mul(rms_norm(x, eps), norm_w) when norm_w is set -- the squares (rounded to float) summed in double over the
// workgroup, the mean rounded to float, x * (1 / sqrtf(mean + eps)) then times the weight, as the separate ops round
// -- and is quantized. Pieces past the preloaded ones are read again after the sum.
template <int TYPE, int NC, int NW>
__device__ __forceinline__ void fused_prologue(const MatvecArgs &a, const float *x, int xi12, int i13,
                                               float4 (&xr)[NC][xpre<NC>()], const float4 (&br)[NC][xpre<NC>()],
                                               const float4 (&wr)[xpre<NC>()], int8_t *xq, float *xd, int *xbs) {
    constexpr int XP = xpre<NC>();
    constexpr int PIECE = 256 * NW;
    constexpr int XDB = TYPE == MX_TYPE_Q8_0 ? 32 : 256;
    const int K = (int)a.K;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ double red[NC][NW];
    const float *gb = a.glu_b ? a.glu_b + xi12 * a.x_b2 + i13 * a.x_b3 : nullptr;
    // glu of one loaded piece; the preloaded pieces' second operands came in with x (br)
    auto piece_b = [&](float4 v, float4 b) -> float4 {
        v.x = v.x / (1.0f + expf(-v.x)) * b.x;
        v.y = v.y / (1.0f + expf(-v.y)) * b.y;
        v.z = v.z / (1.0f + expf(-v.z)) * b.z;
        v.w = v.w / (1.0f + expf(-v.w)) * b.w;
        return v;
    };
    // Every column's elements of the piece at `base`, past the preloaded ones: all of their loads go out before
    // the first is used. (Column after column, a product of several columns waited for K / PIECE - 1 loads of each in a
    // row.)
    auto piece = [&](int base, float4 (&v)[NC]) {
#pragma unroll
        for (int c = 0; c < NC; c++) v[c] = load_x4(x + c * a.x_col_stride, base + 4 * tid, K);
        if (gb) {
            float4 b[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) b[c] = load_x4(gb + c * a.x_col_stride, base + 4 * tid, K);
#pragma unroll
            for (int c = 0; c < NC; c++) v[c] = piece_b(v[c], b[c]);
        }
    };
    if (gb) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < XP; i++) xr[c][i] = piece_b(xr[c][i], br[c][i]);
    }
    float scale[NC];
    if (a.norm_w) {
        auto square = [](float4 v) {
            return (double)(v.x * v.x) + (double)(v.y * v.y) + (double)(v.z * v.z) + (double)(v.w * v.w);
        };
        double ss[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            ss[c] = 0.0;
#pragma unroll
            for (int i = 0; i < XP; i++) ss[c] += square(xr[c][i]);  // zero past K
        }
        for (int base = PIECE * XP; base < K; base += PIECE) {
            float4 v[NC];
            piece(base, v);
#pragma unroll
            for (int c = 0; c < NC; c++) ss[c] += square(v[c]);
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
            ss[c] = wave_sum_d(ss[c]);
            if (lane == 0) red[c][wave] = ss[c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NC; c++) {
            double tot = red[c][0];
#pragma unroll
            for (int w = 1; w < NW; w++) tot += red[c][w];
            const float mean = (float)(tot / (double)K);
            scale[c] = 1.0f / sqrtf(mean + a.norm_eps);
        }
    }
    auto normed = [&](int c, int base, int i, float4 v) -> float4 {  // i: the preloaded piece, or -1
        if (a.norm_w) {
            const float4 w = i >= 0 ? wr[i] : load_x4(a.norm_w, base + 4 * tid, K);
            v.x = (v.x * scale[c]) * w.x;
            v.y = (v.y * scale[c]) * w.y;
            v.z = (v.z * scale[c]) * w.z;
            v.w = (v.w * scale[c]) * w.w;
        }
        return v;
    };
    auto quantize = [&](int c, int base, int i, float4 v) {
        quantize_piece<TYPE>(normed(c, base, i, v), base, K, a.rounding, xq + c * K, xd + c * (K / XDB),
                             xbs + c * xbs_per_col<TYPE>(K));
    };
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < XP; i++)
            if (PIECE * i < K) quantize(c, PIECE * i, i, xr[c][i]);
    for (int base = PIECE * XP; base < K; base += PIECE) {
        float4 v[NC];
        piece(base, v);
#pragma unroll
        for (int c = 0; c < NC; c++) quantize(c, base, -1, v[c]);
    }
}

// The plain prologue: every column quantized into LDS, the preloaded pieces first, the others piece by piece with all
// columns' loads in flight.
template <int TYPE, int NC, int NW>
__device__ __forceinline__ void plain_prologue(const MatvecArgs &a, const float *x, const float4 (&xr)[NC][xpre<NC>()],
                                               int8_t *xq, float *xd, int *xbs) {
    constexpr int XP = xpre<NC>();
    constexpr int PIECE = 256 * NW;
    constexpr int XDB = TYPE == MX_TYPE_Q8_0 ? 32 : 256;
    const int K = (int)a.K;
    auto quantize = [&](int c, int base, float4 v) {
        quantize_piece<TYPE>(v, base, K, a.rounding, xq + c * K, xd + c * (K / XDB), xbs + c * xbs_per_col<TYPE>(K));
    };
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < XP; i++)
            if (PIECE * i < K) quantize(c, PIECE * i, xr[c][i]);
    for (int base = PIECE * XP; base < K; base += PIECE) {
        float4 v[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) v[c] = load_x4(x + c * a.x_col_stride, base + 4 * (int)threadIdx.x, K);
#pragma unroll
        for (int c = 0; c < NC; c++) quantize(c, base, v[c]);
    }
}

// FUSED: the instantiation that reads the fused operands (norm weight, SwiGLU input, residual); the plain one is
// compiled without them, so products with no fusion keep their smaller register footprint.
template <int TYPE, int NC, int LPR, bool FUSED, bool WIDE>
__global__ __launch_bounds__((64 * mv_waves<TYPE, WIDE>())) void k_matvec(MatvecArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int NW = mv_waves<TYPE, WIDE>();
    const int K = (int)a.K;
    const int tid = threadIdx.x;
    // The argument block's fields on the way to the first weight load, requested together into scalar registers:
    // left to the compiler, the branches below would each wait on a scalar load of their own, several round trips in
    // a row before the weights could be requested.
    const MatvecProblem p = pick_problem(a, (int)blockIdx.y);
    {
        const int nbatch = a.nbatch, rounding = a.rounding;
        const int32_t *ids = a.ids;
        const float *xa = a.x;
        const int64_t xcs = a.x_col_stride;
        asm volatile("" ::"s"(nbatch), "s"(rounding), "s"(ids), "s"(xa), "s"(xcs), "s"(a.K), "s"(a.x_b2), "s"(a.x_b3),
                     "s"(p.w.p0), "s"(p.w.p1), "s"(p.N), "s"(p.row0));
        if constexpr (TYPE != MX_TYPE_Q8_0) asm volatile("" ::"s"(p.w.p2));
        if constexpr (TYPE == MX_TYPE_Q5_K || TYPE == MX_TYPE_Q6_K) asm volatile("" ::"s"(p.w.p3));
        if constexpr (FUSED) asm volatile("" ::"s"(a.glu_b), "s"(a.norm_w), "s"(p.res));
    }
    // a narrower problem of a group: the grid is the widest one's
    if ((int64_t)blockIdx.x * (NW * (64 / LPR)) >= p.N) return;
    // Batch slice; a single slice (decode) takes no division.
    int i12 = 0, i13 = 0, mat = 0;
    if (a.nbatch > 1) {
        const unsigned z = blockIdx.z;
        i12 = (int)(z % (unsigned)a.ne12);
        i13 = (int)(z / (unsigned)a.ne12);
        mat = (int)((unsigned)i12 / (unsigned)a.r2) + (int)((unsigned)i13 / (unsigned)a.r3) * a.ne02;
    }
    int xi12 = i12;
    if (a.ids) {  // routed expert: the slice's matrix comes from ids (uniform over the workgroup)
        mat = *(const int32_t *)((const uint8_t *)a.ids + i12 * a.ids_nb0 + i13 * a.ids_nb1);
        if (mat < 0 || mat >= a.n_mats) {  // ggml-cpu asserts; this pair's output is left as it was and reported
            if (tid == 0) atomicOr(a.err, 2);
            return;
        }
        xi12 = (int)((unsigned)i12 % (unsigned)a.x_ne12);
    }
    const float *x = a.x + xi12 * a.x_b2 + i13 * a.x_b3;

    // The activation loads go first: x -> quantization -> LDS is the prologue's critical path, and the memory counter
    // retires loads in order, so waiting for x then does not wait for the weight loads issued after it.
    constexpr int XP = xpre<NC>();
    constexpr int PIECE = 256 * NW;
    float4 xr[NC][XP];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < XP; i++) xr[c][i] = load_x4(x + c * a.x_col_stride, PIECE * i + 4 * tid, K);
    // the fused prologue's other operands come in with x: SwiGLU's second input and the norm weight
    float4 br[NC][XP], wr[XP];
    if (FUSED && a.glu_b) {
        const float *gb = a.glu_b + xi12 * a.x_b2 + i13 * a.x_b3;
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < XP; i++) br[c][i] = load_x4(gb + c * a.x_col_stride, PIECE * i + 4 * tid, K);
    }
    if (FUSED && a.norm_w) {
#pragma unroll
        for (int i = 0; i < XP; i++) wr[i] = load_x4(a.norm_w, PIECE * i + 4 * tid, K);
    }

    constexpr int G = 64 / LPR;  // rows in flight per wave
    const int lane = tid & 63, wave = tid >> 6;
    const int sub = lane % LPR, grp = lane / LPR;
    int64_t row = (int64_t)blockIdx.x * (NW * G) + wave * G + grp;
    const bool has_row = row < p.N;
    // Rows past the end load (and then ignore) the last row, chunks past the end the last chunk: the preloads carry no
    // lane-dependent branch, so they issue back to back.
    const int64_t row00 = p.row0 + (int64_t)mat * p.N;
    int64_t grow = row00 + (has_row ? row : p.N - 1);
    const int nchunks = K / chunk_elems<TYPE>();

    // the residual the epilogue adds, requested now rather than after the reduction
    const int64_t ybase = i12 * a.y_b2 + i13 * a.y_b3;
    float rr[NC];
    if (FUSED && p.res && has_row && sub == LPR - 1) {
#pragma unroll
        for (int c = 0; c < NC; c++) rr[c] = p.res[ybase + row + c * p.y_col_stride];
    }

    // weight chunks requested before the activation prologue, so the weight stream's first HBM round trip overlaps
    // the load and quantization of x instead of following it
    constexpr int PRE = preload_of<TYPE>();
    WChunk<TYPE> pre[PRE];
#pragma unroll
    for (int i = 0; i < PRE; i++) {
        const int c = sub + i * LPR;
        pre[i] = load_chunk<TYPE>(p.w, grow, K, c < nchunks ? c : nchunks - 1);
    }

    int8_t *xq = (int8_t *)smem;
    float *xd = (float *)(smem + (size_t)NC * K);
    constexpr int XDB = TYPE == MX_TYPE_Q8_0 ? 32 : 256;
    int *xbs = (int *)(xd + NC * (K / XDB));
    if constexpr (FUSED) {
        if (a.glu_b || a.norm_w) {  // uniform: the fused prologue
            fused_prologue<TYPE, NC, NW>(a, x, xi12, i13, xr, br, wr, xq, xd, xbs);
        } else {
            plain_prologue<TYPE, NC, NW>(a, x, xr, xq, xd, xbs);
        }
    } else {
        plain_prologue<TYPE, NC, NW>(a, x, xr, xq, xd, xbs);
    }
    __syncthreads();
    if (!has_row) return;  // whole LPR-lane groups leave together; no barrier follows

    while (true) {
        float acc[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) acc[c] = 0.0f;
#pragma unroll
        for (int i = 0; i < PRE; i++) {
            const int c = sub + i * LPR;
            if (c < nchunks) dot_chunk<TYPE, NC, false>(pre[i], K, c, xq, xd, xbs, NC, acc);
        }
        if constexpr (TYPE == MX_TYPE_Q4_K) {  // a unit's registers are four chunks': one at a time
#pragma unroll 1
            for (int c = sub + PRE * LPR; c < nchunks; c += LPR)
                chunk_dot<TYPE, NC, false>(p.w, grow, K, c, xq, xd, xbs, NC, acc);
        } else {
#pragma unroll 4
            for (int c = sub + PRE * LPR; c < nchunks; c += LPR)
                chunk_dot<TYPE, NC, false>(p.w, grow, K, c, xq, xd, xbs, NC, acc);
        }
        const int64_t next = row + (int64_t)gridDim.x * (NW * G);
        const bool more = WIDE && next < p.N;
        if (more) {  // the next rows' first chunks, ahead of this row's reduction and store
            grow = row00 + next;
#pragma unroll
            for (int i = 0; i < PRE; i++) {
                const int c = sub + i * LPR;
                pre[i] = load_chunk<TYPE>(p.w, grow, K, c < nchunks ? c : nchunks - 1);
            }
        }
#pragma unroll
        for (int c = 0; c < NC; c++) acc[c] = sum_lanes<LPR>(acc[c]);
        if (sub == LPR - 1) {  // the lane holding the group's sum
            float *y = p.y + ybase + row;
            if (FUSED && p.res) {  // the residual ADD that follows the product, fused
#pragma unroll
                for (int c = 0; c < NC; c++) y[c * p.y_col_stride] = rr[c] + acc[c];
            } else {
#pragma unroll
                for (int c = 0; c < NC; c++) y[c * p.y_col_stride] = acc[c];
            }
        }
        if (!more) return;
        row = next;
        if (FUSED && p.res && sub == LPR - 1) {
#pragma unroll
            for (int c = 0; c < NC; c++) rr[c] = p.res[ybase + row + c * p.y_col_stride];
        }
    }
}

// Lanes per row: the fewest (16, 32 or 64) whose chunks per lane all fit the preload, so every weight byte of a lane
// is requested before the activation prologue; rows longer than that take 64 lanes. Measured on the decode shapes
// (K 1024..3072): one full preload beats more workgroups with shorter streams. A backend's option forces it.
static int pick_lpr(int64_t nchunks, int preload, int forced) {
    if (forced == 16 || forced == 32 || forced == 64) return forced;
    int lpr = 16;
    while (lpr < 64 && nchunks > (int64_t)preload * lpr) lpr *= 2;
    return lpr;
}

// The wide workgroups to launch at most: as many as the chip holds at a time by the kernel's registers and by LDS, behind a
// fused prologue one to a CU (2 x 6144 Q8_0 rows of K = 2048, four columns: 256 workgroups 10.2 us, 512 12.0).
template <int TYPE, int NC, int LPR, bool FUSED>
static int64_t mv_most(size_t lds) {
    if constexpr (FUSED) return 256;
    static const int regs = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *)k_matvec<TYPE, NC, LPR, FUSED, true>,
                                                         64 * mv_waves<TYPE, true>(), 0) != hipSuccess)
            (void)hipGetLastError();
        return std::max(n, 1);
    }();
    return 256 * std::max<int64_t>(1, std::min<int64_t>(regs, 160 * 1024 / (int64_t)(lds + 1024)));
}

static int64_t mv_groups(const MatvecArgs &a, int64_t rows) {  // workgroups of so many rows that hold every problem
    int64_t n = 0;
    for (int i = 0; i < a.nprob; i++) n += (a.prob[i].N + rows - 1) / rows;
    return n * a.nbatch;
}

// Wide or narrow (us, narrow / wide):
//   Q4_K, Q6_K. A wave quantizes whole super-blocks, so only four of eight would up to K = 1024. Q4_K, 2 x 3072 rows of K =
//     1024, two columns 4.6 / 4.7, behind a norm 6.0 / 6.2 (eight columns 12.2 / 12.0); 1024 rows, four columns 5.3 / 6.1;
//     16,384 rows, four columns 8.6 / 7.9. Q6_K, 2 x 6144 rows of K = 1024, eight columns 11.5 / 11.8, behind a norm
//     27.2 / 15.0 (narrow takes 256 registers there). K = 2048, 2 x 3072 rows, two columns: Q4_K 5.8 / 5.0, Q6_K 7.1 / 6.4.
//   Q5_K. One wide workgroup fits a CU (256 registers), two or three narrow ones up to four columns: 2 x 6144 rows of K =
//     2048, two columns 9.2 / 10.8, three 13.3 / 12.8, four 15.4 / 14.8, five (narrow 256 registers too) 25.6 / 16.2. A
//     second round that is half empty costs the wide form most: 2 x 3072 rows, four columns 9.9 / 11.5.
template <int TYPE, int NC, bool FUSED>
static bool mv_wide(const MatvecArgs &a, int lpr) {
    if constexpr (!mv_narrow<TYPE, NC, FUSED>()) return true;
    if (NC == 1) return false;
    if (TYPE == MX_TYPE_Q5_K) {
        const int64_t groups = mv_groups(a, 4 * (64 / lpr)), cap = 256;
        if (groups <= cap) return FUSED || 2 * groups > cap;
        return NC == 2 ? a.K >= 4096 : groups >= 2 * cap;
    }
    return a.K > 1024 || mv_groups(a, 1) >= 16384;
}

template <int TYPE, int NC, int LPR, bool FUSED, bool WIDE>
static hipError_t launch_one(const MatvecArgs &a, int64_t maxN, size_t lds, hipStream_t s) {
    if constexpr (WIDE ? NC >= 2 : mv_narrow<TYPE, NC, FUSED>()) {
        constexpr int NW = mv_waves<TYPE, WIDE>(), R = NW * (64 / LPR);  // rows of a workgroup
        int64_t groups = (maxN + R - 1) / R;
        if constexpr (WIDE) {
            // They go on to further rows once there are more than that. Q8_0, five columns: gate and up of 2 x 6144 rows, K =
            // 2048, behind a norm, as 256 / 384 / 768 workgroups 11.2 / 16.8 / 19.3 us; 151,936 rows of K = 1024 (two fit a
            // CU) as 256 / 512 / 768 / 4748 37.1 / 31.6 / 34.2 / 44.2 us. Q6_K, 37,984 rows of K = 2048, four columns (one
            // fits), as 256 / 512 21.8 / 27.0 us.
            const int64_t cap = mv_most<TYPE, NC, LPR, FUSED>(lds), per = (mv_groups(a, R) + cap - 1) / cap;
            groups = (groups + per - 1) / per;
        }
        const dim3 grid((unsigned)groups, (unsigned)a.nprob, (unsigned)a.nbatch);
        hipLaunchKernelGGL((k_matvec<TYPE, NC, LPR, FUSED, WIDE>), grid, dim3(64 * NW), lds, s, a);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;  // (mv_wide picks what there is)
}

template <int TYPE, int NC, bool FUSED>
static hipError_t launch_lpr(const MatvecArgs &a, int64_t maxN, size_t lds, hipStream_t s) {
    const int64_t nchunks = a.K / chunk_elems<TYPE>();
    int lpr = pick_lpr(nchunks, preload_of<TYPE>(), a.lpr);
    const bool wide = mv_wide<TYPE, NC, FUSED>(a, lpr);
    if (wide && mv_waves<TYPE, true>() > 4 && a.lpr == 0)
        // eight waves: fewer rows each rather than CUs left idle, while every lane has a chunk
        while (lpr < 64 && nchunks >= 2 * lpr && mv_groups(a, 512 / lpr) < 128) lpr *= 2;
    switch (lpr) {
        case 16:
            return wide ? launch_one<TYPE, NC, 16, FUSED, true>(a, maxN, lds, s) : launch_one<TYPE, NC, 16, FUSED, false>(a, maxN, lds, s);
        case 32:
            return wide ? launch_one<TYPE, NC, 32, FUSED, true>(a, maxN, lds, s) : launch_one<TYPE, NC, 32, FUSED, false>(a, maxN, lds, s);
        default:
            return wide ? launch_one<TYPE, NC, 64, FUSED, true>(a, maxN, lds, s) : launch_one<TYPE, NC, 64, FUSED, false>(a, maxN, lds, s);
    }
}

template <int TYPE, int NC>
static hipError_t launch_nc(const MatvecArgs &a, int64_t maxN, size_t lds, hipStream_t s) {
    bool fused = a.glu_b || a.norm_w;
    for (int i = 0; i < a.nprob; i++) fused = fused || a.prob[i].res;
    return fused ? launch_lpr<TYPE, NC, true>(a, maxN, lds, s) : launch_lpr<TYPE, NC, false>(a, maxN, lds, s);
}

template <int TYPE>
static hipError_t launch_type(const MatvecArgs &a, int64_t maxN, hipStream_t s) {
    const size_t lds = act_lds_bytes(TYPE, a.K, a.ncols);
    switch (a.ncols) {
        case 1: return launch_nc<TYPE, 1>(a, maxN, lds, s);
        case 2: return launch_nc<TYPE, 2>(a, maxN, lds, s);
        case 3: return launch_nc<TYPE, 3>(a, maxN, lds, s);
        case 4: return launch_nc<TYPE, 4>(a, maxN, lds, s);
        case 5: return launch_nc<TYPE, 5>(a, maxN, lds, s);
        case 6: return launch_nc<TYPE, 6>(a, maxN, lds, s);
        case 7: return launch_nc<TYPE, 7>(a, maxN, lds, s);
        case 8: return launch_nc<TYPE, 8>(a, maxN, lds, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_matvec(const MatvecArgs &a, hipStream_t s) {
    int64_t maxN = 0;
    for (int i = 0; i < a.nprob; i++) maxN = a.prob[i].N > maxN ? a.prob[i].N : maxN;
    if (maxN == 0) return hipSuccess;
    if (a.type == MX_TYPE_F16 || a.type == MX_TYPE_F32) return launch_matvec_f(a, s);
    switch (a.type) {
        case MX_TYPE_Q8_0: return launch_type<MX_TYPE_Q8_0>(a, maxN, s);
        case MX_TYPE_Q4_K: return launch_type<MX_TYPE_Q4_K>(a, maxN, s);
        case MX_TYPE_Q5_K: return launch_type<MX_TYPE_Q5_K>(a, maxN, s);
        case MX_TYPE_Q6_K: return launch_type<MX_TYPE_Q6_K>(a, maxN, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mx
