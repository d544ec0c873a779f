// k3x_prefill.hip - the prefill path of the MoE block (more than 8 tokens per call):
//
//   pf_rows     fp32 activations to bf16 hi and lo rows (the GEMMs' B source)
//   pf_router   router logits of every (token, expert) in double, with a bound on their
//               distance from the reference's chain (k3_router, k3_ops.c:1666-1688)
//   pf_topk     sigmoid, + bias (:1691-1692), each token's top-k by one wave (:1700-1716),
//               logits that the bound does not prove and that could reach it worked out
//               again as the chain, so the routing is the reference's bit for bit; and
//               the per-expert histogram
//   pf_scan     per-expert offsets (prefix sum) and the GEMM tile lists
//   pf_scatter  each (token, slot) to its row in its expert's segment
//   pf_gemm32   grouped GEMMs: gate/up of every expert segment with SwiGLU and the
//               routing weight (k3_matmul_mxfp4 :3323-3776, k3_situ_glu :148-161), then
//               down (pf_gemm_mx in the MXFP8 mode)
//   pf_dense    the shared expert's bf16 products (:1848-1860), the latent projections
//               and the trunk matrices
//   pf_combine  per token, the K expert rows summed in top-k order (:1941-1942), plus
//               the shared row (:1951), plus an optional residual
//
// The GEMMs run on v_mfma_f32_32x32x16_bf16 with MXFP4 weights dequantised exactly in
// registers; the activations are bf16 hi + lo pairs (hi only when the input is bf16,
// whose lo part is zero), so products are exact and only the fp32 accumulation rounds.
#include "k3x_device.h"
#include "k3x_topk.h"

#include <stdio.h>
#include <string.h>

#include <mutex>

#define PF_NT 256

// ------------------------------------------------------------------ rows
// The GEMMs' B source is rows of bf16: a bf16 call's activations as they are, and of fp32
// ones (z in the latent form among them) the hi and the lo rows that this kernel writes,
// x [T][ldx] fp32 -> hi [T][n], then lo [T][n].  bf16 x: rows copied (strided trunk rows).
__global__ void __launch_bounds__(PF_NT) pf_rows(const void *x, int x_bf16, int T, int n, int ldx,
                                                 uint16_t *hl)
{
    const int n8 = n >> 3;
    const size_t f = (size_t)blockIdx.x * PF_NT + threadIdx.x;
    if (f >= (size_t)T * n8) return;
    const size_t t = f / n8, c = (f % n8) * 8;
    if (x_bf16) {
        *(u32x4 *)(hl + t * n + c) = ld16((const uint16_t *)x + t * ldx + c);
        return;
    }
    float v[8];
    load_x8(x, 0, t * ldx + c, v);
    uint32_t hi[8], lo[8];
#pragma unroll
    for (int k = 0; k < 8; k++) split_bf16(v[k], hi[k], lo[k]);
    u32x4 h, l;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        h[k] = hi[2 * k] | (hi[2 * k + 1] << 16);
        l[k] = lo[2 * k] | (lo[2 * k + 1] << 16);
    }
    *(u32x4 *)(hl + t * n + c) = h;
    *(u32x4 *)(hl + ((size_t)T + t) * n + c) = l;
}

// ------------------------------------------------------------------ router
// Logits of every (token, expert) pair in double on the FP64 matrix cores, K cut into
// segments that run side by side, with a bound on how far the reference's logit, one
// sequential chain over i = 0 .. H-1 (k3_router, k3_ops.c:1666-1688), can lie from each
// sum.  The float logit is the chain's wherever the bound proves it (float_proven);
// pf_topk works a pair that it does not prove out again as the chain, where the pair could
// reach the token's selection.
//
// The bound.  A product of two floats is exact in double, so a chain of additions is off
// the exact sum by at most 2^-53 times the sum of its partial sums' magnitudes.  Over a
// chunk c of RM_KC elements every partial sum, in whatever order, is at most |S_c| + P_c:
// S_c the sum before the chunk, P_c = sum |w_i| max |x_i| over it.  So the two sums
// together are off by at most 2^-53 of sum_c RM_KC (|S_c| + P_c) for the chain (S_c the
// prefix: the segment's start plus the segment's own sum before c) and the same with the
// segment's own sums for this kernel: 2^-53 (sum over segments of n_s |start_s| + 128 B_s),
// B_s = sum_c (|S_c, own| + P_c), kept in float beside the accumulators; the factor
// 1 + 2^-10 covers the float roundings and the bound's second-order terms, n 2^-126 the
// products that underflow in P_c.  On N(0, 1) tokens at the K2 shape that leaves about one
// (token, expert) pair in 3 10^4 unproven, and one token in a few thousand whose selection
// it could change (about 45 us of the top-k then); a bound of 2^-53 n sum|p|, for any
// order, leaves fifteen times as many.
//
// The split.  A wave holds 32 experts x 16 NTT tokens (2 x NTT tiles of v_mfma_f64_16x16x4)
// of one segment; its operands come straight from memory, 32 k a step (lane (r, g): row r,
// k 8g .. 8g+7, element j the k-slot g of MFMA j: the order of a chunk's additions is
// free), the next step's loads in flight.  A workgroup's four waves hold four segments,
// summed in LDS; where the tiles are few, gridDim gives each to SG workgroups as well,
// whose parts pf_topk adds.  Bound by the FP64 matrix cores past a few hundred tokens, by
// load latency below.  One sequential chain per tile (three waves a SIMD, 48 experts x 64
// tokens a workgroup) made a routing call, router and top-k, 226 us at 16 tokens x 384 experts
// (8 workgroups, the chain's 1792 dependent steps and a load's latency every 64 k), 227 at 301,
// 229 at 1500, 231 at 2048 and 615 at 2048 x 896; now 20, 55, 208, 250 and 509.  It was the
// faster only where its tiles fill a round of the CUs (1700 to 2048 x 384, and twice that, by
// 2 to 10%).  (Tried at 2048 x 384 and within 2% of this: 64 tokens a wave, P_c by a float
// MFMA instead of shuffles, each workgroup starting its segments at another chunk.)
#define RM_E  32
#define RM_KC 64
#define RM_NT 256
#define RM_NW (RM_NT / WAVE)
#define RM_SGMAX K3X_PF_PARTS

struct PfRouterArgs {
    const void  *x;
    int          x_bf16;
    const float *W;
    int          T, H, E;
    int          sg;                 // workgroups along K
    // sg == 1: the float logit and how far the chain's float logit can lie from it (0:
    // proven), [T][E]; else the parts' sums and bounds [sg][T][E]
    float       *logit, *gap;
    double      *psum;
    float       *pbnd;
    int         *counts;             // [E] histogram that the top-k adds to, cleared here
};

typedef double f64x4 __attribute__((ext_vector_type(4)));

// chunks of segment s of S over H
__device__ __forceinline__ int rm_seg(int s, int S, int H)
{
    return (int)((unsigned)(H / RM_KC) * (unsigned)s / (unsigned)S);     // s <= 32
}

// The float logit of a sum v and the distance its chain's float logit can lie from it,
// given bnd = sum n_s |start_s| + 128 sum B_s.  A sum that is not finite met an infinity
// or a NaN, as the chain does whatever the order: proven.
__device__ __forceinline__ float rm_gap(double v, float bnd, int H)
{
    const double d = ((double)bnd * (1.0 + 0x1p-10) + fabs(v) * 64.0 + (double)H * 0x1p-126) * 0x1p-53;
    const float f = (float)v;
    if (!isfinite(v) || float_proven(v, d)) return 0.0f;
    const float lo = (float)(v - d), hi = (float)(v + d);
    const float gap = fmaxf(hi - f, f - lo);
    return gap == gap ? gap : __builtin_inff();          // a bound that overflowed: unknown
}

template <int NTT, bool BF>
__global__ void __launch_bounds__(RM_NT, 3) pf_router(PfRouterArgs a)
{
    constexpr int TT = 16 * NTT, NV = 2 * NTT * 4;           // tokens, values a lane
    constexpr int XL = BF ? 1 : 2;                           // 16-byte loads of 8 activations
    __shared__ double sd[RM_NW][NV][WAVE];
    __shared__ float  sb[RM_NW][NV][WAVE];
    if (blockIdx.x == 0 && a.counts)
        for (int e = threadIdx.x; e < a.E; e += RM_NT) a.counts[e] = 0;
    const int nEB = (a.E + RM_E - 1) / RM_E, nTB = (a.T + TT - 1) / TT;
    const int eb = blockIdx.x % nEB, tb = (blockIdx.x / nEB) % nTB, sg = blockIdx.x / (nEB * nTB);
    const int e0 = eb * RM_E, t0 = tb * TT;
    const int wave = wave_id(), lane = threadIdx.x % WAVE, r = lane & 15, g = lane >> 4;
    const int S = a.sg * RM_NW, s = sg * RM_NW + wave;
    const int c0 = rm_seg(s, S, a.H), c1 = rm_seg(s + 1, S, a.H);
    constexpr uint32_t xes = BF ? 2u : 4u;
    // rows past the experts or the tokens read out of range: zeros
    const rsrc_t rw = make_rsrc(a.W + (size_t)e0 * a.H, (uint32_t)min(RM_E, a.E - e0) * (uint32_t)a.H * 4u);
    const rsrc_t rx = make_rsrc((const uint8_t *)a.x + (size_t)t0 * a.H * xes,
                                (uint32_t)min(TT, a.T - t0) * (uint32_t)a.H * xes);
    const uint32_t wo = ((uint32_t)r * (uint32_t)a.H + 8u * g) * 4u;
    const uint32_t xo = ((uint32_t)r * (uint32_t)a.H + 8u * g) * xes;
    const uint32_t wrow = 16u * (uint32_t)a.H * 4u, xrow = 16u * (uint32_t)a.H * xes;

    u32x4 wv[2][2][2], xv[2][NTT][XL];
    auto ld = [&](int slot, int k0) AI {
        const bool on = k0 < c1 * RM_KC;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                wv[slot][i][h] = bload16(rw, on ? wo + i * wrow + (uint32_t)k0 * 4u + 16u * h : K3X_OOB);
#pragma unroll
        for (int i = 0; i < NTT; i++)
#pragma unroll
            for (int h = 0; h < XL; h++)
                xv[slot][i][h] = bload16(rx, on ? xo + i * xrow + (uint32_t)k0 * xes + 16u * h : K3X_OOB);
    };
    f64x4 acc[2][NTT];
    float bnd[2][NTT][4], l1[2], mx[NTT];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NTT; j++) {
            acc[i][j] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int v = 0; v < 4; v++) bnd[i][j][v] = 0.0f;
        }
    auto xval = [&](int slot, int i, int j) AI -> float {
        if (BF) {
            const uint32_t d = xv[slot][i][0][j >> 1];
            return (j & 1) ? __uint_as_float(d & 0xFFFF0000u) : __uint_as_float(d << 16);
        }
        return __uint_as_float(xv[slot][i][BF ? 0 : j >> 2][j & 3]);
    };
    auto use = [&](int slot) AI {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float wf[2], xf[NTT];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                wf[i] = __uint_as_float(wv[slot][i][j >> 2][j & 3]);
                l1[i] += fabsf(wf[i]);
            }
#pragma unroll
            for (int i = 0; i < NTT; i++) {
                xf[i] = xval(slot, i, j);
                mx[i] = fmaxf(mx[i], fabsf(xf[i]));
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int t = 0; t < NTT; t++)
                    acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)wf[i], (double)xf[t],
                                                                     acc[i][t], 0, 0, 0);
        }
    };
    SCHED_FENCE();
    ld(0, c0 * RM_KC);
    SCHED_FENCE();
    ld(1, c0 * RM_KC + 32);
    SCHED_FENCE();
    for (int c = c0; c < c1; c++) {
        // the chunk's start, before its products
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < NTT; t++)
#pragma unroll
                for (int v = 0; v < 4; v++) bnd[i][t][v] += fabsf((float)acc[i][t][v]);
#pragma unroll
        for (int i = 0; i < 2; i++) l1[i] = 0.0f;
#pragma unroll
        for (int i = 0; i < NTT; i++) mx[i] = 0.0f;
        use(0);
        SCHED_FENCE();
        ld(0, (c + 1) * RM_KC);
        SCHED_FENCE();
        use(1);
        SCHED_FENCE();
        ld(1, (c + 1) * RM_KC + 32);
        SCHED_FENCE();
        // P_c: row r's sum |w| and token r's max |x| over the four lanes that share them;
        // value v of a tile is expert g + 4v
#pragma unroll
        for (int i = 0; i < 2; i++) {
            l1[i] += __shfl_xor(l1[i], 16);
            l1[i] += __shfl_xor(l1[i], 32);
        }
#pragma unroll
        for (int i = 0; i < NTT; i++) {
            mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 16));
            mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 32));
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float p = __shfl(l1[i], g + 4 * v);
#pragma unroll
                for (int t = 0; t < NTT; t++) bnd[i][t][v] += p * mx[t];
            }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int t = 0; t < NTT; t++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                sd[wave][(i * NTT + t) * 4 + v][lane] = acc[i][t][v];
                sb[wave][(i * NTT + t) * 4 + v][lane] = bnd[i][t][v];
            }
    __syncthreads();
    // value v of lane (r, g) of tile (i, t): expert 16i + g + 4v, token 16t + r
    for (int p = threadIdx.x; p < RM_E * TT; p += RM_NT) {
        const int el = p % RM_E, tl = p / RM_E, e = e0 + el, t = t0 + tl;
        if (e >= a.E || t >= a.T) continue;
        const int sl = ((el >> 4) * NTT + (tl >> 4)) * 4 + ((el & 15) >> 2);
        const int ln = (el & 3) * 16 + (tl & 15);
        double sum = 0.0;
        float b = 0.0f;
#pragma unroll
        for (int w = 0; w < RM_NW; w++) {
            const int sw = sg * RM_NW + w;
            const float nw = (float)((rm_seg(sw + 1, S, a.H) - rm_seg(sw, S, a.H) + 1) * RM_KC);
            b += nw * fabsf((float)sum) + 128.0f * sb[w][sl][ln];
            sum += sd[w][sl][ln];
        }
        if (a.sg == 1) {
            const size_t o = (size_t)t * a.E + e;
            a.logit[o] = (float)sum;
            a.gap[o] = rm_gap(sum, b, a.H);
        } else {
            const size_t o = ((size_t)sg * a.T + t) * a.E + e;
            a.psum[o] = sum;
            a.pbnd[o] = b;
        }
    }
}

// ------------------------------------------------------------------ top-k
struct PfTopkArgs {
    PfRouterArgs r;                      // the router's inputs and its results
    const float *bias;                   // [E]
    int          K, renorm;
    float        routed_scale;
    int         *idx;   float *wt;       // [T][K]
    int         *uidx;  float *uwt;      // optional caller copies
};

// The reference's logit of (token t, expert e), one double chain over i = 0 .. H-1
// (k3_ops.c:1666-1688), by one wave: the lanes form CH_N products a step (exact in double;
// -0.0, the identity of the sum, past H) in the wave's LDS buffer, the next step's loads in
// flight, and every lane adds them in order.
#define CH_N 256
__device__ double pf_chain(const PfRouterArgs &a, int t, int e, double *buf, int lane)
{
    const uint32_t H = (uint32_t)a.H, xes = a.x_bf16 ? 2u : 4u;
    const rsrc_t rw = make_rsrc(a.W + (size_t)e * H, H * 4u);
    const rsrc_t rx = make_rsrc((const uint8_t *)a.x + (size_t)t * H * xes, H * xes);
    u32x4 w;
    u32x2 x0, x1;
    auto ld = [&](uint32_t k) AI {
        const uint32_t el = k + 4u * (uint32_t)lane;
        w = bload16(rw, el < H ? el * 4u : K3X_OOB);
        x0 = __builtin_amdgcn_raw_buffer_load_b64(rx, el < H ? el * xes : K3X_OOB, 0, 0);
        x1 = __builtin_amdgcn_raw_buffer_load_b64(rx, el < H && xes == 4u ? el * 4u + 8u : K3X_OOB, 0, 0);
    };
    double s = 0.0;
    ld(0u);
    for (uint32_t k = 0; k < H; k += CH_N) {
        const bool on = k + 4u * (uint32_t)lane < H;          // H is a multiple of 4
        float xf[4];
        if (a.x_bf16) {
            xf[0] = bf2f(x0[0] & 0xFFFFu); xf[1] = bf2f(x0[0] >> 16);
            xf[2] = bf2f(x0[1] & 0xFFFFu); xf[3] = bf2f(x0[1] >> 16);
        } else {
            xf[0] = __uint_as_float(x0[0]); xf[1] = __uint_as_float(x0[1]);
            xf[2] = __uint_as_float(x1[0]); xf[3] = __uint_as_float(x1[1]);
        }
        double p[4];
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = on ? (double)__uint_as_float(w[q]) * (double)xf[q] : -0.0;
        *(f64x2 *)(buf + 4 * lane) = (f64x2){p[0], p[1]};
        *(f64x2 *)(buf + 4 * lane + 2) = (f64x2){p[2], p[3]};
        ld(k + CH_N);
        // one wave: its LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 8
        for (int j = 0; j < CH_N; j += 2) {
            const f64x2 v = *(const f64x2 *)(buf + j);
            s += v[0];
            s += v[1];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    return s;
}

// One wave per token, TK_W tokens a workgroup: the scores and choices from the router's
// logits, the selection, and, while an expert whose logit is not proven could reach it
// (slack_reaches: its choice plus its slack is at least the K-th choice; every selected
// expert's is), those experts' logits as the chain and the selection again.  Every pass
// proves at least one more expert, so the loop ends; then the selected experts' choices
// are the reference's and every other one lies below the K-th: the selection and its
// weights are the reference's.  The per-expert histogram is counted in LDS first and
// added to the global counts once per workgroup and expert: a device-scope atomic per
// (token, slot) serialised on the busiest experts' counters (the Zipf chunk's first expert
// takes every token).
#define TK_W 4
template <int NE>
__global__ void __launch_bounds__(TK_W * WAVE) pf_topk(PfTopkArgs a)
{
    __shared__ int      s_idx[TK_W][K3X_MAX_TOPK];
    __shared__ float    s_w[TK_W][K3X_MAX_TOPK];
    __shared__ int      hist[1024];
    __shared__ __attribute__((aligned(16))) double chain[TK_W][CH_N];
    __shared__ TkList   list[TK_W];
    const int wave = wave_id(), lane = threadIdx.x % WAVE;
    const int T = a.r.T, E = a.r.E, H = a.r.H;
    const int t = blockIdx.x * TK_W + wave;
    if (a.r.counts)
        for (int e = threadIdx.x; e < E; e += TK_W * WAVE) hist[e] = 0;
    __syncthreads();
    if (t < T) {                                       // uniform over the wave
        // range-checked loads (an expert past E reads zeros): a load behind a branch would
        // be waited for on its own
        float sc[NE], cv[NE], sl[NE], bi[NE];
        const uint32_t ro = (uint32_t)(t * E);
        const rsrc_t rb = make_rsrc(a.bias, (uint32_t)E * 4u);
#pragma unroll
        for (int c = 0; c < NE; c++) bi[c] = bload_f32<0>(rb, 4u * (uint32_t)(c * WAVE + lane));
        if (a.r.sg == 1) {
            const rsrc_t rl = make_rsrc(a.r.logit, (uint32_t)(T * E) * 4u);
            const rsrc_t rg = make_rsrc(a.r.gap, (uint32_t)(T * E) * 4u);
#pragma unroll
            for (int c = 0; c < NE; c++) {
                const int e = c * WAVE + lane;
                const uint32_t o = e < E ? 4u * (ro + e) : K3X_OOB;
                sc[c] = bload_f32<0>(rl, o);
                sl[c] = bload_f32<0>(rg, o);
            }
        } else {
            const int sg = a.r.sg;
            const rsrc_t rs = make_rsrc(a.r.psum, (uint32_t)(sg * T * E) * 8u);
            const rsrc_t rg = make_rsrc(a.r.pbnd, (uint32_t)(sg * T * E) * 4u);
            double sum[NE];
            float b[NE];
#pragma unroll
            for (int c = 0; c < NE; c++) { sum[c] = 0.0; b[c] = 0.0f; }
            // two parts' loads in flight (one where the registers hold no more)
            constexpr int D = NE <= 8 ? 2 : 1;
            u32x2 v[D][NE];
            float w[D][NE];
            auto ld = [&](int i, int g) AI {
#pragma unroll
                for (int c = 0; c < NE; c++) {
                    const int e = c * WAVE + lane;
                    const uint32_t o = ((g < sg) & (e < E)) ? ro + e + (uint32_t)(g * T * E) : K3X_OOB / 8u;
                    v[i][c] = __builtin_amdgcn_raw_buffer_load_b64(rs, 8u * o, 0, 0);
                    w[i][c] = bload_f32<0>(rg, 4u * o);
                }
            };
#pragma unroll
            for (int i = 0; i < D; i++) {
                SCHED_FENCE();
                ld(i, i);
            }
            SCHED_FENCE();
            for (int g0 = 0; g0 < sg; g0 += D) {
#pragma unroll
                for (int i = 0; i < D; i++) {
                    const int g = g0 + i, S = sg * RM_NW;   // a part past the last adds zeros
                    const float n = (float)((rm_seg((g + 1) * RM_NW, S, H) - rm_seg(g * RM_NW, S, H) + 1) * RM_KC);
#pragma unroll
                    for (int c = 0; c < NE; c++) {
                        b[c] += (g < sg ? n * fabsf((float)sum[c]) : 0.0f) + w[i][c];
                        sum[c] += __builtin_bit_cast(double, v[i][c]);
                    }
                    SCHED_FENCE();
                    ld(i, g + D);
                    SCHED_FENCE();
                }
            }
#pragma unroll
            for (int c = 0; c < NE; c++) {
                sc[c] = (float)sum[c];
                sl[c] = rm_gap(sum[c], b[c], H);
            }
        }
#pragma unroll
        for (int c = 0; c < NE; c++) {
            sc[c] = sigmoid_ref(sc[c]);
            cv[c] = sc[c] + bi[c];
            if (sl[c] != 0.0f) sl[c] = logit_slack(sl[c], bi[c]);
        }
        for (;;) {
            float ck;
            wave_topk_vals<NE, true>(cv, sc, E, a.K, a.renorm, a.routed_scale, s_idx[wave],
                                     s_w[wave], lane, list[wave], nullptr, nullptr, &ck);
            uint32_t crit = 0u;
#pragma unroll
            for (int c = 0; c < NE; c++)
                if (c * WAVE + lane < E && sl[c] > 0.0f && slack_reaches(slack_key(cv[c], sl[c]), ck))
                    crit |= 1u << c;
            if (__ballot(crit != 0u) == 0ull) break;
            for (;;) {
                const uint64_t m = __ballot(crit != 0u);
                if (m == 0ull) break;
                const int l0 = (int)__builtin_ctzll(m);
                const int cc = __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)crit, l0));
                const float f = (float)pf_chain(a.r, t, cc * WAVE + l0, chain[wave], lane);
                const float s = sigmoid_ref(f);
                if (lane == l0) crit &= crit - 1u;
#pragma unroll
                for (int c = 0; c < NE; c++)
                    if (lane == l0 && c == cc) { sc[c] = s; cv[c] = s + bi[c]; sl[c] = 0.0f; }
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (lane < a.K) {
            const size_t o = (size_t)t * a.K + lane;
            const int e = s_idx[wave][lane];
            a.idx[o] = e;
            a.wt[o] = s_w[wave][lane];
            if (a.uidx) { a.uidx[o] = e; a.uwt[o] = s_w[wave][lane]; }
            if (a.r.counts) atomicAdd(&hist[e], 1);
        }
    }
    if (!a.r.counts) return;                               // uniform
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += TK_W * WAVE)
        if (hist[e]) atomicAdd(&a.r.counts[e], hist[e]);
}

// ------------------------------------------------------------------ scan
// One workgroup of 1024 threads (E <= 1024): offsets[e] = sum of counts below e, and the
// tile bases of the two routed GEMMs.  Each GEMM has PF_NC tile classes by an expert's
// tokens: of at most lim[0], of at most lim[1] (empty when that is lim[0]), and the others;
// class c takes nrb[c] x ceil(count / tpb[c]) tiles of tpb[c] columns.  tb[e] is the first
// tile of expert e in the GEMM's list (class 0's tiles first, then class 1's, then class
// 2's); tb[E + 2c] and tb[E + 2c + 1] are class c's number of tiles and its first.  Cursors
// cleared.  1 + 2 PF_NC inclusive scans, one element per thread (shuffles within each wave,
// then the waves' totals).
#define PF_NC 3
#define PF_NSC (1 + 2 * PF_NC)

struct PfScanArgs {
    const int *counts;
    int        E;
    int       *offsets, *cursor;
    int       *tb[2];                   // gate/up, down
    int        tpb[2][PF_NC];           // columns of a tile
    int        nrb[2][PF_NC];           // row blocks
    int        lim[2][2];               // most tokens of an expert of class 0, of class 1
};

__device__ __forceinline__ int pf_class(const PfScanArgs &a, int m, int c)
{
    return c <= a.lim[m][0] ? 0 : (c <= a.lim[m][1] ? 1 : 2);
}

__global__ void __launch_bounds__(1024) pf_scan(PfScanArgs a)
{
    __shared__ int wsum[PF_NSC][16], woff[PF_NSC][16], tot[PF_NSC];
    const int e = threadIdx.x, E = a.E, wave = e / WAVE, lane = e % WAVE;
    const int c = e < E ? a.counts[e] : 0;
    int v[PF_NSC];
    v[0] = c;
#pragma unroll
    for (int m = 0; m < 2; m++) {
        const int k = pf_class(a, m, c);
#pragma unroll
        for (int q = 0; q < PF_NC; q++)
            v[1 + PF_NC * m + q] = k == q ? a.nrb[m][q] * ((c + a.tpb[m][q] - 1) / a.tpb[m][q]) : 0;
    }
    if (e < E) a.cursor[e] = 0;
    // inclusive sums: within each wave by shuffles, then the waves' totals (wave 0)
    int in[PF_NSC];
#pragma unroll
    for (int i = 0; i < PF_NSC; i++) {
        in[i] = v[i];
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const int t = __shfl_up(in[i], o);
            if (lane >= o) in[i] += t;
        }
        if (lane == WAVE - 1) wsum[i][wave] = in[i];
    }
    __syncthreads();
    if (wave == 0 && lane < 16) {
#pragma unroll
        for (int i = 0; i < PF_NSC; i++) {
            int x = wsum[i][lane], inc = x;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const int t = __shfl_up(inc, o, 16);
                if (lane >= o) inc += t;
            }
            woff[i][lane] = inc - x;
            if (lane == 15) tot[i] = inc;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PF_NSC; i++) in[i] += woff[i][wave];
    // the exclusive value of e is its inclusive sum less its own
    if (e < E) {
        a.offsets[e] = in[0] - v[0];
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const int k = pf_class(a, m, c);
            int base = 0;
#pragma unroll
            for (int q = 0; q < PF_NC; q++) {
                if (k == q) a.tb[m][e] = base + in[1 + PF_NC * m + q] - v[1 + PF_NC * m + q];
                base += tot[1 + PF_NC * m + q];
            }
        }
    }
    if (e == 0) {
        a.offsets[E] = tot[0];
#pragma unroll
        for (int m = 0; m < 2; m++) {
            int base = 0;
#pragma unroll
            for (int q = 0; q < PF_NC; q++) {
                a.tb[m][E + 2 * q] = tot[1 + PF_NC * m + q];
                a.tb[m][E + 2 * q + 1] = base;
                base += tot[1 + PF_NC * m + q];
            }
        }
    }
}

// ------------------------------------------------------------------ scatter
// Each (token, slot) to a row of its expert's segment: a workgroup ranks its items per
// expert in LDS, reserves each expert's run with one device-scope atomic, and places its
// items in that run (the order within a segment is free: every row's products are its
// own, and the combine finds each row through pos_of).
__global__ void __launch_bounds__(PF_NT) pf_scatter(const int *idx, const float *wt, int TK, int K,
                                                    int E, const int *offsets, int *cursor,
                                                    int *perm_tok, float *perm_w, int *pos_of)
{
    __shared__ int cnt[1024], base[1024];
    for (int e = threadIdx.x; e < E; e += PF_NT) cnt[e] = 0;
    __syncthreads();
    const int i = blockIdx.x * PF_NT + threadIdx.x;
    const int e = i < TK ? idx[i] : 0;
    const int r = i < TK ? atomicAdd(&cnt[e], 1) : 0;
    __syncthreads();
    for (int f = threadIdx.x; f < E; f += PF_NT)
        if (cnt[f]) base[f] = offsets[f] + atomicAdd(&cursor[f], cnt[f]);
    __syncthreads();
    if (i >= TK) return;
    const int p = base[e] + r;
    perm_tok[p] = i / K;
    perm_w[p] = wt[i];
    pos_of[i] = p;
}

// ------------------------------------------------------------------ tile tables
// One descriptor per GEMM tile: {group, row block, first permuted row, tokens}; expert e
// owns tiles tb[e] .. of the GEMM's list, row blocks outer, column blocks inner.
__global__ void __launch_bounds__(PF_NT) pf_tiles(const int *counts, const int *offsets,
                                                  PfScanArgs a, int4 *desc_gu, int4 *desc_dn)
{
    const int e = blockIdx.x, c = counts[e], off = offsets[e];
    for (int m = 0; m < 2; m++) {
        const int k = pf_class(a, m, c), tpb = a.tpb[m][k], nrb = a.nrb[m][k];
        int4 *desc = (m ? desc_dn : desc_gu) + a.tb[m][e];
        const int nc = (c + tpb - 1) / tpb;
        for (int rel = threadIdx.x; rel < nrb * nc; rel += PF_NT) {
            const int rb = rel / nc, cb = rel % nc;
            desc[rel] = make_int4(e, rb, off + cb * tpb, min(tpb, c - cb * tpb));
        }
    }
}

// ------------------------------------------------------------------ GEMMs
// Y[p][r] = sum_k W_g[r][k] B[p][k] over the rows p of group g: an expert's segment of
// permuted rows (the grouped GEMMs, pf_gemm32 and pf_gemm_mx), or all rows of one dense
// product (pf_dense).
//
// K advances through a ring of slots: a slot holds one step's weights (registers,
// range-checked buffer loads, or LDS) and its B block (LDS, filled by buffer loads
// straight to LDS: lane i of a load writes 16 bytes at the load's LDS base + 16 i; rows
// past the block's tokens read out of range and land as zeros).  Each step waits for its
// own slot's loads, meets the other waves at one barrier (after which every wave's share
// of the block is in LDS and the slot used by the previous step is free), refills that
// slot and runs the step's MFMAs.
//
// B sources are bf16 rows [HL][brows][ldb] (hi, then lo).  A load to LDS takes whole runs
// of a row (256 bytes of a quad of 128 k, 128 of pf_dense's 64), the 16-byte k-groups of
// column c in the order pos ^ f(c), so that the LDS reads of one k-group over 16
// consecutive columns fall into distinct banks.  (Planes [2][K/8][rows][8], with a gather
// of the routed rows into their permuted order, read LDS the same way but cost that pass:
// 145 us of a 2048-token chunk at the K2 shape, 354 of the latent one, 32 to 57 us of a
// small call, where it was bound by latency.)
struct PfGemmArgs {
    const uint8_t  *wm[2];      // group 0's matrices (gate, up) or (down), tiled
    size_t          gstride;    // bytes between groups' records
    int             R, K;       // rows and inner dimension of each matrix
    const int4     *desc;       // grouped: per tile {group, row block, first row, rows}
    const int      *ntile;      // tiles in this launch's list
    const int      *dbase;      // the list starts at desc + *dbase
    int             n0;         // pf_dense: rows
    const uint16_t *bsrc;       // B rows [HL][brows][ldb] bf16
    int             brows;      // rows of each part
    int             ldb;        // elements between rows
    const int      *perm;       // B row of permuted row p, or NULL: row_base + p
    int             row_base;
    const float    *pw;         // weight of permuted row p (gate/up epilogue), or NULL: 1
    uint16_t       *act;        // gate/up output rows [2][arows][R] bf16 (hi, lo)
    int             arows;
    float          *y;          // down output rows [*][R] fp32
    int             out_base;   // output row = out_base + p
    float           b1, b2;     // SiTU betas of the gate/up epilogue (0: uncapped)
    int             ldy;        // floats between output rows (0: R)
    // MXFP8 mode (pf_gemm_mx): B codes [K/16][brows][16] bytes and scales [K/128][brows]
    // dwords (byte b = the 32-k block 4q + b); the gate/up output in the same two forms
    // over R, arows rows
    const uint8_t  *b8;
    const uint32_t *b8s;
    uint8_t        *o8, *o8s;
};


// ------------------------------------------------------------------ dense GEMM
// One dense product Y[p][r] = sum_k W[r][k] B[p][k] with bf16 weights (the shared
// experts, the latent projections, the trunk matrices): W in the 16-row tile layout
// (per 128-k quad, 16-byte runs at t*1024 + (row + 16*kq)*16 for k = 32kq + 8t .. +7), B
// the activation rows.  Both operands go through LDS, fetched by loads straight to LDS,
// so that every weight byte a workgroup reads serves all of its columns and every B byte
// all of its rows; the four waves (2 x 2) take RW x CW tiles of 32 x 32 each (NMAT
// matrices: gate and up of the same rows together) on v_mfma_f32_32x32x16_bf16.
//
// K advances 64 at a time through a ring of NS stages.  A stage holds the workgroup's
// A block as [matrix][k-group g][row][8] (16-byte runs), so that the 32 lanes of an MFMA
// operand that share a k-group read 512 consecutive bytes, and its B block as
// [column][g ^ (column / 2 % 8)][8].  Each step waits for its stage (the loads issued after it are the NS - 2 stages
// ahead: stages past the end load out of range, which reads nothing and keeps the count
// exact), meets the other waves, refills the stage freed by the previous step and runs
// its 16 k-steps' MFMAs.
template <int NMAT, int RW, int CW, int HL, bool GU, int NS>
__global__ void __launch_bounds__(PF_NT) pf_dense(PfGemmArgs a)
{
    constexpr int BM = 2 * RW * 32;                // rows of each matrix per workgroup
    constexpr int BN = 2 * CW * 32;                // B columns per workgroup
    constexpr int TPB = BN / HL;                   // tokens per workgroup
    constexpr int SA = NMAT * BM * 128;            // A bytes per stage (64 k)
    constexpr int SB = BN * 128;
    constexpr int SS = SA + SB;
    constexpr int NJA = SA / (PF_NT * 16), NJB = SB / (PF_NT * 16);
    constexpr int LPS = NJA + NJB;                 // vector loads per stage per wave
    static_assert(NJA * PF_NT * 16 == SA && NJB * PF_NT * 16 == SB, "stage must split evenly");
    static_assert(NS >= 2 && (NS - 2) * LPS < 64, "vmcnt range");
    __shared__ __attribute__((aligned(16))) uint8_t sm[NS * SS];

    const int wave = wave_id(), lane = threadIdx.x % WAVE, tid = threadIdx.x;
    const int wr = wave >> 1, wc = wave & 1;
    int rb, p0, ntok;
    {
        // tiles dealt to the 8 XCDs in contiguous runs (workgroups go round-robin), so
        // that the column blocks of a row block run back to back on one XCD and read its
        // weights from that XCD's L2; the grid is a multiple of 8, surplus workgroups
        // leave at once
        const int nrb = (a.R + BM - 1) / BM, nc = (a.n0 + TPB - 1) / TPB, ntiles = nrb * nc;
        const int per = (ntiles + 7) >> 3;
        const int k = blockIdx.x >> 3, dt = (blockIdx.x & 7) * per + k;
        if (k >= per || dt >= ntiles) return;
        rb = dt / nc;
        p0 = (dt % nc) * TPB;
        ntok = min(TPB, a.n0 - p0);
    }
    const int nst = a.K >> 6;

    // ---- A: the row block's weights of each matrix; rows past R read out of range
    const uint32_t tbytes = (uint32_t)a.K * 32u;
    const int t16 = rb * (BM / 16), R16 = a.R >> 4;
    const uint32_t ntl = (uint32_t)(R16 - t16 < BM / 16 ? R16 - t16 : BM / 16);
    rsrc_t ra[NMAT];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
        ra[m] = make_rsrc(a.wm[m] + (size_t)t16 * tbytes, ntl * tbytes);
    // load j of a stage: 16-byte run c = j*256 + tid -> (matrix, g, row) of the A block,
    // or (column, position) of the B block; its offset in the stage's source, less the
    // stage's own step (A: (st>>1)*4096 + (st&1)*512, B: st*128 bytes)
    uint32_t aoff[NJA], boff[NJB];
#pragma unroll
    for (int j = 0; j < NJA; j++) {
        const int c = j * PF_NT + tid;
        const int rem = c % (BM * 8), g = rem / BM, r = rem % BM;
        aoff[j] = (uint32_t)(r >> 4) * tbytes + (uint32_t)(g & 3) * 1024u +
                  (uint32_t)((r & 15) + 16 * (g >> 2)) * 16u;
    }
    const rsrc_t rbs = make_rsrc(a.bsrc, (uint32_t)((size_t)HL * a.brows * a.ldb * 2));
#pragma unroll
    for (int j = 0; j < NJB; j++) {
        const int c = j * PF_NT + tid;
        const int col = c >> 3, g = (c & 7) ^ ((col >> 1) & 7), tok = col / HL, hl = col % HL;
        boff[j] = tok < ntok ? (uint32_t)(hl * a.brows + a.row_base + p0 + tok) * (uint32_t)a.ldb * 2u +
                                   (uint32_t)g * 16u
                             : K3X_OOB;
    }

    auto ld = [&](int slot, int st) AI {
        const bool on = st < nst;
        const uint32_t sa = (uint32_t)(st >> 1) * 4096u + (uint32_t)(st & 1) * 512u;
        uint8_t *base = sm + slot * SS;
#pragma unroll
        for (int j = 0; j < NJA; j++) {
            const int m = (j * PF_NT) / (BM * 8);            // uniform per load
            // (resource and offset through locals: the host pass of this template
            // rejects a captured array element as the builtin's operand)
            const rsrc_t r = ra[m];
            const uint32_t o = on ? aoff[j] + sa : K3X_OOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                r, (lds_void *)(base + (j * PF_NT + wave * WAVE) * 16), 16, o, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < NJB; j++) {
            // (a column past the tokens keeps an out-of-range offset: K3X_OOB plus at most
            // K/64 steps of 128 bytes stays below 2^32 and past the rows)
            const uint32_t o = on ? boff[j] + (uint32_t)st * 128u : K3X_OOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rbs, (lds_void *)(base + SA + (j * PF_NT + wave * WAVE) * 16), 16, o, 0, 0, 0);
        }
    };

    f32x16 acc[NMAT][RW][CW];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int c = 0; c < CW; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[m][i][c][v] = 0.f;

    const int l32 = lane & 31, h = lane >> 5;
    auto compute = [&](int slot) AI {
        const uint8_t *base = sm + slot * SS;
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            const int g = 2 * s4 + h;
            bf16x8 bf[CW];
#pragma unroll
            for (int c = 0; c < CW; c++)
                bf[c] = as_bf16x8(*(const u32x4 *)(base + SA + ((wc * CW + c) * 32 + l32) * 128 +
                                                   ((g ^ ((l32 >> 1) & 7)) << 4)));
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < RW; i++) {
                    const bf16x8 av = as_bf16x8(
                        *(const u32x4 *)(base + ((m * 8 + g) * BM + (wr * RW + i) * 32 + l32) * 16));
#pragma unroll
                    for (int c = 0; c < CW; c++) acc[m][i][c] = mfma32(av, bf[c], acc[m][i][c]);
                }
        }
    };

#pragma unroll
    for (int s = 0; s < NS - 1; s++) {
        SCHED_FENCE();
        ld(s, s);
    }
    SCHED_FENCE();
    for (int st = 0; st < nst; st++) {
        meet<(NS - 2) * LPS>();
        SCHED_FENCE();
        ld((st + NS - 1) % NS, st + NS - 1);
        SCHED_FENCE();
        compute(st % NS);
    }
    // no load to LDS may still be landing when the workgroup ends
    WAIT_VMCNT_LGKM0(0);

    // ---- epilogue: lane holds column l32 of each column tile, rows 8aa + 4h + b
#pragma unroll
    for (int c = 0; c < CW; c++) {
        const int col = (wc * CW + c) * 32 + l32;
        const int tl = col / HL;
        const bool writer = (HL == 1 || (col & 1) == 0) && tl < ntok;
        const int p = p0 + tl;
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int aa = 0; aa < 4; aa++) {
                const int r0 = rb * BM + (wr * RW + i) * 32 + 8 * aa + 4 * h;
                float v0[4], v1[4];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    v0[b] = acc[0][i][c][4 * aa + b];
                    if (HL == 2) v0[b] += __shfl_xor(v0[b], 1);
                    if (NMAT == 2) {
                        v1[b] = acc[NMAT - 1][i][c][4 * aa + b];
                        if (HL == 2) v1[b] += __shfl_xor(v1[b], 1);
                    }
                }
                if (!writer || r0 >= a.R) continue;
                if (GU) {
                    uint32_t hi[4], lo[4];
#pragma unroll
                    for (int b = 0; b < 4; b++) split_bf16(situ(v0[b], v1[b], a.b1, a.b2), hi[b], lo[b]);
                    const size_t o = (size_t)(a.out_base + p) * a.R + r0;
                    const size_t plane = (size_t)a.arows * a.R;
                    *(u32x2 *)(a.act + o) = (u32x2){hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
                    *(u32x2 *)(a.act + plane + o) = (u32x2){lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
                } else {
                    float *dst = a.y + (size_t)(a.out_base + p) * (a.ldy ? a.ldy : a.R) + r0;
                    *(f32x4 *)dst = (f32x4){v0[0], v0[1], v0[2], v0[3]};
                }
            }
    }
}

// ------------------------------------------------------------------ grouped GEMM, 32x32
// The routed GEMMs (MXFP4 weights) on v_mfma_f32_32x32x16_bf16.  A workgroup computes
// NW*RT32*32 weight rows (NMAT matrices: gate and up together) by CT32 column tiles of 32
// B columns (HL columns per token: hi, or hi and lo); a wave owns RT32 row tiles of 32
// rows (two 16-row tiles of the fp4 layout), its weights held in registers through a
// ring of 4 quads of 128 k, and the waves share each quad's B block in LDS.
//
// K order.  Within a quad, lane L (row R = L%32, h = L/32) loads two 16-byte scale
// groups of row R: group kq = h (load 0) and kq = 2 + h (load 1).  Dword d of load g
// feeds the MFMA of step (g, d) with k = 64g + 32h + 8d .. +7, so one 32x32x16 step
// multiplies k-slots {64g + 8d .. +7} (lanes 0-31) and {64g + 32 + 8d .. +7} (lanes
// 32-63).  The B block in LDS holds column col's 16 k-groups of the quad at
// 16 col + (k-group ^ col % 16).  Every product of the quad is formed exactly once;
// only the order of the fp32 additions differs from the 16x16 form.
template <bool EXACT, int NMAT, int RT32, int CT32, int HL, bool GU, int NW, int MINW>
__global__ void __launch_bounds__(NW * WAVE, MINW) pf_gemm32(PfGemmArgs a)
{
    constexpr int NTH = NW * WAVE;
    constexpr int NCOL = CT32 * 32;
    constexpr int QB = NCOL * 128 * 2;
    constexpr int NJ = QB / (NTH * 16);
    constexpr int RING = 4;
    // vector loads a quad issues per wave: 2 code loads per 32 rows and the B pieces, plus
    // (the first quad of a super-quad) 2 scale dwords per 32 rows, which hold the scale
    // bytes of the super-quad's four quads
    constexpr int LPI = NMAT * RT32 * 2 + NJ;
    constexpr int LPS = LPI + NMAT * RT32 * 2;
    static_assert(NJ * NTH * 16 == QB, "B quad must split evenly");
    static_assert(LPI + LPS < 64, "vmcnt range");
    __shared__ __attribute__((aligned(16))) uint8_t sB[RING * QB];

    const int wave = wave_id(), lane = threadIdx.x % WAVE;
    int g, rb, ntok, p0;
    {
        // Workgroups are dealt to the 8 XCDs round-robin; tiles are dealt to them in
        // contiguous runs instead (XCD x takes tiles x*per .. x*per + per-1 in order), so
        // the column blocks of one weight row block run back to back on one XCD and
        // re-read the weights from its L2.  The grid is a multiple of 8.
        // the descriptor words are read into scalar registers (readfirstlane): the
        // weight resources built from them must be wave-uniform, or every buffer load
        // becomes a loop over distinct descriptors
        const int ntiles = __builtin_amdgcn_readfirstlane(*a.ntile);
        const int per = (ntiles + 7) >> 3;
        const int k = blockIdx.x >> 3, tile = (blockIdx.x & 7) * per + k;
        if (k >= per || tile >= ntiles) return;
        const int4 d = a.desc[__builtin_amdgcn_readfirstlane(*a.dbase) + tile];
        g = __builtin_amdgcn_readfirstlane(d.x); rb = __builtin_amdgcn_readfirstlane(d.y);
        p0 = __builtin_amdgcn_readfirstlane(d.z); ntok = __builtin_amdgcn_readfirstlane(d.w);
    }
    const int nQ = a.K >> 7;

    // ---- weights: row tile pair i = 16-row tiles 2*tp, 2*tp+1 of this wave
    const uint32_t tbytes = (uint32_t)fp4_tile_bytes(a.K);
    const int R16 = a.R >> 4;
    const int Rl = lane & 31, h = lane >> 5;
    rsrc_t ra[NMAT][RT32];
    int tp16[RT32];
#pragma unroll
    for (int i = 0; i < RT32; i++) {
        const int t16 = ((rb * NW + wave) * RT32 + i) * 2;
        tp16[i] = t16;
        // readfirstlane: the clamp is a VALU med3, whose result would make the weight
        // resource a vector operand
        const int ntl = __builtin_amdgcn_readfirstlane(R16 - t16 < 0 ? 0 : (R16 - t16 > 2 ? 2 : R16 - t16));
#pragma unroll
        for (int m = 0; m < NMAT; m++)
            ra[m][i] = make_rsrc(a.wm[m] + (size_t)g * a.gstride + (size_t)t16 * tbytes,
                                 (uint32_t)ntl * tbytes);
    }
    // this lane's offsets inside a pair: its 16-row tile, row, and group h (load 0)
    const uint32_t lc = (uint32_t)(Rl >> 4) * tbytes + (uint32_t)((Rl & 15) + 16 * h) * 16u;
    const uint32_t ls = (uint32_t)(Rl >> 4) * tbytes + 4096u + (uint32_t)((Rl & 15) + 16 * h) * 4u;

    // ---- B pieces: entry e = (wave*NJ + j)*64 + lane = 16 col + pos, k-group pos ^ col%16
    const rsrc_t rbs = make_rsrc(a.bsrc, (uint32_t)((size_t)HL * a.brows * a.ldb * 2));
    uint32_t boff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int e = (wave * NJ + j) * WAVE + lane;
        const int col = e >> 4, kg = (e ^ col) & 15;
        const int tok = col / HL, hl = col % HL;
        if (tok < ntok) {
            const int row = a.perm ? a.perm[p0 + tok] : a.row_base + p0 + tok;
            boff[j] = (uint32_t)(hl * a.brows + row) * (uint32_t)a.ldb * 2u + (uint32_t)kg * 16u;
        } else {
            boff[j] = K3X_OOB;
        }
    }

    struct AQ {
        u32x4    c[NMAT][RT32][2];
    };
    AQ A[RING];
    // scale dwords: sn is loaded with the first quad of a super-quad (slot 0: quad q is
    // always computed from slot q % 4), and copied to sc before that quad is computed,
    // while the three other quads of the previous super-quad still read sc
    uint32_t sn[NMAT][RT32][2], sc[NMAT][RT32][2];
    auto ld = [&](int slot, int q) AI {
        const bool on = q < nQ;
        const uint32_t qc = (uint32_t)(q >> 2) * 4352u + (uint32_t)(q & 3) * 1024u;
        const uint32_t qs = (uint32_t)(q >> 2) * 4352u;
#pragma unroll
        for (int m = 0; m < NMAT; m++)
#pragma unroll
            for (int i = 0; i < RT32; i++)
#pragma unroll
                for (int gl = 0; gl < 2; gl++) {
                    A[slot].c[m][i][gl] = wld16(ra[m][i], on ? lc + qc + 512u * gl : K3X_OOB);
                    if (slot == 0) sn[m][i][gl] = wld4(ra[m][i], on ? ls + qs + 128u * gl : K3X_OOB);
                }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint32_t o = boff[j] + (uint32_t)q * 256u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rbs, (lds_void *)(sB + slot * QB + (wave * NJ + j) * 1024), 16, o, 0, 0, 0);
        }
    };

    f32x16 acc[NMAT][RT32][CT32];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < RT32; i++)
#pragma unroll
            for (int c = 0; c < CT32; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[m][i][c][v] = 0.f;

    // k-group 8 gl + 4 h + d of column Rl (the two xor terms share no bits with it)
    const int bl = Rl * 256 + (((4 * h) ^ (Rl & 15)) << 4);
    auto compute = [&](int slot, int q) AI {
        const uint8_t *bb = sB + slot * QB;
        const int sh = 8 * (q & 3);
        if (slot == 0) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < RT32; i++)
#pragma unroll
                    for (int gl = 0; gl < 2; gl++) sc[m][i][gl] = sn[m][i][gl];
        }
#pragma unroll
        for (int gl = 0; gl < 2; gl++)
#pragma unroll
            for (int d = 0; d < 4; d++) {
                bf16x8 bf[CT32];
#pragma unroll
                for (int c = 0; c < CT32; c++)
                    bf[c] = as_bf16x8(*(const u32x4 *)(bb + c * 8192 + (bl ^ ((8 * gl + d) << 4))));
#pragma unroll
                for (int m = 0; m < NMAT; m++)
#pragma unroll
                    for (int i = 0; i < RT32; i++) {
                        const uint32_t sb = (sc[m][i][gl] >> sh) & 255u;
                        const bf16x8 av = EXACT ? dq8_exact(A[slot].c[m][i][gl][d], sb)
                                                : dq8(A[slot].c[m][i][gl][d], e8m0_scale(sb));
#pragma unroll
                        for (int c = 0; c < CT32; c++) acc[m][i][c] = mfma32(av, bf[c], acc[m][i][c]);
                    }
            }
    };

#pragma unroll
    for (int s = 0; s < RING - 1; s++) {
        SCHED_FENCE();
        ld(s, s);
    }
    SCHED_FENCE();
    int q = 0;
    // meet quad q + s once the loads issued after its own are all that remain: those of
    // quads q + s + 1 and q + s + 2, of which q + 4 (the next super-quad's first) also
    // loads the scale dwords
    static_assert(RING == 4, "written for a ring of 4");
    for (; q + RING <= nQ; q += RING) {
        meet<2 * LPI>();       SCHED_FENCE(); ld(3, q + 3); SCHED_FENCE(); compute(0, q);
        meet<2 * LPI>();       SCHED_FENCE(); ld(0, q + 4); SCHED_FENCE(); compute(1, q + 1);
        meet<LPI + LPS>();     SCHED_FENCE(); ld(1, q + 5); SCHED_FENCE(); compute(2, q + 2);
        meet<LPS + LPI>();     SCHED_FENCE(); ld(2, q + 6); SCHED_FENCE(); compute(3, q + 3);
    }
    if (q < nQ)     { meet<2 * LPI>(); compute(0, q); }
    if (q + 1 < nQ) { meet<LPI>();     compute(1, q + 1); }
    if (q + 2 < nQ) { meet<0>();       compute(2, q + 2); }
    WAIT_VMCNT_LGKM0(0);

    // ---- epilogue: lane holds column Rl of each column tile, rows 8a + 4h + b
#pragma unroll
    for (int c = 0; c < CT32; c++) {
        const int col = c * 32 + Rl;
        const int tl = col / HL;
        const bool writer = (HL == 1 || (col & 1) == 0) && tl < ntok;
        const int p = p0 + tl;
#pragma unroll
        for (int i = 0; i < RT32; i++)
#pragma unroll
            for (int aa = 0; aa < 4; aa++) {
                const int r0 = tp16[i] * 16 + 8 * aa + 4 * h;
                float v0[4], v1[4];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    v0[b] = acc[0][i][c][4 * aa + b];
                    if (HL == 2) v0[b] += __shfl_xor(v0[b], 1);
                    if (NMAT == 2) {
                        v1[b] = acc[NMAT - 1][i][c][4 * aa + b];
                        if (HL == 2) v1[b] += __shfl_xor(v1[b], 1);
                    }
                }
                if (!writer || r0 >= a.R) continue;
                if (GU) {
                    const float w = a.pw ? a.pw[p] : 1.0f;
                    uint32_t hi[4], lo[4];
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        const float yv = (w == 0.0f) ? 0.0f : w * situ(v0[b], v1[b], a.b1, a.b2);
                        split_bf16(yv, hi[b], lo[b]);
                    }
                    const size_t o = (size_t)(a.out_base + p) * a.R + r0;
                    const size_t plane = (size_t)a.arows * a.R;
                    *(u32x2 *)(a.act + o) = (u32x2){hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
                    *(u32x2 *)(a.act + plane + o) = (u32x2){lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
                } else {
                    float *dst = a.y + (size_t)(a.out_base + p) * (a.ldy ? a.ldy : a.R) + r0;
                    *(f32x4 *)dst = (f32x4){v0[0], v0[1], v0[2], v0[3]};
                }
            }
    }
}

// ------------------------------------------------------------------ MXFP8 mode
// The opt-in prefill mode K3X_PREFILL_MXFP8: the routed expert products on the scaled
// matrix cores (v_mfma_scale_f32_32x32x64_f8f6f4), the weights as stored (E2M1 codes,
// E8M0 scale per 32 k, applied by the matrix core), the activations quantised to MXFP8:
// blocks of 32 k sharing an E8M0 scale 2^X, X the least integer with max|v| <= 448 * 2^X
// over the block's finite values (clamped to [-127, 127]; -127 for a block with no
// non-zero finite value), each finite value v * 2^-X rounded to the nearest E4M3 (FN
// encoding) value, ties to the even code, a non-finite one the NaN code.  The gate/up
// input is the token's row (x, or z in a LatentMoE layer); the down input is the
// gate/up output w * SiTU(gate, up), quantised in the gate/up epilogue.

typedef int i32x8 __attribute__((ext_vector_type(8)));

// E8M0 byte of a block whose largest finite magnitude is m
__device__ __forceinline__ int mx8_scale(float m)
{
    if (!(m > 0.0f)) return 0;
    const uint32_t b = __float_as_uint(m);
    int X = (int)((b >> 23) & 255u) - 127 - 8 + ((b & 0x7FFFFFu) > 0x600000u ? 1 : 0);
    X = X < -127 ? -127 : (X > 127 ? 127 : X);
    return X + 127;
}

// v (finite, |v| <= 448) to its E4M3 code, nearest value, ties to the even code
__device__ __forceinline__ uint32_t e4m3_rne(float v)
{
    const uint32_t sign = (__float_as_uint(v) >> 24) & 0x80u;
    const float a = fabsf(v);
    if (a < 0x1p-6f) return sign | (uint32_t)rintf(a * 512.0f);     // steps of 2^-9
    const int E = (int)((__float_as_uint(a) >> 23) & 255u) - 127;     // -6 .. 8
    const uint32_t m = (uint32_t)rintf(a * __uint_as_float((uint32_t)(127 + 3 - E) << 23));
    return sign | (m == 16u ? (uint32_t)(E + 8) << 3 : ((uint32_t)(E + 7) << 3) | (m - 8u));
}

// SiTU out of line: its inlined expansion over the sixteen values of a quantisation block
// would take the registers the accumulators need
__device__ __attribute__((noinline)) float situ_call(float g, float u, float b1, float b2)
{
    return situ(g, u, b1, b2);
}

// the code of v in a block of scale byte sb (inv = 2^-X)
__device__ __forceinline__ uint32_t mx8_code(float v, float inv)
{
    if (!isfinite(v)) return ((__float_as_uint(v) >> 24) & 0x80u) | 0x7Fu;
    return e4m3_rne(v * inv);
}

__device__ __forceinline__ float mx8_inv(int sb) { return __uint_as_float((uint32_t)(254 - sb) << 23); }

// The routed experts' MXFP8 input in permuted order: src row perm_tok[p] (bf16 or fp32,
// rows ld elements apart), X elements -> codes [X/16][TK][16], scales [X/128][TK] dwords.
// A workgroup takes MX_R rows by one 128-k quad, one thread per (row, 32-k block); the
// codes go through LDS so that the stores run along the rows of a k16-group (1 KB
// contiguous) and each row's four scale bytes are one dword.
#define MX_R 64

static inline unsigned pf_mx8_grid(int TK, int X) { return (unsigned)(((TK + MX_R - 1) / MX_R) * (X / 128)); }

__global__ void __launch_bounds__(PF_NT) pf_mx8_rows(const void *src, int bf16, int ld, int X,
                                                     const int *perm_tok, int TK,
                                                     uint8_t *codes, uint8_t *scales)
{
    static_assert(MX_R * 4 == PF_NT, "a thread per (row, block)");
    __shared__ u32x4 sc[8][MX_R + 1];          // [k16-group of the quad][row]
    __shared__ uint32_t ss[MX_R];
    const int nq = X / 128;
    const int q = blockIdx.x % nq, p0 = (blockIdx.x / nq) * MX_R;
    const int r = threadIdx.x >> 2, b = threadIdx.x & 3, p = p0 + r;
    uint32_t w[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    int sb = 0;
    if (p < TK) {
        const size_t base = (size_t)perm_tok[p] * ld + (size_t)q * 128 + (size_t)b * 32;
        float v[4][8];
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            load_x8(src, bf16, base + 8 * j, v[j]);
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (isfinite(v[j][e])) m = fmaxf(m, fabsf(v[j][e]));
        }
        sb = mx8_scale(m);
        const float inv = mx8_inv(sb);
#pragma unroll
        for (int d = 0; d < 8; d++) {
            uint32_t c = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) c |= mx8_code(v[d / 2][(d % 2) * 4 + e], inv) << (8 * e);
            w[d] = c;
        }
    }
    sc[2 * b][r] = (u32x4){w[0], w[1], w[2], w[3]};
    sc[2 * b + 1][r] = (u32x4){w[4], w[5], w[6], w[7]};
    // the row's four scale bytes, block b at byte b, gathered by its lane group of four
    uint32_t sw = (uint32_t)sb << (8 * b);
    sw |= __shfl_xor(sw, 1);
    sw |= __shfl_xor(sw, 2);
    if (b == 0) ss[r] = sw;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int i = j * PF_NT + threadIdx.x, g = i / MX_R, rr = i % MX_R, pp = p0 + rr;
        if (pp < TK) *(u32x4 *)(codes + ((size_t)(8 * q + g) * TK + pp) * 16) = sc[g][rr];
    }
    if (threadIdx.x < MX_R && p0 + (int)threadIdx.x < TK)
        *(uint32_t *)(scales + ((size_t)q * TK + p0 + threadIdx.x) * 4) = ss[threadIdx.x];
}

// Grouped GEMM on v_mfma_scale_f32_32x32x64_f8f6f4 (A fp4, B fp8 E4M3).  Operand layout
// of the instruction (64 k a step): A lane l holds row l%32, k = 32*(l/32) .. +31 (16
// bytes, low nibble first) with that 32-k group's scale byte; B lane l holds column l%32,
// bytes 0-15 = k 16*(l/32) .. +15 and bytes 16-31 = k 32 + 16*(l/32) .. +15, and lane
// (j + 32b) gives column j's scale of 32-k group b; D as the 32x32x16 bf16 form.  A quad
// of 128 k is two steps whose A operands are pf_gemm32's two code loads and scale dwords
// (k groups 2*step + h).  Tile lists, XCD dealing, ring and barrier protocol as
// pf_gemm32; the B block in LDS: entry gq*NCOL + col = k16-group gq of the quad, column
// col; each lane keeps its column's scale dword per quad in registers.  The gate/up
// epilogue forms w * SiTU(gate, up) and quantises each 32-row block of a column (16
// values in each of two lanes) to MXFP8 codes and a scale byte.
template <int NMAT, int RT32, int CT, bool GU, int NW>
__global__ void __launch_bounds__(NW * WAVE) pf_gemm_mx(PfGemmArgs a)
{
    constexpr int NTH = NW * WAVE;
    constexpr int NCOL = CT * 32;
    constexpr int QB = 8 * NCOL * 16;
    constexpr int NJ = QB / (NTH * 16);
    constexpr int RING = 4;
    // loads a quad issues per wave (as pf_gemm32's, plus a scale dword per column tile)
    constexpr int LPI = NMAT * RT32 * 2 + NJ + CT;
    constexpr int LPS = LPI + NMAT * RT32 * 2;
    static_assert(NJ * NTH * 16 == QB, "B quad must split evenly");
    static_assert(LPI + LPS < 64, "vmcnt range");
    __shared__ __attribute__((aligned(16))) uint8_t sB[RING * QB];

    const int wave = wave_id(), lane = threadIdx.x % WAVE;
    int g, rb, ntok, p0;
    {
        const int ntiles = __builtin_amdgcn_readfirstlane(*a.ntile);
        const int per = (ntiles + 7) >> 3;
        const int k = blockIdx.x >> 3, tile = (blockIdx.x & 7) * per + k;
        if (k >= per || tile >= ntiles) return;
        const int4 d = a.desc[__builtin_amdgcn_readfirstlane(*a.dbase) + tile];
        g = __builtin_amdgcn_readfirstlane(d.x); rb = __builtin_amdgcn_readfirstlane(d.y);
        p0 = __builtin_amdgcn_readfirstlane(d.z); ntok = __builtin_amdgcn_readfirstlane(d.w);
    }
    const int nQ = a.K >> 7;

    const uint32_t tbytes = (uint32_t)fp4_tile_bytes(a.K);
    const int R16 = a.R >> 4;
    const int Rl = lane & 31, h = lane >> 5;
    rsrc_t ra[NMAT][RT32];
    int tp16[RT32];
#pragma unroll
    for (int i = 0; i < RT32; i++) {
        const int t16 = ((rb * NW + wave) * RT32 + i) * 2;
        tp16[i] = t16;
        const int ntl = __builtin_amdgcn_readfirstlane(R16 - t16 < 0 ? 0 : (R16 - t16 > 2 ? 2 : R16 - t16));
#pragma unroll
        for (int m = 0; m < NMAT; m++)
            ra[m][i] = make_rsrc(a.wm[m] + (size_t)g * a.gstride + (size_t)t16 * tbytes,
                                 (uint32_t)ntl * tbytes);
    }
    const uint32_t lc = (uint32_t)(Rl >> 4) * tbytes + (uint32_t)((Rl & 15) + 16 * h) * 16u;
    const uint32_t ls = (uint32_t)(Rl >> 4) * tbytes + 4096u + (uint32_t)((Rl & 15) + 16 * h) * 4u;

    // ---- B: entry e = (wave*NJ + j)*64 + lane = gq*NCOL + col
    const rsrc_t rbc = make_rsrc(a.b8, (uint32_t)((size_t)a.K * a.brows));
    const rsrc_t rbsc = make_rsrc(a.b8s, (uint32_t)((size_t)(a.K >> 7) * a.brows * 4));
    const uint32_t qstep = (uint32_t)a.brows * 128u, sstep = (uint32_t)a.brows * 4u;
    uint32_t boff[NJ], soff[CT];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int e = (wave * NJ + j) * WAVE + lane;
        const int gq = e / NCOL, col = e % NCOL;
        boff[j] = col < ntok ? ((uint32_t)gq * (uint32_t)a.brows + (uint32_t)(a.row_base + p0 + col)) * 16u
                             : K3X_OOB;
    }
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const int col = c * 32 + Rl;
        soff[c] = col < ntok ? (uint32_t)(a.row_base + p0 + col) * 4u : K3X_OOB;
    }

    struct AQ {
        u32x4    c[NMAT][RT32][2];
        uint32_t bs[CT];
    };
    AQ A[RING];
    uint32_t sn[NMAT][RT32][2], sc[NMAT][RT32][2];     // as in pf_gemm32
    auto ld = [&](int slot, int q) AI {
        const bool on = q < nQ;
        const uint32_t qc = (uint32_t)(q >> 2) * 4352u + (uint32_t)(q & 3) * 1024u;
        const uint32_t qs = (uint32_t)(q >> 2) * 4352u;
#pragma unroll
        for (int m = 0; m < NMAT; m++)
#pragma unroll
            for (int i = 0; i < RT32; i++)
#pragma unroll
                for (int gl = 0; gl < 2; gl++) {
                    A[slot].c[m][i][gl] = wld16(ra[m][i], on ? lc + qc + 512u * gl : K3X_OOB);
                    if (slot == 0) sn[m][i][gl] = wld4(ra[m][i], on ? ls + qs + 128u * gl : K3X_OOB);
                }
#pragma unroll
        for (int c = 0; c < CT; c++)
            A[slot].bs[c] = __builtin_amdgcn_raw_buffer_load_b32(
                rbsc, (!on | (soff[c] == K3X_OOB)) ? K3X_OOB : soff[c] + (uint32_t)q * sstep, 0, 0);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            // (bitwise, not short-circuit: a branch on the uniform `on` would split the
            // step into blocks, and the MFMAs would then sink past the next barriers)
            const uint32_t o = ((boff[j] == K3X_OOB) | !on) ? K3X_OOB : boff[j] + (uint32_t)q * qstep;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rbc, (lds_void *)(sB + slot * QB + (wave * NJ + j) * 1024), 16, o, 0, 0, 0);
        }
    };

    f32x16 acc[NMAT][RT32][CT];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < RT32; i++)
#pragma unroll
            for (int c = 0; c < CT; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[m][i][c][v] = 0.f;

    auto compute = [&](int slot, int q) AI {
        const uint8_t *bb = sB + slot * QB;
        const int sh = 8 * (q & 3);
        if (slot == 0) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < RT32; i++)
#pragma unroll
                    for (int gl = 0; gl < 2; gl++) sc[m][i][gl] = sn[m][i][gl];
        }
#pragma unroll
        for (int st = 0; st < 2; st++) {
            i32x8 bv[CT];
            int sbv[CT];
#pragma unroll
            for (int c = 0; c < CT; c++) {
                const u32x4 b0 = *(const u32x4 *)(bb + ((4 * st + h) * NCOL + c * 32 + Rl) * 16);
                const u32x4 b1 = *(const u32x4 *)(bb + ((4 * st + 2 + h) * NCOL + c * 32 + Rl) * 16);
                bv[c] = (i32x8){(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3],
                                (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
                sbv[c] = (int)((A[slot].bs[c] >> (8 * (2 * st + h))) & 255u);
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < RT32; i++) {
                    const u32x4 cw = A[slot].c[m][i][st];
                    const i32x8 av = {(int)cw[0], (int)cw[1], (int)cw[2], (int)cw[3], 0, 0, 0, 0};
                    const int sa = (int)((sc[m][i][st] >> sh) & 255u);
#pragma unroll
                    for (int c = 0; c < CT; c++)
                        acc[m][i][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                            av, bv[c], acc[m][i][c], 4, 0, 0, sa, 0, sbv[c]);
                }
        }
    };

#pragma unroll
    for (int s = 0; s < RING - 1; s++) {
        SCHED_FENCE();
        ld(s, s);
    }
    SCHED_FENCE();
    int q = 0;
    // meet quad q + s once the loads issued after its own are all that remain: those of
    // quads q + s + 1 and q + s + 2, of which q + 4 (the next super-quad's first) also
    // loads the scale dwords
    static_assert(RING == 4, "written for a ring of 4");
    for (; q + RING <= nQ; q += RING) {
        meet<2 * LPI>();       SCHED_FENCE(); ld(3, q + 3); SCHED_FENCE(); compute(0, q);
        meet<2 * LPI>();       SCHED_FENCE(); ld(0, q + 4); SCHED_FENCE(); compute(1, q + 1);
        meet<LPI + LPS>();     SCHED_FENCE(); ld(1, q + 5); SCHED_FENCE(); compute(2, q + 2);
        meet<LPS + LPI>();     SCHED_FENCE(); ld(2, q + 6); SCHED_FENCE(); compute(3, q + 3);
    }
    if (q < nQ)     { meet<2 * LPI>(); compute(0, q); }
    if (q + 1 < nQ) { meet<LPI>();     compute(1, q + 1); }
    if (q + 2 < nQ) { meet<0>();       compute(2, q + 2); }
    WAIT_VMCNT_LGKM0(0);

    // ---- epilogue: lane holds column Rl of each column tile, rows 8a + 4h + b
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const int tl = c * 32 + Rl;
        const bool writer = tl < ntok;
        const int p = p0 + tl;
#pragma unroll
        for (int i = 0; i < RT32; i++) {
            const int rt = tp16[i] * 16;              // first row of the 32-row tile
            if (GU) {
                const float w = writer && a.pw ? a.pw[p] : 1.0f;
                float yv[16];
                float m = 0.0f;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    yv[v] = (w == 0.0f) ? 0.0f : w * situ_call(acc[0][i][c][v], acc[NMAT - 1][i][c][v], a.b1, a.b2);
                    if (isfinite(yv[v])) m = fmaxf(m, fabsf(yv[v]));
                }
                m = fmaxf(m, __shfl_xor(m, 32));
                if (!writer || rt >= a.R) continue;
                const int sb = mx8_scale(m);
                const float inv = mx8_inv(sb);
#pragma unroll
                for (int aa = 0; aa < 4; aa++) {
                    const int r0 = rt + 8 * aa + 4 * h;
                    uint32_t wd = 0;
#pragma unroll
                    for (int b = 0; b < 4; b++) wd |= mx8_code(yv[4 * aa + b], inv) << (8 * b);
                    *(uint32_t *)(a.o8 + ((size_t)(r0 >> 4) * a.arows + (size_t)(a.out_base + p)) * 16 + (r0 & 15)) = wd;
                }
                if (h == 0) {
                    const int r32 = rt >> 5;
                    a.o8s[((size_t)(r32 >> 2) * a.arows + (size_t)(a.out_base + p)) * 4 + (r32 & 3)] = (uint8_t)sb;
                }
            } else {
                if (!writer) continue;
#pragma unroll
                for (int aa = 0; aa < 4; aa++) {
                    const int r0 = rt + 8 * aa + 4 * h;
                    if (r0 >= a.R) continue;
                    float *dst = a.y + (size_t)(a.out_base + p) * (a.ldy ? a.ldy : a.R) + r0;
                    *(f32x4 *)dst = (f32x4){acc[0][i][c][4 * aa], acc[0][i][c][4 * aa + 1],
                                            acc[0][i][c][4 * aa + 2], acc[0][i][c][4 * aa + 3]};
                }
            }
        }
    }
}

// ------------------------------------------------------------------ latent norm
// The latent form's aggregates (agg [T][X], one workgroup per token): RMSNorm with the
// latent norm weights (k3_rmsnorm, k3_ops.c:132-140 and :1946; double sum of squares, inv
// rounded to float, w*x*inv), or none when nw is NULL, then the hi and lo rows [2][T][X]
// for the up projection.
__global__ void __launch_bounds__(PF_NT) pf_latnorm(const float *agg, const float *nw, float eps,
                                                    int T, int X, uint16_t *hl)
{
    __shared__ double red[PF_NT / WAVE];
    __shared__ float s_inv;
    const int t = blockIdx.x, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const float *row = agg + (size_t)t * X;
    if (nw) {
        double ss = 0.0;
        for (int i = threadIdx.x; i < X; i += PF_NT) ss += (double)row[i] * (double)row[i];
        for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        if (threadIdx.x == 0) {
            double tot = 0.0;
            for (int w = 0; w < PF_NT / WAVE; w++) tot += red[w];
            s_inv = (float)(1.0 / sqrt(tot / (double)X + (double)eps));
        }
        __syncthreads();
    }
    const int G8 = X >> 3;
    for (int gi = threadIdx.x; gi < G8; gi += PF_NT) {
        float v[8];
        load_x8(row, 0, (size_t)gi * 8, v);
        if (nw) {
            float w[8];
            load_x8(nw, 0, (size_t)gi * 8, w);
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = w[j] * v[j] * s_inv;
        }
        uint32_t hi[8], lo[8];
#pragma unroll
        for (int j = 0; j < 8; j++) split_bf16(v[j], hi[j], lo[j]);
        u32x4 h, l;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            h[j] = hi[2 * j] | (hi[2 * j + 1] << 16);
            l[j] = lo[2 * j] | (lo[2 * j + 1] << 16);
        }
        *(u32x4 *)(hl + (size_t)t * X + (size_t)gi * 8) = h;
        *(u32x4 *)(hl + ((size_t)T + t) * X + (size_t)gi * 8) = l;
    }
}

// ------------------------------------------------------------------ combine
// out[t] = ((y[pos(t,0)] + y[pos(t,1)]) + ... ) + ysh[t], then + resid (pos_of NULL: K = 1
// and row t; ysh NULL: none).
__global__ void __launch_bounds__(PF_NT) pf_combine(const float *y, const int *pos_of, int T, int K,
                                                    int H, const float *ysh, const float *resid,
                                                    float *out)
{
    const size_t i = (size_t)blockIdx.x * PF_NT + threadIdx.x;
    const int h4 = H >> 2;
    if (i >= (size_t)T * h4) return;
    const int t = (int)(i / h4), h = (int)(i % h4) * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < K; j++) {
        const size_t row = pos_of ? (size_t)pos_of[(size_t)t * K + j] : (size_t)t;
        s += *(const f32x4 *)(y + row * H + h);
    }
    const size_t o = (size_t)t * H + h;
    if (ysh) s += *(const f32x4 *)(ysh + o);
    if (resid) s += *(const f32x4 *)(resid + o);
    *(f32x4 *)(out + o) = s;
}

// ------------------------------------------------------------------ launcher
static inline int launch_ok(void) { return hipGetLastError() == hipSuccess ? 0 : K3X_E_HIP; }

static inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

template <int NE>
static void launch_topk(const PfTopkArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(pf_topk<NE>, dim3(cdiv(a.r.T, TK_W)), dim3(TK_W * WAVE), 0, s, a);
}

// Launch shapes of the routed GEMMs (pf_gemm32): NW waves of RT 32-row tiles per workgroup
// and CT 32-column tiles, by class.  Class 0 holds the experts of one narrow column tile,
// class 1 those of two, class 2 the others (wide tiles: fewer re-reads of their weights and
// activations).  A gate/up of bf16 rows (one column a token) has no class 1: its single
// column tile holds 32 tokens.  Class 0 of the two-column products is for the small calls,
// whose experts have a few tokens each: with two column tiles for them half the matrix
// work, half the LDS reads and, at 64 KB of LDS, a third of the waves a CU were lost (the
// gate/up of 40 fp32 tokens 520 -> 400 us, of 130 latent ones 1919 -> 1380).
struct PfShape { int nw, rt, ct, minw; };
static constexpr PfShape GU1[PF_NC] = {{4, 2, 1, 2}, {4, 2, 1, 2}, {8, 1, 3, 2}};   // bf16 rows
static constexpr PfShape GU2[PF_NC] = {{4, 1, 1, 3}, {8, 1, 2, 2}, {8, 1, 3, 2}};   // hi and lo columns
static constexpr PfShape DN[PF_NC] = {{4, 2, 1, 3}, {4, 2, 2, 2}, {8, 2, 3, 2}};
// Classes 0 and 1 and class 2 run on two streams, gate/up then down with no event between
// them: an expert has to be of class 2 in both products or in neither.
static_assert(GU1[1].ct * 32 == DN[1].ct * 16 && GU2[1].ct * 16 == DN[1].ct * 16,
              "the most tokens of class 1 differ between gate/up and down");

template <bool EXACT, int HL, int C>
static void launch_gu(const PfGemmArgs &a, unsigned grid, hipStream_t s)
{
    constexpr PfShape p = HL == 1 ? GU1[C] : GU2[C];
    hipLaunchKernelGGL((pf_gemm32<EXACT, 2, p.rt, p.ct, HL, true, p.nw, p.minw>), dim3(grid),
                       dim3(p.nw * WAVE), 0, s, a);
}

template <bool EXACT, int C>
static void launch_dn(const PfGemmArgs &a, unsigned grid, hipStream_t s)
{
    constexpr PfShape p = DN[C];
    hipLaunchKernelGGL((pf_gemm32<EXACT, 1, p.rt, p.ct, 2, false, p.nw, p.minw>), dim3(grid),
                       dim3(p.nw * WAVE), 0, s, a);
}

// MXFP8 mode tiles: small class 32 tokens, large class 64; four waves a workgroup, gate/up
// 128 rows (one 32-row tile a wave), down 256 (two)
#define MX_GU_RT32 1
#define MX_DN_RT32 2
#define MX_CT_S 1
#define MX_CT_B 2
#define MX_NW   4
#ifndef MX_GU_RT32_S
#define MX_GU_RT32_S 1     // 32-row tiles a wave, small-class gate/up
#endif
#ifndef MX_DN_RT32_S
#define MX_DN_RT32_S 2     // the same, small-class down
#endif

static inline unsigned round8(size_t n) { return (unsigned)((n + 7) & ~(size_t)7); }

// stages of the dense GEMM's LDS ring (32 KB each): two, so that two workgroups share a
// CU (measured at 2048 x 7168 x 7168: 325 us, against 371 with three stages and 365 with
// four, one workgroup a CU)
#define DENSE_NS 2
// wave tiles (32 x 32 MFMA tiles per wave, four waves as 2 x 2): the gate/up products,
// and the single-matrix ones
#define DENSE_GU_RW 1
#define DENSE_GU_CW 2
#define DENSE_RW    2
#define DENSE_CW    2

static int launch_rows(const void *x, int x_bf16, int T, int n, int ldx, uint16_t *hl, hipStream_t s)
{
    hipLaunchKernelGGL(pf_rows, dim3(cdiv((size_t)T * (n >> 3), PF_NT)), dim3(PF_NT), 0, s, x, x_bf16,
                       T, n, ldx, hl);
    return launch_ok();
}

// A dense product on pf_dense: NMAT matrices of R rows over a.n0 B rows, HL B columns per
// row (1: bf16 activations, 2: hi and lo parts of fp32 ones)
template <int NMAT, int RW, int CW, bool GU>
static void launch_dense(const PfGemmArgs &a, int HL, hipStream_t s)
{
    const int BM = 2 * RW * 32, BN = 2 * CW * 32;
    const unsigned grid = round8((size_t)cdiv(a.R, BM) * cdiv(a.n0, BN / HL));
    if (HL == 1)
        hipLaunchKernelGGL((pf_dense<NMAT, RW, CW, 1, GU, DENSE_NS>), dim3(grid), dim3(PF_NT), 0, s, a);
    else
        hipLaunchKernelGGL((pf_dense<NMAT, RW, CW, 2, GU, DENSE_NS>), dim3(grid), dim3(PF_NT), 0, s, a);
}

// Rows per expert on average (T K / E) below which a call runs every expert in class 0's
// shape, a larger one in several column blocks (their weights then come from the L2 again),
// on one stream: a second and third launch each end in a tail of a few workgroups, and the
// wide tiles' workgroups, launched on another stream, find no free CU among class 0's until
// those end.  (us a call with three classes and with one, K2 shape: 40 fp32 tokens, 0.8 rows
// an expert, 759 and 665; 100 of bf16, 2.1 rows, 1142 and 1147; 180, 3.8 rows, 1439 and 1475,
// of fp32 1456 and 1457; 250, 5.2 rows, 1542 and 1587; 350 of fp32, 7.3 rows, 1779 and 1852.
// 40 latent tokens, 0.7 rows, 1368 and 1300; 130, 2.3 rows, 2400 and 2358; 440, 7.9 rows, 3426
// and 3493.  MXFP8 mode, whose class 2 runs on the same stream: 40 tokens 736 and 688, 120
// 1242 and 1226, 180 1446 and 1455, 300 1587 and 1634.)
#define PF_ONE_ROWS 4
// and from which class 2's products are the longer part (us a call with them on the caller's
// stream and on the side stream, K2 shape, bf16 rows: 14.6 rows 2082 and 2030, 17.7 2231 and
// 2297, 20.8 2338 and 2407, 25 2530 and 2612, 29 2636 and 2672, 35 2940 and 3027, 42.7 3229
// and 3301; fp32 rows within 1%.  Latent: 19.6 rows 4994 and 4984, 28.6 6339 and 6432, 36.6
// 7426 and 7572.)
#define PF_BIG_ROWS 20

template <int NTT>
static void launch_router(const PfRouterArgs &a, hipStream_t s)
{
    const dim3 grid(cdiv(a.E, RM_E) * cdiv(a.T, 16 * NTT) * (unsigned)a.sg);
    if (a.x_bf16) hipLaunchKernelGGL((pf_router<NTT, true>), grid, dim3(RM_NT), 0, s, a);
    else          hipLaunchKernelGGL((pf_router<NTT, false>), grid, dim3(RM_NT), 0, s, a);
}

// Router and top-k of T rows: idx and wt, copies in uidx and uwt, the histogram in counts
// (all three may be NULL).
static int route_rows(k3x_moe_layer *L, const k3x_prefill_buf *B, const void *x, int x_bf16, int T,
                      int *idx, float *wt, int *uidx, float *uwt, int *counts, hipStream_t s)
{
    const k3x_cfg *c = &L->cfg;
    const int H = c->hidden, E = c->n_experts, K = c->topk;
    const int ntt = T <= 16 ? 1 : 2;
    PfTopkArgs at;
    PfRouterArgs &ar = at.r;
    ar.x = x; ar.x_bf16 = x_bf16; ar.W = L->router; ar.T = T; ar.H = H; ar.E = E;
    // workgroups along K: up to three a CU (the LDS holds three), each wave at least one
    // chunk; the parts' sums and bounds lie where the MXFP8 mode's codes are written after
    // the top-k.  Past one tile a CU, the number of up to four whose last round of workgroups
    // over the CUs is the fullest, a part's store and load (12 bytes an output) weighed
    // against its products: with one workgroup a tile there 1500 tokens x 384 experts took
    // the three rounds of 2048 (a routing call 250 us, now 208; 600 x 896 255, now 212)
    const unsigned tiles = cdiv(E, RM_E) * cdiv(T, 16 * ntt);
    int sg = tiles < 768u / RM_SGMAX ? RM_SGMAX : (int)(768u / tiles);
    if (tiles > 256u) {
        double best = 0.0;
        for (int q = 1; q <= 4; q++) {
            const double cost = (double)cdiv((size_t)tiles * q, 256) / q + (q > 1 ? 8e-5 * tiles * q : 0.0);
            if (q == 1 || cost < best) { best = cost; sg = q; }
        }
    }
    if (sg > H / RM_KC / RM_NW) sg = H / RM_KC / RM_NW;
    const size_t room = k3x_pf_xp_bytes(L, T) / ((size_t)T * E * 12);
    if ((size_t)sg > room) sg = (int)room;
    ar.sg = sg < 1 ? 1 : sg;
    ar.logit = B->logit; ar.gap = B->gap;
    ar.psum = (double *)B->xp;
    ar.pbnd = (float *)(ar.psum + (size_t)ar.sg * T * E);
    ar.counts = counts;
    if (ntt == 1) launch_router<1>(ar, s);
    else          launch_router<2>(ar, s);
    int rc = launch_ok();
    if (rc) return rc;
    at.bias = L->bias; at.K = K; at.renorm = c->moe_renorm; at.routed_scale = c->routed_scale;
    at.idx = idx; at.wt = wt; at.uidx = uidx; at.uwt = uwt;
    if (E <= 128)      launch_topk<2>(at, s);
    else if (E <= 256) launch_topk<4>(at, s);
    else if (E <= 384) launch_topk<6>(at, s);
    else if (E <= 512) launch_topk<8>(at, s);
    else               launch_topk<16>(at, s);
    return launch_ok();
}

static int pf_chunk(k3x_moe_layer *L, const k3x_prefill_buf *B, float *out, const void *x,
                    int x_dtype, int T, const float *resid, int *uidx, float *uwt,
                    hipStream_t s)
{
    const k3x_cfg *c = &L->cfg;
    const int H = c->hidden, E = c->n_experts, K = c->topk, I = c->moe_inter, SI = L->SI;
    const int X = L->XL;                                 // the routed experts' width
    const int TK = T * K;
    const int x_bf16 = (x_dtype == K3X_BF16);
    const int HLg = x_bf16 ? 1 : 2;                      // B columns per token of x
    const int HLr = L->lat ? 2 : HLg;                    // of the routed gate/up input
    int rc;

    // x's rows as the GEMMs read them
    const uint16_t *xr = (const uint16_t *)x;
    if (!x_bf16) {
        if ((rc = launch_rows(x, 0, T, H, H, B->xhl, s))) return rc;
        xr = B->xhl;
    }

    // The layer's side stream runs beside s: z = down . x in the latent form and the shared
    // expert (bf16 weights, every token), which need only x's rows, and the part of the
    // routed products that is not on s.  pf_dense's workgroups, two a CU, let the router and
    // the top-k in beside them: z and then a pf_dense shared expert are forked before those
    // (z here against on s before the routed products: 16 latent tokens 677 and 680 us, of fp32
    // 726 and 744, 130 2354 and 2372, 600 and 2048 within 0.6%).  The library's kernels hold
    // every CU while they run, so that the top-k would wait for a free one: a library shared
    // expert is forked after it (before it, 3 to 5% more at 2048 tokens when the routed input was
    // still gathered), and after the small
    // classes' products where those are on the side stream (there against before them: 1000
    // tokens 2333 and 2344 us, 1400 2630 and 2667, 2048 3239 and 3234).
    // Its T output rows (H floats each) lie in y past the TK routed rows (X floats each) and
    // past rows of H floats, which the latent form's up projection writes: X may be the wider.
    float *const ysh = B->y + (size_t)TK * (X > H ? X : H);
    bool forked = false;
    // The library path (bf16 rows, 2*SI <= H, a kernel for each shape): the gate/up product
    // into fp32 rows [T][2*SI] held in the shared rows of y (nothing else writes them before
    // the down product, which overwrites them), SiTU into bf16 hi and lo rows [T][SI] (in
    // act_sh), then the down product as two GEMMs, hi then lo accumulated, into the shared
    // rows of y.
    const bool lib = L->blas && !B->no_lib;
    const bool sh_blas = SI > 0 && lib && L->sh_gu_rm && x_bf16 &&
                         k3x_blas_ready(L->device, H, 2 * SI, T, 0) == 0 &&
                         k3x_blas_ready(L->device, SI, H, T, 0) == 0 &&
                         k3x_blas_ready(L->device, SI, H, T, 1) == 0;
    hipStream_t side = (hipStream_t)L->pf_side;
    // the side stream behind what s holds so far
    auto fork = [&]() -> int {
        if (hipEventRecord((hipEvent_t)L->pf_ev[0], s) != hipSuccess ||
            hipStreamWaitEvent(side, (hipEvent_t)L->pf_ev[0], 0) != hipSuccess)
            return K3X_E_HIP;
        forked = true;
        return 0;
    };
    // s behind everything on the side stream
    auto join = [&]() -> int {
        if (!forked) return 0;
        forked = false;
        return hipEventRecord((hipEvent_t)L->pf_ev[1], side) == hipSuccess &&
                       hipStreamWaitEvent(s, (hipEvent_t)L->pf_ev[1], 0) == hipSuccess
                   ? 0
                   : K3X_E_HIP;
    };
    // from the fork on, a failed launch joins the side stream before it returns
#define PF_RET(e) do { const int e_ = (e); (void)join(); return e_; } while (0)
    auto shared = [&]() -> int {
        if (sh_blas) {
            uint16_t *ahi = B->act_sh, *alo = B->act_sh + (size_t)T * SI;
            int r = k3x_blas_gemm_bf16(L->device, L->sh_gu_rm, H, 2 * SI, ysh, 2 * SI,
                                       (const uint16_t *)x, H, T, 0, side);
            if (!r) r = k3x_dev_glu_rows(ysh, T, SI, L->b1, L->b2, ahi, alo, side);
            if (!r) r = k3x_blas_gemm_bf16(L->device, L->sh_down_rm, SI, H, ysh, H, ahi, SI, T, 0,
                                           side);
            if (!r) r = k3x_blas_gemm_bf16(L->device, L->sh_down_rm, SI, H, ysh, H, alo, SI, T, 1,
                                           side);
            return r;
        }
        PfGemmArgs sg;
        memset(&sg, 0, sizeof sg);
        sg.wm[0] = (const uint8_t *)L->sh_gate; sg.wm[1] = (const uint8_t *)L->sh_up;
        sg.R = SI; sg.K = H; sg.n0 = T;
        sg.bsrc = xr; sg.brows = T; sg.ldb = H; sg.row_base = 0;
        sg.act = B->act_sh; sg.arows = T; sg.out_base = 0;
        sg.b1 = L->b1; sg.b2 = L->b2;
        launch_dense<2, DENSE_GU_RW, DENSE_GU_CW, true>(sg, HLg, side);
        int r = launch_ok();
        if (r) return r;
        PfGemmArgs sd;
        memset(&sd, 0, sizeof sd);
        sd.wm[0] = (const uint8_t *)L->sh_down; sd.R = H; sd.K = SI; sd.n0 = T;
        sd.bsrc = B->act_sh; sd.brows = T; sd.ldb = SI; sd.row_base = 0;
        sd.y = ysh; sd.out_base = 0;
        launch_dense<1, DENSE_RW, DENSE_CW, false>(sd, 2, side);
        return launch_ok();
    };
    // z = down . x for every token (k3_mmw_batch, k3_ops.c:1871): a plain product, on the
    // library where it serves the shape (bf16 rows), else the dense kernel
    auto zdown = [&](hipStream_t st) -> int {
        if (lib && x_bf16 && k3x_blas_ready(L->device, H, X, T, 0) == 0)
            return k3x_blas_gemm_bf16(L->device, L->ldown_rm, H, X, B->zf, X, (const uint16_t *)x, H,
                                      T, 0, st);
        PfGemmArgs zg;
        memset(&zg, 0, sizeof zg);
        zg.wm[0] = (const uint8_t *)L->ldown; zg.R = X; zg.K = H; zg.n0 = T;
        zg.bsrc = xr; zg.brows = T; zg.ldb = H; zg.row_base = 0;
        zg.y = B->zf; zg.out_base = 0;
        launch_dense<1, DENSE_RW, DENSE_CW, false>(zg, HLg, st);
        return launch_ok();
    };
    const bool mx = L->pf_mode == K3X_PREFILL_MXFP8;
    const bool big_first = TK >= PF_BIG_ROWS * E;
    const bool sh_last = SI > 0 && sh_blas && !mx && big_first;
    const bool zside = L->lat && SI > 0;
    if (zside) {
        if ((rc = fork()) || (rc = zdown(side))) PF_RET(rc);
        if (hipEventRecord((hipEvent_t)L->pf_ev[2], side) != hipSuccess) PF_RET(K3X_E_HIP);
    }
    if (SI > 0 && !sh_blas && ((rc = forked ? 0 : fork()) || (rc = shared()))) PF_RET(rc);
    if ((rc = route_rows(L, B, x, x_bf16, T, B->idx, B->wt, uidx, uwt, B->counts, s))) PF_RET(rc);
    if (SI > 0 && sh_blas && !sh_last && ((rc = fork()) || (rc = shared()))) PF_RET(rc);

    PfScanArgs sa;
    sa.counts = B->counts; sa.E = E; sa.offsets = B->offsets; sa.cursor = B->cursor;
    sa.tb[0] = B->tb_gu; sa.tb[1] = B->tb_dn;
    // calls of few tokens an expert: one class for all (see PF_ONE_ROWS)
    const bool one = TK < PF_ONE_ROWS * E;
    const PfShape mgu[PF_NC] = {{MX_NW, MX_GU_RT32_S, MX_CT_S, 0}, {MX_NW, MX_GU_RT32_S, MX_CT_S, 0},
                                {MX_NW, MX_GU_RT32, MX_CT_B, 0}};
    const PfShape mdn[PF_NC] = {{MX_NW, MX_DN_RT32_S, MX_CT_S, 0}, {MX_NW, MX_DN_RT32_S, MX_CT_S, 0},
                                {MX_NW, MX_DN_RT32, MX_CT_B, 0}};
    const PfShape *shp[2] = {mx ? mgu : (HLr == 1 ? GU1 : GU2), mx ? mdn : DN};
    for (int q = 0; q < PF_NC; q++)
        for (int m = 0; m < 2; m++) {
            const PfShape &p = shp[m][q];
            sa.tpb[m][q] = p.ct * 32 / (mx ? 1 : (m ? 2 : HLr));
            sa.nrb[m][q] = cdiv(m ? X : I, p.nw * p.rt * 32);
            if (q < 2) sa.lim[m][q] = one ? TK : sa.tpb[m][q];
        }
    // grids: upper bounds of each class (an expert of class 0 or 1 has one column block;
    // at most TK / (t + 1) experts have more than t tokens); surplus workgroups leave at
    // once
    unsigned grid[2][PF_NC];
    for (int m = 0; m < 2; m++) {
        const size_t ne = E < TK ? E : TK;
        size_t n[PF_NC] = {ne, (size_t)TK / (sa.lim[m][0] + 1), (size_t)TK / (sa.lim[m][1] + 1)};
        for (int q = 1; q < PF_NC; q++) n[q] = n[q] < ne ? n[q] : ne;
        if (sa.lim[m][1] == sa.lim[m][0]) n[1] = 0;
        size_t tiles = 0;
        for (int q = 0; q < PF_NC; q++) {
            if (n[q] && (q == 2 || sa.lim[m][q] > sa.tpb[m][q])) n[q] += cdiv(TK, sa.tpb[m][q]);
            tiles += sa.nrb[m][q] * n[q];
            grid[m][q] = round8(sa.nrb[m][q] * n[q]);
        }
        // (before any descriptor is written.  The table counts a column block per 16 rows and
        // one more per expert, each of ceil(rows / 64) row blocks, where a class has at least
        // 16 rows a column block and 128 a row block: the bound stays below it)
        if (tiles > (size_t)(m ? B->ndesc_dn : B->ndesc_gu)) PF_RET(K3X_E_SHAPE);
    }

    hipLaunchKernelGGL(pf_scan, dim3(1), dim3(1024), 0, s, sa);
    if ((rc = launch_ok())) PF_RET(rc);
    hipLaunchKernelGGL(pf_scatter, dim3(cdiv(TK, PF_NT)), dim3(PF_NT), 0, s, B->idx, B->wt, TK, K,
                       E, B->offsets, B->cursor, B->perm_tok, B->perm_w, B->pos_of);
    if ((rc = launch_ok())) PF_RET(rc);
    hipLaunchKernelGGL(pf_tiles, dim3(E), dim3(PF_NT), 0, s, B->counts, B->offsets, sa,
                       (int4 *)B->desc_gu, (int4 *)B->desc_dn);
    if ((rc = launch_ok())) PF_RET(rc);
    if (zside) {
        if (hipStreamWaitEvent(s, (hipEvent_t)L->pf_ev[2], 0) != hipSuccess) PF_RET(K3X_E_HIP);
    } else if (L->lat && (rc = zdown(s))) {
        PF_RET(rc);
    }
    // MXFP8 mode: the routed input quantised in permuted order, codes then scales in xp;
    // the gate/up output's codes then scales in act
    uint8_t *xq8 = B->xp, *xs8 = xq8 + (((size_t)TK * X + 255) & ~(size_t)255);
    uint8_t *aq8 = (uint8_t *)B->act, *as8 = aq8 + (((size_t)TK * I + 255) & ~(size_t)255);
    if (mx) {
        const void *src = L->lat ? (const void *)B->zf : x;
        hipLaunchKernelGGL(pf_mx8_rows, dim3(pf_mx8_grid(TK, X)), dim3(PF_NT), 0, s,
                           src, L->lat ? 0 : x_bf16, X, X, B->perm_tok, TK, xq8, xs8);
        if ((rc = launch_ok())) PF_RET(rc);
    } else if (L->lat) {
        // z's hi and lo rows (zhl holds the normalised aggregates' only after the GEMMs)
        if ((rc = launch_rows(B->zf, 0, T, X, X, B->zhl, s))) PF_RET(rc);
    }

    // routed gate/up: B rows are the tokens' rows, through the permutation
    PfGemmArgs g;
    memset(&g, 0, sizeof g);
    g.wm[0] = L->experts + L->gate_off; g.wm[1] = L->experts + L->up_off;
    g.gstride = L->expert_bytes;
    g.R = I; g.K = X; g.desc = (const int4 *)B->desc_gu;
    g.bsrc = L->lat ? B->zhl : xr; g.brows = T; g.ldb = X; g.perm = B->perm_tok; g.row_base = 0;
    g.pw = B->perm_w; g.act = B->act; g.arows = TK; g.out_base = 0;
    g.b1 = L->b1; g.b2 = L->b2;
    const bool ex_gu = (L->special & 3) != 0;
    if (mx) {
        g.brows = TK;
        g.b8 = xq8; g.b8s = (const uint32_t *)xs8; g.o8 = aq8; g.o8s = as8;
    }
    // routed down: B rows are the activation rows, in permuted order
    PfGemmArgs d;
    memset(&d, 0, sizeof d);
    d.wm[0] = L->experts + L->down_off; d.gstride = L->expert_bytes;
    d.R = X; d.K = I; d.desc = (const int4 *)B->desc_dn;
    d.bsrc = B->act; d.brows = TK; d.ldb = I; d.perm = NULL; d.row_base = 0;
    d.y = B->y; d.out_base = 0;
    if (mx) { d.b8 = aq8; d.b8s = (const uint32_t *)as8; }
    const bool ex_dn = (L->special & 4) != 0;
    // class q's tiles of the gate/up (m = 0) or the down GEMM on stream st
    auto gemm = [&](int m, int q, hipStream_t st) -> int {
        const unsigned gr = grid[m][q];
        if (!gr) return 0;
        PfGemmArgs &p = m ? d : g;
        p.ntile = (m ? B->tb_dn : B->tb_gu) + E + 2 * q;
        p.dbase = p.ntile + 1;
        if (mx && !m) {
            if (q == 2) hipLaunchKernelGGL((pf_gemm_mx<2, MX_GU_RT32, MX_CT_B, true, MX_NW>), dim3(gr), dim3(MX_NW * WAVE), 0, st, p);
            else        hipLaunchKernelGGL((pf_gemm_mx<2, MX_GU_RT32_S, MX_CT_S, true, MX_NW>), dim3(gr), dim3(MX_NW * WAVE), 0, st, p);
        } else if (mx) {
            if (q == 2) hipLaunchKernelGGL((pf_gemm_mx<1, MX_DN_RT32, MX_CT_B, false, MX_NW>), dim3(gr), dim3(MX_NW * WAVE), 0, st, p);
            else        hipLaunchKernelGGL((pf_gemm_mx<1, MX_DN_RT32_S, MX_CT_S, false, MX_NW>), dim3(gr), dim3(MX_NW * WAVE), 0, st, p);
        } else if (m) {
            if (q == 0)      ex_dn ? launch_dn<true, 0>(p, gr, st) : launch_dn<false, 0>(p, gr, st);
            else if (q == 1) ex_dn ? launch_dn<true, 1>(p, gr, st) : launch_dn<false, 1>(p, gr, st);
            else             ex_dn ? launch_dn<true, 2>(p, gr, st) : launch_dn<false, 2>(p, gr, st);
        } else if (HLr == 1) {
            if (q == 0)      ex_gu ? launch_gu<true, 1, 0>(p, gr, st) : launch_gu<false, 1, 0>(p, gr, st);
            else if (q == 1) ex_gu ? launch_gu<true, 1, 1>(p, gr, st) : launch_gu<false, 1, 1>(p, gr, st);
            else             ex_gu ? launch_gu<true, 1, 2>(p, gr, st) : launch_gu<false, 1, 2>(p, gr, st);
        } else {
            if (q == 0)      ex_gu ? launch_gu<true, 2, 0>(p, gr, st) : launch_gu<false, 2, 0>(p, gr, st);
            else if (q == 1) ex_gu ? launch_gu<true, 2, 1>(p, gr, st) : launch_gu<false, 2, 1>(p, gr, st);
            else             ex_gu ? launch_gu<true, 2, 2>(p, gr, st) : launch_gu<false, 2, 2>(p, gr, st);
        }
        return launch_ok();
    };
    // In the exact mode the products of classes 0 and 1 and those of class 2 run on two
    // streams, s and the side stream (forked here, after the routed input is written; joined
    // before the combine), the longer of the two on s.  What that gains is the launches' tails,
    // 2 to 6%: a wide workgroup and a narrow one do not share a CU (252 registers of the wide
    // tile's eight waves fill it), so that side by side the two parts take about the sum of
    // their times.  (Two streams against one, K2 shape, bf16 rows: 250 tokens 1540 and 1641 us,
    // 700 2019 and 2145, 1000 2338 and 2384, 2048 3226 and 3300, 4096 5543 and 5459; latent 300
    // 3090 and 3180, 1100 4986 and 5111, 2048 7427 and 7492.)  The MXFP8 products, all on tiles
    // of four waves, measured slower that way and stay on s.
    const bool split = SI > 0 && !mx && !one;
    hipStream_t st[2] = {s, s};                          // classes 0 and 1, class 2
    if (split) {
        if ((rc = fork())) PF_RET(rc);
        st[big_first ? 0 : 1] = side;
    }
    // issued longest first, gate/up before the down that reads it; on one stream every
    // gate/up first
    if (split) {
        const int order[2][3] = {{0, 1, 2}, {2, 0, 1}};
        for (int m = 0; m < 2 && !rc; m++)
            for (int q = 0; q < PF_NC && !rc; q++) {
                const int k = order[big_first][q];
                rc = gemm(m, k, st[k == 2]);
            }
    } else {
        for (int m = 0; m < 2 && !rc; m++)
            for (int q = PF_NC - 1; q >= 0 && !rc; q--) rc = gemm(m, q, s);
    }
    if (!rc && sh_last) rc = shared();
    if (rc) PF_RET(rc);
    if (split && L->lat && (rc = join())) return rc;     // every routed row is in y

    const int *pos = B->pos_of;
    int KC = K;
    if (L->lat) {
        // the routed aggregates in top-k order (:1941-1942), their RMSNorm's hi and lo rows
        // (:1946), then the up projection (:1950) into y rows 0 .. T-1
        hipLaunchKernelGGL(pf_combine, dim3(cdiv((size_t)T * (X / 4), PF_NT)), dim3(PF_NT), 0, s,
                           B->y, B->pos_of, T, K, X, (const float *)NULL, (const float *)NULL,
                           B->zf);
        if ((rc = launch_ok())) PF_RET(rc);
        // the up projection: a plain product over the normalised aggregates' hi and lo
        // rows, on the library where it serves the shapes, else the dense kernel
        const bool up_blas = lib && k3x_blas_ready(L->device, X, H, T, 0) == 0 &&
                             k3x_blas_ready(L->device, X, H, T, 1) == 0;
        hipLaunchKernelGGL(pf_latnorm, dim3(T), dim3(PF_NT), 0, s, B->zf,
                           c->latent_norm ? L->lnw : (const float *)NULL, c->rms_eps, T, X, B->zhl);
        if ((rc = launch_ok())) PF_RET(rc);
        if (up_blas) {
            if ((rc = k3x_blas_gemm_bf16(L->device, L->lup_rm, X, H, B->y, H, B->zhl, X, T, 0,
                                         s)) ||
                (rc = k3x_blas_gemm_bf16(L->device, L->lup_rm, X, H, B->y, H,
                                         B->zhl + (size_t)T * X, X, T, 1, s)))
                PF_RET(rc);
        } else {
            PfGemmArgs ug;
            memset(&ug, 0, sizeof ug);
            ug.wm[0] = (const uint8_t *)L->lup; ug.R = H; ug.K = X; ug.n0 = T;
            ug.bsrc = B->zhl; ug.brows = T; ug.ldb = X; ug.row_base = 0;
            ug.y = B->y; ug.out_base = 0;
            launch_dense<1, DENSE_RW, DENSE_CW, false>(ug, 2, s);
            if ((rc = launch_ok())) PF_RET(rc);
        }
        pos = NULL;
        KC = 1;
    }
    // the shared rows (and the side stream's routed ones) are in y
    if ((rc = join())) return rc;

    hipLaunchKernelGGL(pf_combine, dim3(cdiv((size_t)T * (H / 4), PF_NT)), dim3(PF_NT), 0, s,
                       B->y, pos, T, KC, H, SI > 0 ? ysh : (const float *)NULL, resid, out);
    return launch_ok();
}
#undef PF_RET

// Prefill: the pipeline over chunks of up to K3X_PF_CHUNK tokens.  Each token's result
// depends only on its own routing, so the chunking changes no result.
extern "C" int k3x_dev_prefill(k3x_moe_layer *L, float *out, const void *x, int x_dtype,
                               int T, const float *resid, int *idx, float *wt, void *stream)
{
    const int H = L->cfg.hidden, K = L->cfg.topk;
    const size_t es = (x_dtype == K3X_BF16) ? 2 : 4;
    const int chunk = k3x_pf_chunk_tokens(L);
    int rc = k3x_pf_reserve(L, T, stream);
    if (rc) return rc;
    for (int t0 = 0; t0 < T; t0 += chunk) {
        const int n = T - t0 < chunk ? T - t0 : chunk;
        rc = pf_chunk(L, &L->pf, out + (size_t)t0 * H, (const char *)x + (size_t)t0 * H * es, x_dtype, n,
                      resid ? resid + (size_t)t0 * H : NULL, idx ? idx + (size_t)t0 * K : NULL,
                      wt ? wt + (size_t)t0 * K : NULL, (hipStream_t)stream);
        if (rc) return rc;
    }
    return 0;
}

// The router alone (k3x_moe_route): per chunk, pf_router and each token's top-k into the
// caller's arrays (pf_topk, no histogram).
extern "C" int k3x_dev_route(k3x_moe_layer *L, int *idx, float *wt, const void *x, int x_dtype,
                             int T, void *stream)
{
    const int H = L->cfg.hidden, K = L->cfg.topk;
    const size_t es = (x_dtype == K3X_BF16) ? 2 : 4;
    const int chunk = k3x_pf_chunk_tokens(L);
    hipStream_t s = (hipStream_t)stream;
    int rc = k3x_pf_reserve(L, T, stream);
    if (rc) return rc;
    for (int t0 = 0; t0 < T; t0 += chunk) {
        const int n = T - t0 < chunk ? T - t0 : chunk;
        if ((rc = route_rows(L, &L->pf, (const char *)x + (size_t)t0 * H * es, x_dtype == K3X_BF16, n,
                             idx + (size_t)t0 * K, wt + (size_t)t0 * K, NULL, NULL, NULL, s)))
            return rc;
    }
    return 0;
}

// ------------------------------------------------------------------ without allocation
// The prefill pipeline for callers that cannot allocate (graph capture, serving loops):
// its working buffers come from this static device array instead of the layer's. Each
// device holds its own copy at its own address, found once per device by
// hipGetSymbolAddress; host code uses that address, never the array's name.  Every call
// on a device shares the device's copy (calls that overlap on one device race); no
// kernel needs it to start cleared (the histogram is zeroed by pf_router each run).
static __device__ __align__(256) uint8_t scratch[K3X_NOALLOC_BYTES];

#define K3X_MAX_DEVICES 64
static void *g_scratch[K3X_MAX_DEVICES];
static std::mutex g_scratch_mu;

static void *scratch_ptr(int device)
{
    if (device < 0 || device >= K3X_MAX_DEVICES) return NULL;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[device]) {
        void *p = NULL;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            fprintf(stderr, "k3x: hipGetSymbolAddress(scratch) on device %d failed: %s\n",
                    device, hipGetErrorString(e));
            return NULL;
        }
        g_scratch[device] = p;
    }
    return g_scratch[device];
}

extern "C" int k3x_dev_prefill_noalloc(k3x_moe_layer *L, float *out, const void *x, int x_dtype,
                                       int T, const float *resid, int *idx, float *wt,
                                       void *stream)
{
    const int chunk = k3x_pf_chunk_tokens(L);
    // the limit on T as it is published: fp32 rows of every (token, slot) counted for xp
    const size_t need = k3x_pf_layout(L, T, NULL, NULL) -
                        ((k3x_pf_xp_bytes(L, T) + 255) & ~(size_t)255) + k3x_pf_xp_rows(L, T);
    if (T > chunk || need > K3X_NOALLOC_BYTES) {
        fprintf(stderr, "k3x: a prefill of %d tokens needs %zu bytes of working memory; the "
                        "static array holds %u (and one run at most %d tokens)\n",
                T, need, K3X_NOALLOC_BYTES, chunk);
        return K3X_E_SHAPE;
    }
    if (hipSetDevice(L->device) != hipSuccess) return K3X_E_HIP;
    void *p = scratch_ptr(L->device);
    if (!p) return K3X_E_HIP;
    k3x_prefill_buf B;
    memset(&B, 0, sizeof B);
    k3x_pf_layout(L, T, (char *)p, &B);
    B.no_lib = 1;
    return pf_chunk(L, &B, out, x, x_dtype, T, resid, idx, wt, (hipStream_t)stream);
}

// ------------------------------------------------------------------ trunk products
// Y[t*ldy + o] = W[o] . X[t*ldx] for T activation rows (k3_mmw_batch_ld): X's rows, hi
// then lo, into `planes` (T * in * 4 bytes), then the dense bf16 GEMM.
extern "C" int k3x_dev_trunk_gemm(const uint16_t *W, int in, int out, float *y, int ldy,
                                  const void *x, int x_dtype, int ldx, int T, uint16_t *planes,
                                  void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int x_bf16 = (x_dtype == K3X_BF16), HL = x_bf16 ? 1 : 2;
    int rc = launch_rows(x, x_bf16, T, in, ldx, planes, s);
    if (rc) return rc;
    PfGemmArgs g;
    memset(&g, 0, sizeof g);
    g.wm[0] = (const uint8_t *)W; g.R = out; g.K = in; g.n0 = T;
    g.bsrc = planes; g.brows = T; g.ldb = in; g.row_base = 0;
    g.y = y; g.out_base = 0; g.ldy = ldy;
    launch_dense<1, DENSE_RW, DENSE_CW, false>(g, HL, s);
    return launch_ok();
}
