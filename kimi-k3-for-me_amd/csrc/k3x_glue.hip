// k3x_glue.hip - the decoder layer's glue around the MoE block: the block attention-
// residual aggregation (k3_attn_res, k3_ops.c:1722-1753, with a block count per call or
// per row as k3_decoder_layer_core takes them, :2481-2493) and a float row copy.
#include "k3x_device.h"

#define AR_MAXSRC 64
#define AR_CH 1024                // products of a chain chunk
#define CP_NT 256

__device__ __forceinline__ const float *ar_src(const float *blocks, int maxb, int nb,
                                               const float *pref, int n, int t, int s)
{
    return s < nb ? blocks + ((size_t)t * maxb + s) * n : pref + (size_t)t * n;
}

// Sum over the wave of a double (every lane).
__device__ __forceinline__ double ar_wsum(double v)
{
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Elements of half `half` of a row of n floats for this lane: f(j, v, w) for its elements,
// j counting them (v of row a, w of row b, or of a again with b NULL).  Zeros past the row (a
// key whose scale is not finite meets NaN there: not proven, so its chain decides).  VEC (n a
// multiple of 4, rows 16-byte aligned): float4 loads, U of each row in flight; else single
// floats, U1 in flight, or one at a time where a row passes a buffer's range.
template <bool VEC, int U, int U1, class F>
__device__ __forceinline__ void ar_half(const float *a, const float *b, int n, int half, int lane, F f)
{
    const int l = half * WAVE + lane;
    if (!VEC && n >= (1 << 28)) {
        int j = 0;
        for (int i = l; i < n; i += 2 * WAVE, j++) f(j, a[i], b ? b[i] : a[i]);
        return;
    }
    const rsrc_t ra = make_rsrc(a, (uint32_t)n * 4u), rb = make_rsrc(b ? b : a, (uint32_t)n * 4u);
    // a step of U (U1) pieces, a piece one load of each of the two waves' lanes; the last step
    // leaves out the pieces past the row (uniform branches, 0.6 us if in every step)
    constexpr int E = VEC ? 4 : 1, P = 2 * WAVE * E, N = VEC ? U : U1;
    auto step = [&](int f0, bool whole) AI {
        u32x4 va[N], vb[N];
#pragma unroll
        for (int u = 0; u < N; u++) {
            if (!whole && f0 + P * u >= n) break;
            const uint32_t o = (uint32_t)(f0 + P * u + E * l) * 4u;
            if (VEC) {
                va[u] = bload16(ra, o);
                if (b) vb[u] = bload16(rb, o);
            } else {
                va[u][0] = __builtin_amdgcn_raw_buffer_load_b32(ra, o, 0, 0);
                if (b) vb[u][0] = __builtin_amdgcn_raw_buffer_load_b32(rb, o, 0, 0);
            }
        }
        SCHED_FENCE();
#pragma unroll
        for (int u = 0; u < N; u++) {
            if (!whole && f0 + P * u >= n) break;
#pragma unroll
            for (int k = 0; k < E; k++)
                f(VEC ? k : u, __uint_as_float(va[u][k]), __uint_as_float(b ? vb[u][k] : va[u][k]));
        }
    };
    int f0 = 0;
    for (; f0 + P * N <= n; f0 += P * N) step(f0, true);
    if (f0 < n) step(f0, false);
}

// An upper bound of the sum of the magnitudes of the partial sums S_i of the chain that
// wg_dot_chain adds (every thread): each thread's run of consecutive products, the runs'
// sums scanned, then each run's partial sums.  In double; the roundings of this evaluation
// are covered by the caller's margin.
template <int NT>
__device__ double ar_prefix_mag(const float *a, float s, const float *b, int n, double *wt)
{
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int m = (n + NT - 1) / NT, i0 = threadIdx.x * m, i1 = min(n, i0 + m);
    double run = 0.0;
    for (int i = i0; i < i1; i++) run += (double)(a[i] * s) * (double)b[i];
    double in = run;
    for (int o = 1; o < WAVE; o <<= 1) {
        const double t = __shfl_up(in, o);
        if (lane >= o) in += t;
    }
    __syncthreads();
    if (lane == WAVE - 1) wt[wave] = in;
    __syncthreads();
    double x = in - run;
    for (int w = 0; w < wave; w++) x += wt[w];
    double mag = 0.0;
    for (int i = i0; i < i1; i++) {
        x += (double)(a[i] * s) * (double)b[i];
        mag += fabs(x);
    }
    mag = ar_wsum(mag);
    __syncthreads();
    if (lane == 0) wt[wave] = mag;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < (NT / WAVE); w++) tot += wt[w];
    return tot;
}

// One workgroup per row t: the sources are blocks[t][0 .. nb-1] then pref[t], nb = row
// t's block count: nbv[t * nbs] when nbv is given (device memory; nbs 0 for one count
// shared by every row, 1 for a count per row: K3_NB(t), k3_ops.c:2481-2483, 2493), else
// nb0.  Each source's key is its RMS-normalised row (inv rounded to float, v*inv in
// float) dotted with fold in double, the two double sums formed in a tree; where the
// tree does not prove the float result (inv, or the key rounded to float) to be the
// reference's chain's, that sum is formed again as the chain (rms_inv_proven,
// float_proven, wg_dot_chain); softmax with exp evaluated in double and rounded to
// float (the reference's expf), the double sum z; p = (float)(e/z); h = sum_s p_s v_s in
// float, in source order from 0 (the raw rows are the values).  A device count outside
// 0 .. min(maxb, AR_MAXSRC - 1) (or above 0 without blocks) fills row t with quiet NaNs
// instead: the reference reads past its stack there.
//
// Two waves a source, every source of up to NT / 128 at once: bound by the latency of a row's
// two dependent passes, not by its bytes.  (256 threads walking the sources one after
// another took 59 us at one row of 6 sources of 7168, 61 at 16 rows, 360 to 480 where a key's
// chain was needed, 578 at 2048; now 13, 13, 14 to 47 and 188.)  A key is tested twice: first
// by chain_gap, which assumes every partial sum as large as sum |p| (about one key in 800
// of random rows fails), then by the partial sums' own magnitudes (one in 50,000).
template <bool VEC, int NT>
__global__ void __launch_bounds__(NT, NT == 256 ? 8 : 4) attn_res_kernel(float *h, const float *blocks, int maxb,
                                                         int nb0, const int *nbv, int nbs,
                                                         const float *pref,
                                                         const float *fold, int n, float eps)
{
    // loads in flight a lane: 256 threads leave 64 registers each
    constexpr int U = NT == 256 ? 2 : 7, U1 = NT == 256 ? 4 : 20;
    __shared__ double red[AR_MAXSRC][2];
    __shared__ float reda[AR_MAXSRC][2], inv[AR_MAXSRC], p[AR_MAXSRC], sc[AR_MAXSRC];
    __shared__ int redo[AR_MAXSRC];
    __shared__ double wt[(NT / WAVE)];
    __shared__ __attribute__((aligned(16))) float buf[2 * AR_CH];
    const int t = blockIdx.x, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int nb = nbv ? nbv[(size_t)t * nbs] : nb0;
    if (nb < 0 || nb > maxb || nb + 1 > AR_MAXSRC || (nb > 0 && !blocks)) {
        for (int i = threadIdx.x; i < n; i += NT) h[(size_t)t * n + i] = __int_as_float(0x7FC00000);
        return;
    }
    const int nsrc = nb + 1;
    // sums of squares: an element takes part in at most n/512 + 11 additions
    for (int it = wave; it < 2 * nsrc; it += (NT / WAVE)) {
        double a4[4] = {0.0, 0.0, 0.0, 0.0};
        ar_half<VEC, U, U1>(ar_src(blocks, maxb, nb, pref, n, t, it >> 1), nullptr, n, it & 1, lane,
                     [&](int j, float v, float) AI { a4[j & 3] += (double)v * (double)v; });
        const double ss = ar_wsum((a4[0] + a4[1]) + (a4[2] + a4[3]));
        if (lane == 0) red[it >> 1][it & 1] = ss;
    }
    __syncthreads();
    if (threadIdx.x < nsrc) {
        const double ss = red[threadIdx.x][0] + red[threadIdx.x][1];
        inv[threadIdx.x] = rms_inv(ss, n, eps);
        redo[threadIdx.x] = !rms_inv_proven(ss, n, eps);
    }
    __syncthreads();
    for (int s = 0; s < nsrc; s++) {
        if (!redo[s]) continue;                                          // uniform; rare
        const float *v = ar_src(blocks, maxb, nb, pref, n, t, s);
        const double c = wg_dot_chain(v, 1.0f, v, n, buf, AR_CH, NT);
        if (threadIdx.x == 0) inv[s] = rms_inv(c, n, eps);
        __syncthreads();
    }
    // keys, and sum |v*inv| |fold| for the gap
    for (int it = wave; it < 2 * nsrc; it += (NT / WAVE)) {
        const float iv = inv[it >> 1];
        double a4[4] = {0.0, 0.0, 0.0, 0.0};
        float m4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        ar_half<VEC, U, U1>(ar_src(blocks, maxb, nb, pref, n, t, it >> 1), fold, n, it & 1, lane,
                     [&](int j, float v, float w) AI {
                         const float vi = v * iv;
                         a4[j & 3] += (double)vi * (double)w;
                         m4[j & 3] = fmaf(fabsf(vi), fabsf(w), m4[j & 3]);
                     });
        const double acc = ar_wsum((a4[0] + a4[1]) + (a4[2] + a4[3]));
        float aa = (m4[0] + m4[1]) + (m4[2] + m4[3]);
        for (int off = 32; off >= 1; off >>= 1) aa += __shfl_xor(aa, off);
        if (lane == 0) { red[it >> 1][it & 1] = acc; reda[it >> 1][it & 1] = aa; }
    }
    __syncthreads();
    if (threadIdx.x < nsrc) {
        const int s = threadIdx.x;
        const double acc = red[s][0] + red[s][1];
        sc[s] = (float)acc;
        redo[s] = !float_proven(acc, chain_gap(abs_bound(reda[s][0] + reda[s][1], n), n));
    }
    __syncthreads();
    for (int s = 0; s < nsrc; s++) {
        if (!redo[s]) continue;                                          // uniform; rare
        const float *v = ar_src(blocks, maxb, nb, pref, n, t, s);
        const double acc = red[s][0] + red[s][1];
        const double as = abs_bound(reda[s][0] + reda[s][1], n);
        // the chain is within 2^-53 sum |S_i| of the exact sum, this tree within 2^-53
        // (n/512 + 11) sum |p| (doubled, for the magnitudes' own roundings)
        const double d = (ar_prefix_mag<NT>(v, inv[s], fold, n, wt) * (1.0 + 0x1p-16) +
                          2.0 * ((double)(n >> 9) + 16.0) * as) * 0x1p-53;
        if (float_proven(acc, d)) continue;                              // uniform
        const double c = wg_dot_chain(v, inv[s], fold, n, buf, AR_CH, NT);   // thread 0's
        if (threadIdx.x == 0) sc[s] = (float)c;
        __syncthreads();
    }
    if (wave == 0) {
        float m = sc[0];
        for (int s = 1; s < nsrc; s++) m = sc[s] > m ? sc[s] : m;
        const float e = lane < nsrc ? (float)exp((double)(sc[lane] - m)) : 0.0f;
        double z = 0.0;
        for (int s = 0; s < nsrc; s++) z += (double)__shfl(e, s);
        if (lane < nsrc) p[lane] = (float)((double)e / z);
    }
    __syncthreads();
    if (VEC) {
        for (int i = 4 * threadIdx.x; i < n; i += 4 * NT) {
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
            for (int s0 = 0; s0 < nsrc; s0 += 4) {
                f32x4 v[4];
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (s0 + u < nsrc) v[u] = *(const f32x4 *)(ar_src(blocks, maxb, nb, pref, n, t, s0 + u) + i);
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (s0 + u < nsrc) o += p[s0 + u] * v[u];
            }
            *(f32x4 *)(h + (size_t)t * n + i) = o;
        }
    } else {
        for (int i = threadIdx.x; i < n; i += NT) {
            float o = 0.0f;
            for (int s = 0; s < nsrc; s++) o += p[s] * ar_src(blocks, maxb, nb, pref, n, t, s)[i];
            h[(size_t)t * n + i] = o;
        }
    }
}

__global__ void __launch_bounds__(CP_NT) copy_f32x4(float *dst, const float *src, size_t n4)
{
    const size_t i = (size_t)blockIdx.x * CP_NT + threadIdx.x;
    if (i < n4) ((f32x4 *)dst)[i] = ((const f32x4 *)src)[i];
}

// nbv == NULL: the count nb for every row (checked here); else the rows' counts are read
// on the device from nbv[t * nbs] (nb unused).
extern "C" int k3x_dev_attn_res(float *h, const float *blocks, int maxb, int nb, const int *nbv,
                                int nbs, const float *pref, const float *fold, int n, int T,
                                float eps, void *stream)
{
    if (!nbv && nb + 1 > AR_MAXSRC) return K3X_E_SHAPE;
    // rows of whole 16-byte pieces, every base aligned (blocks is not read when no row has
    // any); a row past 2^31 bytes keeps the plain loop
    const uintptr_t al = (uintptr_t)h | (uintptr_t)blocks | (uintptr_t)pref | (uintptr_t)fold;
    const bool vec = n % 4 == 0 && (al & 15) == 0 && n < (1 << 28);
    // 1024 threads where every row has a CU to itself; past 256 rows two workgroups a CU, and
    // past 512 rows of at most 2048 floats eight small ones.  (1024 threads for all: 36 us at
    // 2048 rows of one source of 128, 63 of six, 10.5 at 300 rows of two of 512, 63 at 2048
    // rows of one of 7168; now 7.7, 17, 7.2 and 44.  512 for the long rows past 512: 25 at 2048
    // rows of one source of 2048, 128 of sixteen; 256 there 14 and 131, and at 7168 floats 45
    // and 591 against 44 and 405.)
    const int nt = T <= 256 ? 1024 : (T <= 512 || n > 2048 ? 512 : 256);
#define AR_LAUNCH(NT)                                                                              \
    do {                                                                                           \
        if (vec)                                                                                   \
            hipLaunchKernelGGL((attn_res_kernel<true, NT>), dim3(T), dim3(NT), 0, (hipStream_t)stream, \
                               h, blocks, maxb, nb, nbv, nbs, pref, fold, n, eps);                 \
        else                                                                                       \
            hipLaunchKernelGGL((attn_res_kernel<false, NT>), dim3(T), dim3(NT), 0, (hipStream_t)stream, \
                               h, blocks, maxb, nb, nbv, nbs, pref, fold, n, eps);                 \
    } while (0)
    if (nt == 1024)     AR_LAUNCH(1024);
    else if (nt == 512) AR_LAUNCH(512);
    else                AR_LAUNCH(256);
#undef AR_LAUNCH
    return hipGetLastError() == hipSuccess ? 0 : K3X_E_HIP;
}

// dst = src, n floats (n a multiple of 4, both 16-byte aligned): a kernel rather than a
// memcpy node, so that a captured sequence holds kernels only.
extern "C" int k3x_dev_copy_f32(float *dst, const float *src, size_t n, void *stream)
{
    const size_t n4 = n / 4;
    hipLaunchKernelGGL(copy_f32x4, dim3((unsigned)((n4 + CP_NT - 1) / CP_NT)), dim3(CP_NT), 0,
                       (hipStream_t)stream, dst, src, n4);
    return hipGetLastError() == hipSuccess ? 0 : K3X_E_HIP;
}
