// k3x_topk.h - one token's top-k selection by one wave, shared by the decode and the
// prefill kernels (the reference's repeated maximum, k3_ops.c:1700-1716).
#ifndef K3X_TOPK_H
#define K3X_TOPK_H

#include "k3x_device.h"

// Order-preserving key of a choice value: larger float -> larger key; -0 is +0 (they
// compare equal in the reference); NaN -> 0 (never selected); -inf -> K_NEG_INF (never
// selected either: the reference's strict '>' against -inf fails).
#define K_NEG_INF 0x007FFFFFu
__device__ __forceinline__ uint32_t choice_key(float f)
{
    uint32_t u = __float_as_uint(f);
    if (f != f) return 0u;
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The choice value of a key (the inverse of choice_key on the values it keeps).
__device__ __forceinline__ float key_choice(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// The choice key (choice_key's order) just above choice + slack: an upper bound of the
// reference's choice for an expert whose logit is not proven.
__device__ __forceinline__ uint32_t slack_key(float choice, float slack)
{
    const uint32_t k = choice_key((float)((double)choice + (double)slack));
    return (k != 0u && k < 0xFF800000u) ? k + 1u : k;
}

// Whether an expert not proven could change a selection whose K-th choice is ck, or one
// of its weights: its choice may reach ck (hk: the token's largest slack_key, 0 = none).
// Every selected expert's choice is at least ck, so a selected one not proven counts.
__device__ __forceinline__ bool slack_reaches(uint32_t hk, float ck)
{
    return hk != 0u && hk >= choice_key(ck);
}

// The slack of a choice whose logit's float can lie df from the one it was worked out from:
// a bound on the distance of the reference's choice, a quarter of df (the sigmoid's slope is
// at most 1/4) plus the roundings of the sigmoid and of the bias add (a few units in the
// last place of |choice| <= 2 + |bias|).
__device__ __forceinline__ float logit_slack(double df, float bias)
{
    return (float)((df * 0.25 + (2.0 + fabs((double)bias)) * 0x1p-21) * 1.01);
}

__device__ __forceinline__ int lanes_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

template <int CP>
__device__ __forceinline__ float bload_f32(rsrc_t r, uint32_t off)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, CP));
}

// Maximum of an unsigned value over the wave: DPP steps within quads and rows, then row
// broadcasts across rows (lane 63 ends with the total), then a read of lane 63.  Lanes
// that a step does not write take 0, the identity.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v)
{
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
    return o > v ? o : v;
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v)
{
    v = dpp_max<0xB1, 0xF>(v);      // quad_perm [1,0,3,2]
    v = dpp_max<0x4E, 0xF>(v);      // quad_perm [2,3,0,1]
    v = dpp_max<0x124, 0xF>(v);     // row_ror:4
    v = dpp_max<0x128, 0xF>(v);     // row_ror:8: every lane holds its row's maximum
    v = dpp_max<0x142, 0xA>(v);     // row_bcast:15 into rows 1 and 3
    v = dpp_max<0x143, 0xC>(v);     // row_bcast:31 into rows 2 and 3
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One token's top-k by one wave, the reference's repeated maximum (k3_ops.c:1700-1708):
// K rounds, each taking the largest remaining choice with the lower index first among
// equal values; that is the K largest words key << 32 | ~index in order.  Lane l holds
// experts l*NE + c, or with ST experts c*64 + l (rows of them load coalesced).
//
// A bound first: the K-th largest distinct lane maximum, or lower, by K wave maxima (every
// word of the selection has at least that key).  The words at or above it, K and a few
// more, go to a list in LDS, and each one's place is the number of listed words above it.
// Where they are more than the list holds (many equal choices, K near 64), K rounds over
// all words: each takes the wave's largest word below the previous winner.  (Those rounds
// for every call walked a lane's NE words each: 64-bit compares, 6700 instructions at 16
// words and 16 rounds.  At two words a lane the list is no loss: decode calls of a layer of 16
// experts, top 4, took 17.4 to 17.8 us at one token either way, 25.8 to 26.0 and 26.4 to 26.6
// at four, 30.0 to 30.5 and 29.9 to 30.1 at eight.)  NaN and -inf are never taken; a place that nothing fills gives
// index 0, weight 0.  Weights are the unbiased scores, renormalised through a double sum
// in slot order and a float reciprocal, then scaled (:1710-1716).  Results in s_idx/s_w
// (LDS), and lane j's (slot j's) in out_e/out_w when given, and the K-th largest choice
// (-inf when fewer than K were selectable) in out_ck.  ts: LDS of this wave.
struct TkList {
    uint64_t w[WAVE];
    float    s[WAVE];
};

template <int NE, bool ST>
__device__ void wave_topk_vals(const float (&cv)[NE], const float (&sc)[NE], int E, int K,
                               int renorm, float routed_scale, int *s_idx, float *s_w,
                               int lane, TkList &ts, int *out_e = nullptr,
                               float *out_w = nullptr, float *out_ck = nullptr)
{
    uint32_t key[NE], lm = 0u, m = 0u;
#pragma unroll
    for (int c = 0; c < NE; c++) {
        const uint32_t k = choice_key(cv[c]);
        key[c] = ((ST ? c * WAVE + lane : lane * NE + c) < E && k > K_NEG_INF) ? k : 0u;
        lm = key[c] > lm ? key[c] : lm;
    }
    for (int j = 0; j < K; j++) {
        m = wave_max_u32(lm);
        if (m == 0u) break;                     // uniform
        lm = lm == m ? 0u : lm;
    }
    const uint32_t thr = m ? m : 1u;            // fewer maxima than K: every word
    int n = 0;
#pragma unroll
    for (int c = 0; c < NE; c++) {
        const bool on = key[c] >= thr;
        const uint64_t mask = __ballot(on);
        const int pos = n + lanes_below(mask);
        if (on && pos < WAVE) {
            ts.w[pos] = ((uint64_t)key[c] << 32) |
                        (uint64_t)(~(uint32_t)(ST ? c * WAVE + lane : lane * NE + c));
            ts.s[pos] = sc[c];
        }
        n += __popcll(mask);
    }
    int mine_e = 0;                             // lane j: slot j's expert and score
    float mine_s = 0.0f;
    float ck = -__builtin_inff();
    if (n <= WAVE) {                            // uniform
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const uint64_t w = lane < n ? ts.w[lane] : 0ull;
        const float s = lane < n ? ts.s[lane] : 0.0f;
        int rank = 0;
        for (int j = 0; j < n; j++) rank += ts.w[j] > w;
        const bool in = lane < n && rank < K;
        if (in) {
            s_idx[rank] = (int)~(uint32_t)w;
            s_w[rank] = s;
        }
        const uint64_t kth = __ballot(lane < n && rank == K - 1);
        if (kth != 0ull)
            ck = key_choice((uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(w >> 32),
                                                                (int)__builtin_ctzll(kth)));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < n && lane < K) {
            mine_e = s_idx[lane];
            mine_s = s_w[lane];
        }
    } else {
        uint64_t prev = ~0ull;    // the previous round's winner (none yet: above all)
        for (int j = 0; j < K; j++) {
            uint64_t best = 0ull;
            float bs = 0.0f;
#pragma unroll
            for (int c = 0; c < NE; c++) {
                const uint64_t pk = ((uint64_t)key[c] << 32) |
                                    (uint64_t)(~(uint32_t)(ST ? c * WAVE + lane : lane * NE + c));
                const uint64_t v = key[c] && pk < prev ? pk : 0ull;
                const bool gt = v > best;
                best = gt ? v : best;
                bs = gt ? sc[c] : bs;
            }
            const uint32_t bk = (uint32_t)(best >> 32);
            const uint32_t mk = wave_max_u32(bk);
            if (mk == 0u) { ck = -__builtin_inff(); break; }    // nothing left (uniform)
            // the lowest index among the lanes that hold that key
            const uint32_t lo = bk == mk ? (uint32_t)best : 0u, ml = wave_max_u32(lo);
            const int w = (int)__builtin_ctzll(__ballot(bk == mk && lo == ml));
            const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bs), w));
            prev = ((uint64_t)mk << 32) | ml;
            if (lane == j) { mine_e = (int)~ml; mine_s = ws; }
            ck = key_choice(mk);
        }
    }
    if (out_ck) *out_ck = ck;
    float wgt = mine_s;
    if (renorm && K > 1) {
        double sum = 0.0;
        for (int j = 0; j < K; j++)
            sum += (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine_s), j));
        const float inv = (float)(1.0 / (sum + 1e-20));
        wgt *= inv;
    }
    wgt *= routed_scale;
    if (lane < K) {
        s_idx[lane] = mine_e;
        s_w[lane] = wgt;
    }
    if (out_e) { *out_e = mine_e; *out_w = wgt; }
}

// wave_topk_vals of choices and scores in memory (CP: the loads' cache policy)
template <int NE, int CP>
__device__ void wave_topk(rsrc_t cr, rsrc_t sr, uint32_t row_off, int E, int K, int renorm,
                          float routed_scale, int *s_idx, float *s_w, int lane, TkList &ts,
                          int *out_e = nullptr, float *out_w = nullptr,
                          float *out_ck = nullptr)
{
    float sc[NE], cv[NE];
#pragma unroll
    for (int c = 0; c < NE; c++) {
        const int e = lane * NE + c;
        const uint32_t o = e < E ? row_off + 4u * (uint32_t)e : K3X_OOB;
        cv[c] = bload_f32<CP>(cr, o);
        sc[c] = bload_f32<CP>(sr, o);
    }
    SCHED_FENCE();      // both rows' loads in flight together: one memory round trip
    wave_topk_vals<NE, false>(cv, sc, E, K, renorm, routed_scale, s_idx, s_w, lane, ts, out_e,
                              out_w, out_ck);
}

// wave_topk for N tokens of one wave (tokens past ntok load nothing and store nothing):
// every token's rows are loaded at once, one memory round trip for all; out_ck[r] is token
// r's K-th choice.
template <int NE, int CP, int N>
__device__ void wave_topk_n(rsrc_t cr, rsrc_t sr, const uint32_t (&row_off)[N], int ntok, int E,
                            int K, int renorm, float routed_scale, int *const (&s_idx)[N],
                            float *const (&s_w)[N], int lane, TkList &ts, float (&out_ck)[N])
{
    float sc[N][NE], cv[N][NE];
#pragma unroll
    for (int r = 0; r < N; r++)
#pragma unroll
        for (int c = 0; c < NE; c++) {
            const int e = lane * NE + c;
            const uint32_t o = (e < E && r < ntok) ? row_off[r] + 4u * (uint32_t)e : K3X_OOB;
            cv[r][c] = bload_f32<CP>(cr, o);
            sc[r][c] = bload_f32<CP>(sr, o);
        }
    SCHED_FENCE();
#pragma unroll
    for (int r = 0; r < N; r++)
        if (r < ntok)
            wave_topk_vals<NE, false>(cv[r], sc[r], E, K, renorm, routed_scale, s_idx[r], s_w[r],
                                      lane, ts, nullptr, nullptr, &out_ck[r]);
}

#endif
