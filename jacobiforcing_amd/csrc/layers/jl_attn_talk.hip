// jl_attn_talk.hip — attention whose heads are mixed after the softmax (talking heads), with a distance bias, a window and kept first tokens, in one sweep.
//   out_h = sum over heads x of talk[h, x] softmax_x(scores) V_(value head of h)
// The mixture is linear, so it need not wait for the softmax's sums: every head x collects O_(x, g) = P_x V_g for ALL value heads g, as the running softmax goes, and a
// second launch adds up out_h = sum_x talk[h, x] O_(x, g(h)) / l_x.  That costs G products with the values instead of one, and saves the second sweep over the keys (scores and
// exponentials again) and the exchange of every weight between the heads.  Weights stay 32-bit numbers on their way into the matrix cores: P = hi + lo in bfloat16 (16 bits
// of mantissa; the mixed weights were rounded to 8 before), two products each.
// Rows of the products are (query, head) pairs of one key head, as in jl_attn_rows.hip: a wavefront forms S^T = K Q^T for its 32 rows, a lane holds keys of ONE row, the
// weights are the next product's operand as they are, and V^T is read by ds_read_b64_tr_b16.  A workgroup has 4 wavefronts (128 rows) over the same keys, or one
// (32 rows: portions of a few tokens, where keys are shared out over workgroups until the chip is full; single tokens of up to 16 heads go to jl_attn_token.hip).  Keys go in tiles of 32 consecutive positions, the kept first ones before the window's; the next
// tile's rows and biases travel while this one is multiplied (one wavefront: other workgroups of the CU fill the wait).  A workgroup collects one value head: two at a time would form
// the scores once instead of twice, but their 128 accumulators leave the tiles' rows no registers (8 heads over 2: 340 us instead of 200).
// What bounds it: issue and latency at two wavefronts per SIMD; G (1 + 2) products of D or Dv per score, a third of the matrix rate at 4 x 2048 tokens.
// Measured against two sweeps with every weight exchanged through LDS (us, norms and gates included, bfloat16, 8 heads over 2 of 128, window 1024, 4 kept):
//   4 x 2048 tokens 797 -> 195 (173 and 22 for the mixture)    777 + 300 tokens beside 30 single ones 258 -> 79    200 tokens 73 -> 23
//   16 heads over 4, 4 x 2048, window 2048: 3000 -> 730
#include "jl_attn.h"

constexpr int AT_KT = 32;
constexpr int AT_BIAS = 5;              // bias entries per thread and tile at most (checked by the launch)

// a bias times log2(e); a finite one stays finite (a mask of the type's lowest value is a number: a row that sees nothing else still has weights)
__device__ __forceinline__ float at_log2_bias(float b) {
    const float v = b * 1.44269504088896341f;
    return __builtin_isinf(v) && !__builtin_isinf(b) ? __builtin_copysignf(__FLT_MAX__, b) : v;
}

static __host__ __device__ inline int at_bias_row(int TQ, int HF) { return (TQ + AT_KT - 1 + 31) / 32 * 32 + (HF < 32 ? 32 / HF : 1); }   // heads of a query meet different banks
static size_t at_lds_bytes(int KU, int VU, int TQ, int HF, int NW) { return (NW > 1 ? 2 : 1) * ((size_t)AT_KT * (KU + VU) * 16 + AT_KT * 4 + (size_t)HF * at_bias_row(TQ, HF) * 4); }

template <int KU, int VU, int NW>                                                     // D <= 8 * KU, Dv <= 8 * VU, wavefronts
__global__ __launch_bounds__(64 * NW, 2) void attn_talk_kernel(jl_attn_args a, int HF, int tile0, int n_tiles) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int THREADS = 64 * NW, BUFS = NW > 1 ? 2 : 1, KT = AT_KT, NDV = VU / 4, BUF = KT * (KU + VU);
    constexpr int KPF = (KT * KU + THREADS - 1) / THREADS, VPF = (KT * VU + THREADS - 1) / THREADS;
    const int H = a.H, G = a.G, D = a.D, Dv = a.Dv, TQ = a.TQ, S = a.splits;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    // key heads (and the value heads' groups) side by side: neighbouring workgroups go to different XCDs, so each keeps few heads' keys in its L2
    const int sides = G * G, side = blockIdx.x % sides, rest = blockIdx.x / sides, split = rest % S, ti = rest / S, c = side / G, g = side - c * G;
    const int *tile = a.tiles + 4 * (int64_t)(tile0 + ti);
    const int b = tile[0], i0 = tile[1], cnt = tile[2], row0 = tile[3], h0 = c * HF;
    if (b < 0 || cnt <= 0) return;
    uint4 *buf0 = (uint4 *)smem;
    int *tokS = (int *)(buf0 + BUFS * BUF);                         // [BUFS][KT] pool tokens of a tile's keys
    float *biasS = (float *)(tokS + BUFS * KT);                     // [BUFS][HF][row] biases times log2(e): entry query - key + KT - 1 (within the tile)
    const int BR = at_bias_row(TQ, HF);
    const int window = a.window > 0 ? a.window : 0x3fffffff;
    const int i_max = i0 + cnt - 1;
    const int keep_first = a.keep_first;
    auto lowest = [&](int i) { return i - window + 1; };        // first key that query i sees
    const int lo = lowest(i0) > 0 ? lowest(i0) : 0;                 // of the first row's
    const int kept = keep_first < lo ? keep_first : lo;             // kept first tokens in front of them
    const int kept_tiles = (kept + KT - 1) / KT, n_kt = kept_tiles + (i_max + 1 - lo + KT - 1) / KT;
    const int share = (n_kt + S - 1) / S, t_lo = split * share, t_hi = t_lo + share < n_kt ? t_lo + share : n_kt;
    // a tile's first position and its keys
    auto first_of = [&](int t) { return t < kept_tiles ? t * KT : lo + (t - kept_tiles) * KT; };
    auto keys_of = [&](int t) { const int e = (t < kept_tiles ? kept : i_max + 1) - first_of(t); return e < KT ? e : KT; };
    const int *bt = a.block_tables + (int64_t)b * a.bt_stride;
    const bf16_t *kc = (const bf16_t *)a.k_cache + (int64_t)c * D, *vc = (const bf16_t *)a.v_cache + (int64_t)g * Dv;
    const int page_shift = (a.page_size & (a.page_size - 1)) == 0 ? __builtin_ctz(a.page_size) : -1;
    for (int e = tid; e < BUFS * BUF; e += THREADS) buf0[e] = make_uint4(0, 0, 0, 0);         // columns beyond D / Dv and rows beyond the last key stay zero or finite

    // this lane's row: (query R / HF, head h0 + R % HF); both half-wavefronts hold it
    const int R = 32 * wave + l32, ii = R / HF, hl = R - ii * HF;
    const bool ok = ii < TQ && ii < cnt;
    const int qi = i0 + ii, q_lo = lowest(qi);
    ar_bf16x8 qf[KU / 2];
#pragma unroll
    for (int x = 0; x < KU / 2; ++x) {
        uint4 w = make_uint4(0, 0, 0, 0);
        if (ok && 16 * x + 8 * hi < D) w = *(const uint4 *)((const bf16_t *)a.q + (int64_t)(row0 + ii) * H * D + (h0 + hl) * D + 16 * x + 8 * hi);
        qf[x] = __builtin_bit_cast(ar_bf16x8, w);
    }
    constexpr float LOG2E = 1.44269504088896341f;                   // scores are kept times log2(e): weights are 2 ** (s - max)
    const float c2 = a.scale * LOG2E;
    float m_run = -INFINITY, l_run = 0.f;
    ar_f32x16 acc[NDV];
#pragma unroll
    for (int t = 0; t < NDV; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    const int wq_first = 32 * wave / HF, wq_last = (32 * wave + 31) / HF < cnt - 1 ? (32 * wave + 31) / HF : cnt - 1;
    const bool wave_live = wq_first < TQ && wq_first < cnt;
    const bool wave_full = (32 * wave + 31) / HF < TQ && (32 * wave + 31) / HF < cnt;      // all 32 rows are rows of the tile

    uint4 kreg[KPF], vreg[VPF];
    auto load16 = [](const bf16_t *p) -> uint4 { const uint4 v = *(const uint4 *)p; return make_uint4(v.x, v.y, v.z, v.w); };
    float breg[AT_BIAS];
    int tok_next = 0;
    auto look_up = [&](int t) {                                  // thread j < KT: the pool token of the tile's key j, two tiles ahead of the products
        if (t >= t_hi || tid >= keys_of(t)) return;
        const int j = first_of(t) + tid, pg = page_shift >= 0 ? j >> page_shift : j / a.page_size;
        tok_next = bt[pg] * a.page_size + (j - pg * a.page_size);
    };
    auto tokens_out = [&](int sel) { if (tid < KT) tokS[sel * KT + tid] = tok_next; };
    const int n_bias = HF * (cnt + KT - 1);
    auto bias_of = [&](int e, int j0) {                             // heads side by side in memory
        const int y = e / HF;
        int n = i0 + y - (KT - 1) - j0;                             // distance of the tile's last key from query y, of key KT - 1 - k from query y - k ..
        n = n < 0 ? 0 : n < a.lut_len ? n : a.lut_len - 1;
        return a.rel[(int64_t)(a.lut ? a.lut[n] : n) * H + h0 + e - y * HF];
    };
    auto fetch = [&](int t, const int *tok) {
        const int nk = keys_of(t), j0 = first_of(t);
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) kreg[it] = load16(kc + (int64_t)tok[jj] * a.k_ld + 8 * u);
        }
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * THREADS, jj = e / VU, u = e % VU;
            if (jj < nk && 8 * u < Dv) vreg[it] = load16(vc + (int64_t)tok[jj] * a.v_ld + 8 * u);
        }
        if (NW > 1 && a.rel)
#pragma unroll
            for (int it = 0; it < AT_BIAS; ++it) {
                const int e = tid + it * THREADS;
                if (e < n_bias) breg[it] = bias_of(e, j0);
            }
    };
    auto stash = [&](int t, int sel) {
        const int nk = keys_of(t);
        uint4 *Ks = buf0 + sel * BUF;
        float *bias = biasS + sel * HF * BR;
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) Ks[jj * KU + ar_key_unit<KU>(jj, u)] = kreg[it];
        }
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * THREADS, jj = e / VU, u = e % VU;
            if (jj < nk && 8 * u < Dv) Ks[KT * KU + jj * VU + ar_value_unit<VU>(jj, u)] = vreg[it];
        }
        if (NW > 1 && a.rel)
#pragma unroll
            for (int it = 0; it < AT_BIAS; ++it) {
                const int e = tid + it * THREADS;
                if (e < n_bias) { const int y = e / HF; bias[(e - y * HF) * BR + y] = at_log2_bias(breg[it]); }
            }
        if (NW == 1 && a.rel) {
            const int j0 = first_of(t);
#pragma unroll 4
            for (int e = tid; e < n_bias; e += THREADS) { const int y = e / HF; bias[(e - y * HF) * BR + y] = at_log2_bias(bias_of(e, j0)); }
        }
    };
    look_up(t_lo);
    tokens_out(0);
    look_up(t_lo + 1);
    if (NW > 1) tokens_out(1);
    __syncthreads();
    if (NW > 1 && t_lo < t_hi) {
        fetch(t_lo, tokS);
        stash(t_lo, 0);
    }
    __syncthreads();
    for (int t = t_lo, sel = 0; t < t_hi; ++t, sel ^= NW > 1) {
        if (NW > 1) {
            if (t + 1 < t_hi) fetch(t + 1, tokS + (sel ^ 1) * KT);
            look_up(t + 2);
        } else {                                                    // other workgroups of the CU fill the wait: registers for them instead of for a tile ahead
            fetch(t, tokS);
            stash(t, 0);
            tokens_out(0);
            look_up(t + 2);
            __syncthreads();
        }
        const uint4 *Ks = buf0 + sel * BUF;
        const int j0 = first_of(t), nk = keys_of(t);
        // wavefront-uniform: keys all behind its last query, or all before its first query's window and not kept
        if (wave_live && j0 <= i0 + wq_last && (j0 < keep_first || j0 + nk - 1 >= lowest(i0 + wq_first))) {
            ar_f32x16 sc;
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = 0.f;
#pragma unroll
            for (int x = 0; x < KU / 2; ++x)
                sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ar_bf16x8, Ks[l32 * KU + ar_key_unit<KU>(l32, 2 * x + hi)]), qf[x], sc, 0, 0, 0);
            if (a.rel) {
                const float *bias = biasS + sel * HF * BR + hl * BR + (ok ? ii : 0) + KT - 1 - 4 * hi;
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = fmaf(sc[r], c2, bias[-(8 * (r >> 2) + (r & 3))]);
            } else
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] *= c2;
            // wavefront-uniform: a full tile whose keys every row of the wavefront sees needs no mask
            const bool inside = nk == KT && wave_full && j0 + KT - 1 <= i0 + wq_first && (j0 >= lowest(i0 + wq_last) || j0 + KT <= keep_first);
            if (!inside) {
                const int first = ok ? q_lo - j0 : KT, last = qi - j0 < nk - 1 ? qi - j0 : nk - 1, keep = ok ? keep_first - j0 : 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kk = 8 * (r >> 2) + 4 * hi + (r & 3);
                    sc[r] = (kk >= first || kk < keep) && kk <= last ? sc[r] : -INFINITY;
                }
            }
            float mx = sc[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run, mx), m_sub = m_new > -INFINITY ? m_new : 0.f;      // a row that has seen no key yet: all weights are 2 ** -inf
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_sub);
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) { sc[r] = __builtin_amdgcn_exp2f(sc[r] - m_sub); sum += sc[r]; }
            l_run = l_run * alpha + sum;
            m_run = m_new;
            if (__any(alpha != 1.0f)) {                             // after the first tiles a row's maximum seldom moves
#pragma unroll
                for (int y = 0; y < NDV; ++y)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[y][r] *= alpha;
            }
            const char *Vs = (const char *)(Ks + KT * KU);
            const int vk = 4 * hi + ((lane & 15) >> 2), vc8 = 8 * (lane & 1), vu = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);      // this lane's key, half unit and unit of a turned block
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                ar_f32x8 pf;
#pragma unroll
                for (int x = 0; x < 8; ++x) pf[x] = sc[8 * s + x];
                const ar_bf16x8 ph = __builtin_convertvector(pf, ar_bf16x8);
                const ar_bf16x8 pl = __builtin_convertvector(pf - __builtin_convertvector(ph, ar_f32x8), ar_bf16x8);
#pragma unroll
                for (int y = 0; y < NDV; ++y) {
                    ar_s16x4 half[2];
#pragma unroll
                    for (int z = 0; z < 2; ++z) {
                        const int key = 16 * s + 8 * z + vk;
                        half[z] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ar_lds_s16x4 *)(Vs + 16 * (key * VU + ar_value_unit<VU>(key, 4 * y + vu)) + vc8));
                    }
                    const ar_bf16x8 va = __builtin_bit_cast(ar_bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
                    acc[y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, ph, acc[y], 0, 0, 0);
                    acc[y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pl, acc[y], 0, 0, 0);
                }
            }
        }
        if (NW > 1) {
            if (t + 1 < t_hi) stash(t + 1, sel ^ 1);
            tokens_out(sel);
        }
        __syncthreads();
    }
    l_run += __shfl_xor(l_run, 32, 64);
    if (!ok) return;
    // shares of the pass's rows: [tile, query][split][head][value head][Dv], and their maxima and sums [..][head][2] behind all of them
    const int64_t row = ((int64_t)ti * TQ + ii) * S + split;
    float *ml = a.scratch + (int64_t)n_tiles * TQ * S * H * G * Dv + (row * H + h0 + hl) * 2;
    if (g == 0 && hi == 0) { ml[0] = m_run; ml[1] = l_run; }
    if (!(l_run > 0.f) && m_run == -INFINITY) return;               // nothing seen: the share counts for nothing (or, all shares like it, the row is not a number)
    float *o = a.scratch + ((row * H + h0 + hl) * G + g) * Dv;
#pragma unroll
    for (int y = 0; y < NDV; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = 32 * y + 8 * q + 4 * hi;                // registers 4q .. 4q + 3: four consecutive value columns
            if (col < Dv) *(float4 *)(o + col) = make_float4(acc[y][4 * q], acc[y][4 * q + 1], acc[y][4 * q + 2], acc[y][4 * q + 3]);
        }
}

// w[split][head] = 2 ** (m - M) / L (not a number where L is none or zero, as the softmax of such scores), then out_h = sum over heads x of talk[h, x] sum over splits of w O_(x, g(h)), gated.  A wavefront per token where shares are whole (bytes bound it:
// 8192 tokens, 8 heads over 2 of 128 in 22 us); a workgroup per token (SPREAD), which adds up the shares of different heads on different wavefronts first, where they are not
constexpr int AM_HEADS = 32;
template <bool SPREAD>
__global__ __launch_bounds__(256) void attn_talk_mix_kernel(jl_attn_args a, int tile0, int n_tiles) {
    extern __shared__ __attribute__((aligned(16))) float mixS[];    // SPREAD: the heads' sums [H][G * Dv]; weights [tokens][S][H], talk [H][H]
    const int H = a.H, G = a.G, Dv = a.Dv, S = a.splits, rep = H / G, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, W = G * Dv;
    float *sums = mixS, *w = mixS + (SPREAD ? H * (W > 2 * S ? W : 2 * S) : wave * H), *talk = SPREAD ? w + S * H : mixS + 4 * H;
    for (int e = threadIdx.x; e < H * H; e += 256) talk[e] = a.talk[e];
    const int64_t r = SPREAD ? blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
    const int ti = (int)(r / a.TQ), ii = (int)(r - (int64_t)ti * a.TQ);
    int cnt = 0, row0 = 0;
    if (ti < n_tiles) { const int *tile = a.tiles + 4 * (int64_t)(tile0 + ti); cnt = tile[0] >= 0 ? tile[2] : 0; row0 = tile[3]; }
    const bool live = ii < cnt;
    if (SPREAD && !live) return;
    const float *ml = a.scratch + (int64_t)n_tiles * a.TQ * S * H * W + r * S * H * 2, *po = a.scratch + r * S * H * W;
    if (SPREAD) {
        float2 *mls = (float2 *)sums;                               // [S][H], where the sums will be
        for (int e = threadIdx.x; e < S * H; e += 256) mls[e] = *(const float2 *)(ml + 2 * e);
        __syncthreads();
        if (threadIdx.x < H) {
            const int x = threadIdx.x;
            float M = -INFINITY, L = 0.f;
            for (int s = 0; s < S; ++s) M = fmaxf(M, mls[s * H + x].x);
            for (int s = 0; s < S; ++s) {
                const float m = mls[s * H + x].x, e = m > -INFINITY ? __builtin_amdgcn_exp2f(m - M) : 0.f;
                w[s * H + x] = e;
                L += mls[s * H + x].y * e;
            }
            const float inv = L > 0.f ? 1.0f / L : NAN;
            for (int s = 0; s < S; ++s) w[s * H + x] *= inv;
        }
    } else if (live && lane < H) w[lane] = ml[2 * lane + 1] > 0.f ? 1.0f / ml[2 * lane + 1] : NAN;
    __syncthreads();
    // a head's sum over the shares, four columns of all value heads; an empty share (weight zero) holds nothing and is not looked at
    auto head_sum = [&](int x, int e) {
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!SPREAD) {
            const float4 p = *(const float4 *)(po + (int64_t)x * W + 4 * e);
            return make_float4(w[x] * p.x, w[x] * p.y, w[x] * p.z, w[x] * p.w);
        }
#pragma unroll 4
        for (int s = 0; s < S; ++s) {
            const float f = w[s * H + x];
            const float4 p = *(const float4 *)(po + (int64_t)(s * H + x) * W + 4 * e);
            o.x = f != 0.f ? fmaf(f, p.x, o.x) : o.x;
            o.y = f != 0.f ? fmaf(f, p.y, o.y) : o.y;
            o.z = f != 0.f ? fmaf(f, p.z, o.z) : o.z;
            o.w = f != 0.f ? fmaf(f, p.w, o.w) : o.w;
        }
        return o;
    };
    if (SPREAD) {
        for (int e = threadIdx.x; e < H * W / 4; e += 256) { const int x = e / (W / 4); ((float4 *)sums)[e] = head_sum(x, e - x * (W / 4)); }
        __syncthreads();
    }
    if (!live) return;
    const bf16_t *gate = (const bf16_t *)a.gate;
    const int64_t n = row0 + ii;
    const int quads = (rep + 3) / 4;
    for (int f = SPREAD ? (int)threadIdx.x : lane; f < quads * W / 4; f += SPREAD ? 256 : 64) {      // four columns of four heads of value head g
        const int y0 = 4 * (f / (W / 4)), e = f % (W / 4), g = 4 * e / Dv, d = 4 * e - g * Dv;
        float v[4][4] = {};
        for (int x = 0; x < H; ++x) {
            const float4 o = SPREAD ? ((const float4 *)sums)[x * (W / 4) + e] : head_sum(x, e);
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const float t = y0 + y < rep ? talk[(g * rep + y0 + y) * H + x] : 0.f;
                v[y][0] += t * o.x; v[y][1] += t * o.y; v[y][2] += t * o.z; v[y][3] += t * o.w;
            }
        }
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            if (y0 + y >= rep) continue;
            const int h = g * rep + y0 + y, col = h * Dv + d;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[y][i] *= a.out_scale;
                if (gate) v[y][i] *= 1.0f / (1.0f + __expf(-ld_f(gate + n * a.gate_ld + (a.gate_heads ? h : col + i))));
            }
            if (a.out_dtype == JL_OUT_F32) st4_f((float *)a.out + n * a.out_ld + col, v[y]);
            else st4_f((bf16_t *)a.out + n * a.out_ld + col, v[y]);
        }
    }
}

extern "C" int jl_attn_talk_ok(int dtype, int32_t H, int32_t G, int32_t D, int32_t Dv, int64_t k_ld, int64_t v_ld) {
    return dtype == JL_BF16 && G > 0 && H % G == 0 && H <= AM_HEADS && G <= 8 && D > 0 && D % 8 == 0 && D <= 128 && Dv > 0 && Dv % 8 == 0 && Dv <= 128 && k_ld % 8 == 0 && v_ld % 8 == 0;
}
extern "C" int jl_attn_talk_tile_rows(int32_t H, int32_t G, int32_t wide) { return (wide ? 128 : 32) / (H / G); }
extern "C" int64_t jl_attn_talk_scratch_floats(int32_t tiles, int32_t TQ, int32_t H, int32_t G, int32_t Dv, int32_t splits) {
    return (int64_t)tiles * TQ * splits * H * (G * (int64_t)Dv + 2);
}

template <int KU, int VU, int NW> static int at_launch(const jl_attn_args &a, int pass_tiles, hipStream_t st) {
    const int HF = a.H / a.G;
    const bool spread = a.splits > 1;
    const size_t lds = at_lds_bytes(KU, VU, a.TQ, HF, NW), mix = (size_t)((spread ? a.H * (a.G * a.Dv > 2 * a.splits ? a.G * a.Dv : 2 * a.splits) + a.splits * a.H : 4 * a.H) + a.H * a.H) * 4;
    if (NW > 1 && HF * (a.TQ + AT_KT - 1) > AT_BIAS * 64 * NW) return jl_fail(JL_E_INVALID, "jl_attn_talk: too many biases per tile");
    auto kern = attn_talk_kernel<KU, VU, NW>;
    auto join = spread ? attn_talk_mix_kernel<true> : attn_talk_mix_kernel<false>;
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess && mix > 64 * 1024) e = hipFuncSetAttribute((const void *)join, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mix);
    if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_attn_talk: cannot get %zu bytes of LDS: %s", lds > mix ? lds : mix, hipGetErrorString(e));
    for (int t0 = 0; t0 < a.n_tiles; t0 += pass_tiles) {            // as many tiles at a time as the scratch holds
        const int nt = a.n_tiles - t0 < pass_tiles ? a.n_tiles - t0 : pass_tiles, rows = nt * a.TQ;
        kern<<<dim3((unsigned)(nt * a.splits * a.G * a.G)), 64 * NW, lds, st>>>(a, HF, t0, nt);
        join<<<dim3((unsigned)(spread ? rows : (rows + 3) / 4)), 256, mix, st>>>(a, t0, nt);
    }
    return jl_check_launch("attn_talk_kernel");
}

extern "C" int jl_attn_talk(const jl_attn_args *ap, int32_t wide, int32_t pass_tiles, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_attn_talk: null arguments");
    jl_attn_args a = *ap;
    if (a.n_tiles <= 0) return JL_OK;
    if (!a.q || !a.k_cache || !a.v_cache || !a.out || !a.block_tables || !a.tiles || !a.talk || !a.scratch) return jl_fail(JL_E_INVALID, "jl_attn_talk: null pointer");
    if (!jl_attn_talk_ok(a.dtype, a.H, a.G, a.D, a.Dv, a.k_ld, a.v_ld) || (a.Gv > 0 && a.Gv != a.G) || a.k_ld < (int64_t)a.G * a.D || a.v_ld < (int64_t)a.G * a.Dv ||
        (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)a.scratch) & 15))
        return jl_fail(JL_E_INVALID, "jl_attn_talk: sizes or alignment (ask jl_attn_talk_ok)");
    if (a.sink || a.chunk > 0 || a.softcap > 0.f || (a.lut && !a.rel) || (a.rel && a.lut_len <= 0) || a.page_size <= 0 || a.keep_first < 0)
        return jl_fail(JL_E_INVALID, "jl_attn_talk: no sink, chunks or cap; a lut needs rel, and rel needs lut_len");
    if (a.TQ != jl_attn_talk_tile_rows(a.H, a.G, wide) || a.splits <= 0 || a.splits > 64 || pass_tiles <= 0 || a.out_ld < (int64_t)a.H * a.Dv || a.out_ld % 4 || a.Dv % 4 ||
        (int64_t)(pass_tiles < a.n_tiles ? pass_tiles : a.n_tiles) * a.splits * a.G * a.G > INT32_MAX / 256)
        return jl_fail(JL_E_INVALID, "jl_attn_talk: tiles, splits or output rows");
    if (a.out_dtype != JL_OUT_SAME && a.out_dtype != JL_OUT_F32) return jl_fail(JL_E_INVALID, "jl_attn_talk: unknown out_dtype");
    if ((uintptr_t)a.out & (a.out_dtype == JL_OUT_F32 ? 15 : 7)) return jl_fail(JL_E_INVALID, "jl_attn_talk: output rows start at the borders of four values");
    hipStream_t st = (hipStream_t)stream;
    if (!wide && pass_tiles >= a.n_tiles && jl_attn_token_fits(a, false)) return jl_attn_token_launch(a, false, st);
    const int ku = a.D <= 64 ? 8 : 16, vu = a.Dv <= 64 ? 8 : 16;
#define AT_CASE(K, V) if (ku == K && vu == V) return wide ? at_launch<K, V, 4>(a, pass_tiles, st) : at_launch<K, V, 1>(a, pass_tiles, st)
    AT_CASE(8, 8); AT_CASE(8, 16); AT_CASE(16, 8); AT_CASE(16, 16);
#undef AT_CASE
    return jl_fail(JL_E_INVALID, "jl_attn_talk: unsupported size");
}

// ---- without mixed heads: tiles of up to 32 rows, each wavefront with keys of its own (jl_attn_token.hip) -----------------------------------------
extern "C" int jl_attn_narrow_ok(int dtype, int32_t H, int32_t G, int32_t Gv, int32_t D, int32_t Dv, int64_t k_ld, int64_t v_ld) {
    return jl_attn_talk_ok(dtype, H, G, D, Dv, k_ld, v_ld) && Gv > 0 && G % Gv == 0;
}

extern "C" int jl_attn_narrow(const jl_attn_args *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_attn_narrow: null arguments");
    jl_attn_args a = *ap;
    if (a.n_tiles <= 0) return JL_OK;
    if (!a.q || !a.k_cache || !a.v_cache || !a.out || !a.block_tables || !a.tiles || (a.splits > 1 && !a.scratch)) return jl_fail(JL_E_INVALID, "jl_attn_narrow: null pointer");
    if (!jl_attn_narrow_ok(a.dtype, a.H, a.G, a.Gv, a.D, a.Dv, a.k_ld, a.v_ld) || a.k_ld < (int64_t)a.G * a.D || a.v_ld < (int64_t)a.Gv * a.Dv ||
        (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)a.scratch) & 15))
        return jl_fail(JL_E_INVALID, "jl_attn_narrow: sizes or alignment (ask jl_attn_narrow_ok)");
    if (a.talk || a.rel || a.keep_first > 0 || (a.chunk > 0 && a.window > 0) || a.page_size <= 0) return jl_fail(JL_E_INVALID, "jl_attn_narrow: no bias, mixed heads or kept tokens; chunks exclude a window");
    if (a.TQ != jl_attn_talk_tile_rows(a.H, a.G, 0) || a.splits <= 0 || a.splits > 64 || a.out_ld < (int64_t)a.H * a.Dv || a.out_ld % 4 ||
        (int64_t)a.n_tiles * a.splits * a.G > INT32_MAX / 64 || (int64_t)a.n_tiles * a.TQ * a.H > INT32_MAX)
        return jl_fail(JL_E_INVALID, "jl_attn_narrow: tiles, splits or output rows");
    if (a.out_dtype != JL_OUT_SAME && a.out_dtype != JL_OUT_F32) return jl_fail(JL_E_INVALID, "jl_attn_narrow: unknown out_dtype");
    if ((uintptr_t)a.out & (a.out_dtype == JL_OUT_F32 ? 15 : 7)) return jl_fail(JL_E_INVALID, "jl_attn_narrow: output rows start at the borders of four values");
    hipStream_t st = (hipStream_t)stream;
    if (a.longest <= 0 || a.longest > a.TQ) a.longest = a.TQ;
    return jl_attn_token_launch(a, false, st);
}
