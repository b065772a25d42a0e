// jl_attn_token.hip — attention of single tokens and of portions of a few: every wavefront has keys of its own, the eight of a workgroup meet once, at the end.
// Rows of the products are (query, head) pairs, up to 16 (NB = 1) or 32: the heads of one key head, or with mixed heads all of them (a row takes its scores from its own key head's product, so that
// every key and value is read once for up to two value heads and a key that is not finite stays with its own heads).  A wavefront walks every eighth tile of 16 or 32 keys: a key's units go from memory
// straight into the lanes that hold the operand of S^T = K Q^T, values through LDS of the wavefront's own, from where they are read turned (ds_read_b64_tr_b16) for O^T = V^T P^T; a lane holds
// values of ONE row, so that only the maximum is exchanged, with three other lanes.  The next tile's loads leave before this one's weights are formed, and no wavefront waits for another before
// the end, where all scale their sums to the row's maximum and add them up through LDS.
// What bounds it: reading keys and values where they are many (32 tokens at 2048, 16 heads of 128 over 4: 4.6 TB/s), else one trip to memory behind another: tile, page, keys, and the join's.  The forms before
// had four wavefronts meet at three barriers per 32 keys (jl_attn_sweep.hip), or one wavefront per workgroup, whose shares (16 to 64 of a row) all went through memory.  us of both launches, before / so:
//   32 tokens at 2048   16 heads of 128 over 4  43 / 31    8 over 1 at 1500  22 / 13    latent of 512 + 64, 16 heads  55 / 30    of 256 + 64 (48 at 1000)  29 / 17    of 128 + 32 (30 at 1500), 8 heads  19 / 10
//   one token at 700, 8 over 2  16 / 10     at 16000  46 / 20     200 tokens at 1000  33 / 21     8 x 40 at 500  26 / 18     777 + 389 beside 30, latent of 128 + 32, 8 heads  59 / 32
//   mixed heads, window 1024: 32 tokens at 2048, 8 over 2  49 / 18, 16 over 4  107 / 29;  one at 700  27 / 13
#include "jl_attn.h"

constexpr int TK_NW = 8;

// of a score (a sink, a share's maximum) less the row's maximum.  Scores stay as they are: times log2(e) the last third of the largest binade would be infinite
__device__ __forceinline__ float tk_exp(float d) { return __builtin_amdgcn_exp2f(d * 1.44269504088896341f); }

typedef float tk_f32x4 __attribute__((ext_vector_type(4)));
typedef float tk_f32x8 __attribute__((ext_vector_type(8)));

// unit u of key k lies at u ^ tk_swap(k) in its row of U units: sixteen keys that are written together, and eight keys by 32 bytes that are read turned together, meet different banks
template <int U> __device__ __forceinline__ int tk_swap(int k) { return U % 16 == 0 ? (k & 3) << 2 | (k >> 2 & 1) << 1 | (k >> 3 & 1) : (k >> 1 & 3) << 1 | (k >> 3 & 1); }

// Z: sixteens of keys per tile; KX: 32 depths of a key at most; VY: sixteens of value columns at most; NG: key heads (mixed heads; else 1); GV: value heads collected; VIK: values are the keys' first columns
template <int NB, int Z, int KX, int VY, int NG, int GV, bool VIK, bool MIX> struct TkSizes {
    static constexpr int U = 2 * VY, OWN = GV * Z * 16 * U, SLOT = GV * NB * VY * 64, QU = NB * KX > 8 ? NB * KX * 64 : 0;      // 16-byte units: a wavefront's values, its sums, the queries
    static constexpr int BODY = TK_NW * OWN > TK_NW / 2 * SLOT ? TK_NW * OWN : TK_NW / 2 * SLOT;
    static constexpr size_t BYTES = (size_t)(BODY + QU) * 16 + TK_NW * NB * 16 * 8;
};

template <int NB, int Z, int KX, int VY, int NG, int GV, bool VIK, bool MIX>
__global__ __launch_bounds__(64 * TK_NW, 2) void attn_token_kernel(jl_attn_args a, int rep, int tile0) {
    typedef TkSizes<NB, Z, KX, VY, NG, GV, VIK, MIX> Sizes;
    constexpr int KT = 16 * Z, U = Sizes::U, VX = VY / 2, OWN = Sizes::OWN, SLOT = Sizes::SLOT;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int H = a.H, D = a.D, Dv = a.Dv, S = a.splits;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
    // sides: key heads, or with mixed heads runs of GV value heads
    const int sides = MIX ? a.G / GV : a.G, side = blockIdx.x % sides, rest = blockIdx.x / sides, split = rest % S, ti = tile0 + rest / S;
    const int *tile = a.tiles + 4 * (int64_t)ti;
    const int b = tile[0], i0 = tile[1], cnt = tile[2], row0 = tile[3];
    if (b < 0 || cnt <= 0) return;                                  // the whole workgroup
    const int heads = MIX ? H : rep, h0 = MIX ? 0 : side * rep;     // rows: (query R / heads, head h0 + R % heads)
    uint4 *const own = (uint4 *)smem + wave * OWN;                  // this wavefront's values
    uint4 *const qS = (uint4 *)smem + Sizes::BODY;
    float *const mS = (float *)(qS + Sizes::QU), *const lS = mS + TK_NW * NB * 16;
    const int window = a.window > 0 ? a.window : 0x3fffffff, chunk = MIX ? 0 : a.chunk, keep_first = MIX ? a.keep_first : 0;
    auto lowest = [&](int i) { return chunk > 0 ? i - i % chunk : i - window + 1; };        // first key that query i sees
    const int i_max = i0 + cnt - 1, lo = lowest(i0) > 0 ? lowest(i0) : 0, kept = keep_first < lo ? keep_first : lo;      // kept first tokens in front of the window
    const int kept_tiles = (kept + KT - 1) / KT, n_kt = kept_tiles + (i_max + 1 - lo + KT - 1) / KT;
    const int share = (n_kt + S - 1) / S, t_lo = split * share, t_hi = t_lo + share < n_kt ? t_lo + share : n_kt;
    auto first_of = [&](int t) { return t < kept_tiles ? t * KT : lo + (t - kept_tiles) * KT; };
    auto keys_of = [&](int t) { const int e = (t < kept_tiles ? kept : i_max + 1) - first_of(t); return e < KT ? e : KT; };
    const int *bt = a.block_tables + (int64_t)b * a.bt_stride;
    const bf16_t *kc = (const bf16_t *)a.k_cache + (MIX ? 0 : (int64_t)side * D), *vc = (const bf16_t *)a.v_cache + (int64_t)(MIX ? side * GV : side % a.Gv) * Dv;
    const int page_shift = (a.page_size & (a.page_size - 1)) == 0 ? __builtin_ctz(a.page_size) : -1;

    // this lane's rows
    int ii[NB], h[NB], q_lo[NB];
    bool ok[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        ii[nb] = (16 * nb + l16) / heads;
        h[nb] = h0 + 16 * nb + l16 - ii[nb] * heads;
        ok[nb] = ii[nb] < a.longest && ii[nb] < cnt;
        q_lo[nb] = lowest(i0 + ii[nb]);
    }
    auto q_unit = [&](int nb, int x) {
        uint4 w = make_uint4(0, 0, 0, 0);
        if (ok[nb] && 8 * (4 * x + quad) < D) w = *(const uint4 *)((const bf16_t *)a.q + ((int64_t)(row0 + ii[nb]) * H + h[nb]) * D + 8 * (4 * x + quad));
        return w;
    };
    uint4 qf[Sizes::QU ? 1 : NB * KX];
    if constexpr (Sizes::QU == 0) {
#pragma unroll
        for (int e = 0; e < NB * KX; ++e) qf[e] = q_unit(e / KX, e % KX);
    } else {
        for (int x = wave; x < KX; x += TK_NW)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) qS[(nb * KX + x) * 64 + lane] = q_unit(nb, x);
        __syncthreads();
    }
    int key_head[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) key_head[nb] = NG == 1 ? 0 : h[nb] / rep;
    float m_run[NB], l_run[NB];
    tk_f32x4 acc[GV][NB][VY];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m_run[nb] = -INFINITY;
        l_run[nb] = 0.f;
#pragma unroll
        for (int g = 0; g < GV; ++g)
#pragma unroll
            for (int y = 0; y < VY; ++y) acc[g][nb][y] = (tk_f32x4){0.f, 0.f, 0.f, 0.f};
    }

    // this lane's keys of a tile: l16 and l16 + 16 (one that does not exist repeats the last; its values are put to zero); of each the units 4 x + quad
    auto token = [&](int t, int z) {
        const int nk = keys_of(t), k = 16 * z + l16, j = first_of(t) + (k < nk ? k : nk - 1), pg = page_shift >= 0 ? j >> page_shift : j / a.page_size;
        return bt[pg] * a.page_size + (j - pg * a.page_size);
    };
    uint4 kr[NG][Z][KX], vr[VIK ? 1 : GV][Z][VIK ? 1 : VX];
    int tok[Z], row_of_bias[MIX ? 4 * Z : 1];
    auto load = [&]() {
#pragma unroll
        for (int z = 0; z < Z; ++z) {
            const bf16_t *kp = kc + (int64_t)tok[z] * a.k_ld + 8 * quad, *vp = vc + (int64_t)tok[z] * a.v_ld + 8 * quad;
#pragma unroll
            for (int c = 0; c < NG; ++c)
#pragma unroll
                for (int x = 0; x < KX; ++x) {
                    kr[c][z][x] = make_uint4(0, 0, 0, 0);
                    if (8 * (4 * x + quad) < D) kr[c][z][x] = *(const uint4 *)(kp + c * D + 32 * x);
                }
            if constexpr (!VIK)
#pragma unroll
                for (int g = 0; g < GV; ++g)
#pragma unroll
                    for (int x = 0; x < VX; ++x)
                        if (8 * (4 * x + quad) < Dv) vr[g][z][x] = *(const uint4 *)(vp + g * Dv + 32 * x);
        }
    };
    // rows of the bias table for this lane's scores: keys 16 z + 4 quad + r
    auto bias_rows = [&](int t) {
        if constexpr (MIX) {
            if (!a.rel) return;
            const int j0 = first_of(t);
#pragma unroll
            for (int e = 0; e < 4 * Z; ++e) {
                int n = i0 + ii[0] - (j0 + 16 * (e >> 2) + 4 * quad + (e & 3));
                n = n < 0 ? 0 : n < a.lut_len ? n : a.lut_len - 1;
                row_of_bias[e] = a.lut ? a.lut[n] : n;
            }
        }
    };
    auto look_up = [&](int t) {
#pragma unroll
        for (int z = 0; z < Z; ++z) tok[z] = token(t, z);
    };
    auto sync = [] {                                                // LDS written by some lanes is read by others of the same wavefront
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    int t = t_lo + wave;
    if (t < t_hi) {
        look_up(t);
        load();
        bias_rows(t);
        if (t + TK_NW < t_hi) look_up(t + TK_NW);
    }
    for (; t < t_hi; t += TK_NW) {
        const int j0 = first_of(t), nk = keys_of(t);
        // where this lane writes and reads values, formed anew for every tile: kept, the addresses take the registers of the rows on their way
        int put = quad ^ tk_swap<U>(l16), get = (lane >> 1 & 1) ^ tk_swap<U>(4 * quad + (l16 >> 2));
        asm("" : "+v"(put), "+v"(get));
        float bias[MIX ? 4 * Z : 1];
        if constexpr (MIX)
            if (a.rel)
#pragma unroll
                for (int e = 0; e < 4 * Z; ++e) bias[e] = a.rel[(int64_t)row_of_bias[e] * H + h[0]];
        // values into this wavefront's LDS
        sync();
#pragma unroll
        for (int z = 0; z < Z; ++z) {
            const bool real = 16 * z + l16 < nk;
#pragma unroll
            for (int g = 0; g < GV; ++g)
#pragma unroll
                for (int x = 0; x < VX; ++x) {
                    const uint4 v = VIK ? kr[0][z][x < KX ? x : 0] : vr[VIK ? 0 : g][z][VIK ? 0 : x];
                    own[((g * Z + z) * 16 + l16) * U + (4 * x ^ put)] = make_uint4(real ? v.x : 0, real ? v.y : 0, real ? v.z : 0, real ? v.w : 0);
                }
        }
        tk_f32x4 sc[NB][Z];
#pragma unroll
        for (int c = 0; c < NG; ++c) {
            tk_f32x4 of[NB][Z];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int z = 0; z < Z; ++z) of[nb][z] = (tk_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < KX; ++x)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const ar_bf16x8 q = __builtin_bit_cast(ar_bf16x8, Sizes::QU ? qS[(nb * KX + x) * 64 + lane] : qf[Sizes::QU ? 0 : nb * KX + x]);
#pragma unroll
                    for (int z = 0; z < Z; ++z) of[nb][z] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ar_bf16x8, kr[c][z][x]), q, of[nb][z], 0, 0, 0);
                }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int z = 0; z < Z; ++z)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sc[nb][z][r] = c == 0 || key_head[nb] == c ? of[nb][z][r] : sc[nb][z][r];
        }
        // the next tile's rows travel from here on
        if (t + TK_NW < t_hi) {
            load();
            bias_rows(t + TK_NW);
            if (t + 2 * TK_NW < t_hi) look_up(t + 2 * TK_NW);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int qi = i0 + ii[nb], first = ok[nb] ? q_lo[nb] - j0 : KT, last = qi - j0 < nk - 1 ? qi - j0 : nk - 1, keep = ok[nb] ? keep_first - j0 : 0;
            float mx = -INFINITY;
            if (!MIX && a.softcap > 0.f) {
#pragma unroll
                for (int z = 0; z < Z; ++z)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sc[nb][z][r] = soft_cap_fast(sc[nb][z][r] * a.scale, a.softcap);
            } else if (MIX && a.rel) {
#pragma unroll
                for (int z = 0; z < Z; ++z)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sc[nb][z][r] = fmaf(sc[nb][z][r], a.scale, bias[MIX ? 4 * z + r : 0]);
            } else {
#pragma unroll
                for (int z = 0; z < Z; ++z) sc[nb][z] *= a.scale;
            }
#pragma unroll
            for (int z = 0; z < Z; ++z)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int kk = 16 * z + 4 * quad + r;
                    float s = sc[nb][z][r];
                    s = (kk >= first || kk < keep) && kk <= last ? s : -INFINITY;
                    sc[nb][z][r] = s;
                    mx = fmaxf(mx, s);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run[nb], mx), m_sub = m_new > -INFINITY ? m_new : 0.f;      // a row that has seen no key yet: all weights are zero
            const float alpha = tk_exp(m_run[nb] - m_sub);
            float sum = 0.f;
#pragma unroll
            for (int z = 0; z < Z; ++z)
#pragma unroll
                for (int r = 0; r < 4; ++r) { sc[nb][z][r] = tk_exp(sc[nb][z][r] - m_sub); sum += sc[nb][z][r]; }
            l_run[nb] = l_run[nb] * alpha + sum;
            m_run[nb] = m_new;
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int g = 0; g < GV; ++g)
#pragma unroll
                    for (int y = 0; y < VY; ++y) acc[g][nb][y] *= alpha;
            }
        }
        sync();
        const char *Vs = (const char *)own + 8 * (lane & 1);
        const int vk = 4 * quad + (l16 >> 2);                       // this lane's key of a turned block
        if constexpr (Z == 2) {
            ar_bf16x8 ph[NB], pl[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const tk_f32x4 lo4 = sc[nb][0], hi4 = sc[nb][Z - 1];
                const tk_f32x8 pf = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
                ph[nb] = __builtin_convertvector(pf, ar_bf16x8);
                pl[nb] = __builtin_convertvector(pf - __builtin_convertvector(ph[nb], tk_f32x8), ar_bf16x8);
            }
#pragma unroll
            for (int g = 0; g < GV; ++g)
#pragma unroll
                for (int y = 0; y < VY; ++y) {
                    ar_s16x4 half[2];
#pragma unroll
                    for (int z = 0; z < 2; ++z) half[z] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ar_lds_s16x4 *)(Vs + 16 * (((g * Z + z) * 16 + vk) * U + (2 * y ^ get))));
                    const ar_bf16x8 va = __builtin_bit_cast(ar_bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        acc[g][nb][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, ph[nb], acc[g][nb][y], 0, 0, 0);
                        if (MIX) acc[g][nb][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pl[nb], acc[g][nb][y], 0, 0, 0);
                    }
                }
        } else {
            typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
            ar_s16x4 ph[NB], pl[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const bf16x4 h4 = __builtin_convertvector(sc[nb][0], bf16x4), l4 = __builtin_convertvector(sc[nb][0] - __builtin_convertvector(h4, tk_f32x4), bf16x4);
                ph[nb] = __builtin_bit_cast(ar_s16x4, h4);
                pl[nb] = __builtin_bit_cast(ar_s16x4, l4);
            }
#pragma unroll
            for (int g = 0; g < GV; ++g)
#pragma unroll
                for (int y = 0; y < VY; ++y) {
                    const ar_s16x4 va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ar_lds_s16x4 *)(Vs + 16 * ((g * 16 + vk) * U + (2 * y ^ get))));
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        acc[g][nb][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va, ph[nb], acc[g][nb][y], 0, 0, 0);
                        if (MIX) acc[g][nb][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va, pl[nb], acc[g][nb][y], 0, 0, 0);
                    }
                }
        }
    }
    // the eight runs meet: all of them scaled to the row's maximum, the upper four added to the lower four, those added up by everybody
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        l_run[nb] += __shfl_xor(l_run[nb], 16, 64);
        l_run[nb] += __shfl_xor(l_run[nb], 32, 64);
        if (quad == 0) { mS[(wave * NB + nb) * 16 + l16] = m_run[nb]; lS[(wave * NB + nb) * 16 + l16] = l_run[nb]; }
    }
    __syncthreads();                                                // and everybody is done with the values
    float M[NB], L[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        M[nb] = -INFINITY;
        L[nb] = 0.f;
        float f = 0.f;                                              // of this wavefront's sums
#pragma unroll
        for (int w = 0; w < TK_NW; ++w) M[nb] = fmaxf(M[nb], mS[(w * NB + nb) * 16 + l16]);
#pragma unroll
        for (int w = 0; w < TK_NW; ++w) {                           // a sum that is not a number stays one
            const float m = mS[(w * NB + nb) * 16 + l16], e = m > -INFINITY ? tk_exp(m - M[nb]) : 0.f;
            L[nb] += lS[(w * NB + nb) * 16 + l16] * e;
            f = w == wave ? e : f;
        }
        const bool any = m_run[nb] > -INFINITY;
#pragma unroll
        for (int g = 0; g < GV; ++g)
#pragma unroll
            for (int y = 0; y < VY; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[g][nb][y][r] = any ? acc[g][nb][y][r] * f : 0.f;
    }
    tk_f32x4 *const slots = (tk_f32x4 *)smem;
    if (wave >= TK_NW / 2)
#pragma unroll
        for (int g = 0; g < GV; ++g)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int y = 0; y < VY; ++y) slots[(wave - TK_NW / 2) * SLOT + ((g * NB + nb) * VY + y) * 64 + lane] = acc[g][nb][y];
    __syncthreads();
    if (wave < TK_NW / 2)
#pragma unroll
        for (int g = 0; g < GV; ++g)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int y = 0; y < VY; ++y) {
                    tk_f32x4 *at = slots + wave * SLOT + ((g * NB + nb) * VY + y) * 64 + lane;
                    *at = acc[g][nb][y] + *at;
                }
    __syncthreads();
    // four columns of a row per thread and turn
    const int GW = MIX ? a.G : 1;
    const bool whole = !MIX && S == 1;
    const bf16_t *gate = (const bf16_t *)a.gate;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (!ok[nb]) continue;
        const int64_t row = ((int64_t)ti * a.TQ + ii[nb]) * S + split, n = row0 + ii[nb];      // shares: [tile, query][split][head][value head][Dv], maxima and sums [..][head][2] behind all of them
        float inv = 0.f;
        if (whole) {                                                // what the joining launch does with one share
            const float sink = a.sink ? a.sink[h[nb]] : -INFINITY, Ms = fmaxf(sink, M[nb]), w = M[nb] > -INFINITY ? tk_exp(M[nb] - Ms) : 0.f;
            const float Ls = (a.sink ? tk_exp(sink - Ms) : 0.f) + w * L[nb];
            inv = Ls != 0.f ? w * (a.out_scale / Ls) : 0.f;         // a sum that is not a number reaches the outputs
        } else if (wave == 0 && quad == 0 && (!MIX || side == 0)) {
            float *ml = a.scratch + (int64_t)a.n_tiles * a.TQ * S * H * GW * Dv + (row * H + h[nb]) * 2;
            ml[0] = M[nb];
            ml[1] = L[nb];
        }
        for (int y = wave; y < GV * VY; y += TK_NW) {
            const int g = y / VY, col = 16 * (y - g * VY) + 4 * quad;
            if (col >= Dv) continue;
            const tk_f32x4 *at = slots + ((g * NB + nb) * VY + y - g * VY) * 64 + lane;
            tk_f32x4 s = at[0];
#pragma unroll
            for (int w = 1; w < TK_NW / 2; ++w) s += at[w * SLOT];
            float v[4] = {s[0], s[1], s[2], s[3]};
            if (!whole) {
                st4_f(a.scratch + ((row * H + h[nb]) * GW + (MIX ? side * GV + g : 0)) * Dv + col, v);
                continue;
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                v[x] *= inv;
                if (gate) v[x] *= 1.0f / (1.0f + __expf(-ld_f(gate + n * a.gate_ld + (a.gate_heads ? h[nb] : h[nb] * Dv + col + x))));
            }
            if (a.out_dtype == JL_OUT_F32) st4_f((float *)a.out + n * a.out_ld + h[nb] * Dv + col, v);
            else st4_f((bf16_t *)a.out + n * a.out_ld + h[nb] * Dv + col, v);
        }
    }
}

// Mixed heads: w[split][head] = exp(m - M) / L (not a number where L is none or zero, as the softmax of such scores), out_h = sum over heads x of talk[h, x] sum over splits of w O_(x, g(h)), gated.  A
// workgroup has 32 columns of a token's value head: its chain of loads is as long as for all of them, and a token's are on as many CUs.
constexpr int TK_HEADS = 16, TK_SPLITS = 64;
__global__ __launch_bounds__(128) void attn_token_mix_kernel(jl_attn_args a, int chunks) {
    __shared__ float w[TK_SPLITS][TK_HEADS];
    __shared__ float4 sums[TK_HEADS][8];
    const int H = a.H, G = a.G, Dv = a.Dv, S = a.splits, rep = H / G, x = threadIdx.x >> 3, j = threadIdx.x & 7;
    const int at = blockIdx.x % (G * chunks), g = at / chunks, col = 32 * (at - g * chunks) + 4 * j, t = blockIdx.x / (G * chunks), ti = t / a.longest, ii = t - ti * a.longest;
    const int *tile = a.tiles + 4 * (int64_t)ti;
    if (tile[0] < 0 || ii >= tile[2]) return;                       // the whole workgroup
    const int64_t r = (int64_t)ti * a.TQ + ii, n = tile[3] + ii, step = (int64_t)H * G * Dv;
    const float *ml = a.scratch + (int64_t)a.n_tiles * a.TQ * S * step + r * S * H * 2, *po = a.scratch + r * S * step + ((int64_t)x * G + g) * Dv + col;
    const bool in = x < H && col < Dv;
    constexpr int AHEAD = 8;
    float4 p[AHEAD];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) p[s] = in && s < S ? *(const float4 *)(po + s * step) : make_float4(0.f, 0.f, 0.f, 0.f);
    if (x < H) {                                                    // eight lanes per head, every eighth share each
        float M = -INFINITY, L = 0.f;
        for (int s = j; s < S; s += 8) M = fmaxf(M, ml[(s * H + x) * 2]);
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 8));
        for (int s = j; s < S; s += 8) {
            const float m = ml[(s * H + x) * 2], e = m > -INFINITY ? tk_exp(m - M) : 0.f;
            w[s][x] = e;
            L += ml[(s * H + x) * 2 + 1] * e;
        }
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) L += __shfl_xor(L, off, 8);
        const float inv = L > 0.f ? 1.0f / L : NAN;
        for (int s = j; s < S; s += 8) w[s][x] *= inv;
    }
    __syncthreads();
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](float f, float4 v) {                             // an empty share (weight zero) holds zeros
        o.x = fmaf(f, v.x, o.x); o.y = fmaf(f, v.y, o.y); o.z = fmaf(f, v.z, o.z); o.w = fmaf(f, v.w, o.w);
    };
    if (x < H) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s)
            if (s < S) add(w[s][x], p[s]);
#pragma unroll 8
        for (int s = AHEAD; s < S; ++s) add(w[s][x], in ? *(const float4 *)(po + s * step) : make_float4(0.f, 0.f, 0.f, 0.f));
    }
    sums[x][j] = o;
    __syncthreads();
    if (x >= rep || col >= Dv) return;
    const int h = g * rep + x, to = h * Dv + col;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int y = 0; y < H; ++y) {
        const float f = a.talk[h * H + y];
        const float4 q = sums[y][j];
        v[0] = fmaf(f, q.x, v[0]); v[1] = fmaf(f, q.y, v[1]); v[2] = fmaf(f, q.z, v[2]); v[3] = fmaf(f, q.w, v[3]);
    }
    const bf16_t *gate = (const bf16_t *)a.gate;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] *= a.out_scale;
        if (gate) v[i] *= 1.0f / (1.0f + __expf(-ld_f(gate + n * a.gate_ld + (a.gate_heads ? h : to + i))));
    }
    if (a.out_dtype == JL_OUT_F32) st4_f((float *)a.out + n * a.out_ld + to, v);
    else st4_f((bf16_t *)a.out + n * a.out_ld + to, v);
}

// Shares of the keys added up: out = sum over shares of exp(m - M) O / L, the sink as one more share that holds nothing, times the gate.  `per` lanes (a power of two) have a (query, head) row, four columns each
__global__ __launch_bounds__(256) void attn_token_join_kernel(jl_attn_args a, int per, int rows) {
    const int r = blockIdx.x * (256 / per) + threadIdx.x / per, lane = threadIdx.x % per;
    if (r >= rows) return;
    const int H = a.H, Dv = a.Dv, S = a.splits, h = r % H, t = r / H, ti = t / a.longest, ii = t - ti * a.longest;
    const int *tile = a.tiles + 4 * (int64_t)ti;
    if (tile[0] < 0 || ii >= tile[2] || 4 * lane >= Dv) return;
    const int64_t n = tile[3] + ii, rt = (int64_t)ti * a.TQ + ii, step = (int64_t)H * Dv;
    const float *ml = a.scratch + (int64_t)a.n_tiles * a.TQ * S * H * Dv + (rt * S * H + h) * 2, *po = a.scratch + (rt * S * H + h) * Dv + 4 * lane;
    constexpr int AHEAD = 8;
    float4 p[AHEAD];
    float2 st[AHEAD];
    auto fetch = [&](int s0) {                                      // eight shares on their way at once; what there is not counts for nothing
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            p[s] = s0 + s < S ? *(const float4 *)(po + (s0 + s) * step) : make_float4(0.f, 0.f, 0.f, 0.f);
            st[s] = s0 + s < S ? *(const float2 *)(ml + (s0 + s) * H * 2) : make_float2(-INFINITY, 0.f);
        }
    };
    fetch(0);
    const float sink = a.sink ? a.sink[h] : -INFINITY;
    float M = sink;
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) M = fmaxf(M, st[s].x);
#pragma unroll 8
    for (int s = AHEAD; s < S; ++s) M = fmaxf(M, ml[s * H * 2]);
    float L = a.sink ? tk_exp(sink - M) : 0.f, v[4] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](float2 stat, float4 o) {
        const float w = stat.x > -INFINITY ? tk_exp(stat.x - M) : 0.f;
        L = fmaf(w, stat.y, L);                                     // an empty share (m = -inf) holds zeros, or a sum that is not a number
        v[0] = fmaf(w, o.x, v[0]); v[1] = fmaf(w, o.y, v[1]); v[2] = fmaf(w, o.z, v[2]); v[3] = fmaf(w, o.w, v[3]);
    };
    for (int s0 = 0; s0 < S; s0 += AHEAD) {
        if (s0 > 0) fetch(s0);
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) add(st[s], p[s]);
    }
    const float inv = L != 0.f ? a.out_scale / L : 0.f;             // a sum that is not a number reaches the outputs
    const bf16_t *gate = (const bf16_t *)a.gate;
    const int col = h * Dv + 4 * lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] *= inv;
        if (gate) v[i] *= 1.0f / (1.0f + __expf(-ld_f(gate + n * a.gate_ld + (a.gate_heads ? h : col + i))));
    }
    if (a.out_dtype == JL_OUT_F32) st4_f((float *)a.out + n * a.out_ld + col, v);
    else st4_f((bf16_t *)a.out + n * a.out_ld + col, v);
}

bool jl_attn_token_fits(const jl_attn_args &a, bool v_in_k) {
    const bool mixed = a.talk != nullptr;
    const int64_t rows = (int64_t)a.longest * (mixed ? a.H : a.H / a.G);
    if (a.longest <= 0 || a.longest > a.TQ || rows > (mixed ? 16 : 32) || a.dtype != JL_BF16 || a.D % 8 || a.Dv % 8 || a.k_ld % 8 || a.v_ld % 8 || a.out_ld % 4 || a.splits > TK_SPLITS ||
        (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)a.scratch) & 15) || ((uintptr_t)a.out & (a.out_dtype == JL_OUT_F32 ? 15 : 7)) ||
        (int64_t)a.n_tiles * a.longest * a.H * (mixed ? 16 : 1) > INT32_MAX / 4)
        return false;
    if (v_in_k) return !mixed && a.G == 1 && a.Dv <= a.D && a.Dv <= (rows > 16 ? 256 : 512) && a.D <= (a.Dv + 127) / 128 * 128 + 64;
    return a.D <= 128 && a.Dv <= 128 && (!mixed || a.G == 1 || a.G == 2 || a.G == 4);
}

template <int NB, int Z, int KX, int VY, int NG, int GV, bool VIK, bool MIX> static int tk_launch(const jl_attn_args &a, hipStream_t st) {
    constexpr size_t lds = TkSizes<NB, Z, KX, VY, NG, GV, VIK, MIX>::BYTES;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    auto kern = attn_token_kernel<NB, Z, KX, VY, NG, GV, VIK, MIX>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "attn_token_kernel: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    const int per_tile = a.splits * (MIX ? a.G / GV : a.G), most = INT32_MAX / 512 / per_tile;      // up to 2 ** 31 threads a launch
    for (int t0 = 0; t0 < a.n_tiles; t0 += most) kern<<<dim3((unsigned)((a.n_tiles - t0 < most ? a.n_tiles - t0 : most) * per_tile)), 64 * TK_NW, lds, st>>>(a, a.H / a.G, t0);
    return jl_check_launch("attn_token_kernel");
}

int jl_attn_token_launch(const jl_attn_args &a, bool v_in_k, hipStream_t st) {
    const bool half = a.D <= 64 && a.Dv <= 64;
    int rc;
    if (a.talk) {
        if (a.G == 1) rc = half ? tk_launch<1, 2, 2, 4, 1, 1, false, true>(a, st) : tk_launch<1, 2, 4, 8, 1, 1, false, true>(a, st);
        else if (a.G == 2) rc = half ? tk_launch<1, 1, 2, 4, 2, 2, false, true>(a, st) : tk_launch<1, 1, 4, 8, 2, 2, false, true>(a, st);
        else rc = half ? tk_launch<1, 1, 2, 4, 4, 2, false, true>(a, st) : tk_launch<1, 1, 4, 8, 4, 2, false, true>(a, st);
        if (rc != JL_OK) return rc;
        const int chunks = (a.Dv + 31) / 32;
        attn_token_mix_kernel<<<dim3((unsigned)(a.n_tiles * a.longest * a.G * chunks)), 128, 0, st>>>(a, chunks);
        return jl_check_launch("attn_token_mix_kernel");
    }
    const bool two = a.longest * (a.H / a.G) > 16;                  // thirty-two rows
    if (v_in_k) {
        const int nt = (a.Dv + 127) / 128;
        if (two) rc = nt == 1 ? tk_launch<2, 2, 6, 8, 1, 1, true, false>(a, st) : tk_launch<2, 1, 10, 16, 1, 1, true, false>(a, st);
        else rc = nt == 1 ? tk_launch<1, 2, 6, 8, 1, 1, true, false>(a, st) : nt == 2 ? tk_launch<1, 1, 10, 16, 1, 1, true, false>(a, st) :
                  nt == 3 ? tk_launch<1, 1, 14, 24, 1, 1, true, false>(a, st) : tk_launch<1, 1, 18, 32, 1, 1, true, false>(a, st);
    } else if (two) rc = half ? tk_launch<2, 2, 2, 4, 1, 1, false, false>(a, st) : tk_launch<2, 2, 4, 8, 1, 1, false, false>(a, st);
    else rc = half ? tk_launch<1, 2, 2, 4, 1, 1, false, false>(a, st) : tk_launch<1, 2, 4, 8, 1, 1, false, false>(a, st);
    if (rc != JL_OK || a.splits == 1) return rc;
    int per = 8;
    while (4 * per < a.Dv) per *= 2;
    const int rows = a.n_tiles * a.longest * a.H;
    attn_token_join_kernel<<<dim3((unsigned)((rows + 256 / per - 1) / (256 / per))), 256, 0, st>>>(a, per, rows);
    return jl_check_launch("attn_token_join_kernel");
}
