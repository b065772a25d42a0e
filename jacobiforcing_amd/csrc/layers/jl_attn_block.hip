// jl_attn_block.hip — attention of a draft block: R rows of T new tokens over a cache (one row per prompt, or pages), each token seeing the row's committed keys and
// the block up to itself; a candidate row's block lies in a scratch of its own.
// The structure is jl_attn_rows.hip's (32 (head, token) rows per wavefront, S^T = K Q^T, weights straight into the second product, V^T through ds_read_b64_tr_b16).  Lengths, cache
// rows, pages and scratch rows are read by the kernel, so the host builds no mask and gathers no prefix, and the outputs leave token by token as the next product reads them.
// Two forms.  Many rows: tiles of 128 (head, token) rows, four wavefronts that share every tile of 64 keys, two workgroups per CU.  Few (layer_ops._block_plan draws the line): tiles of 64 rows, and a
// workgroup of eight wavefronts takes four tiles of 32 keys at a time, a pair of wavefronts each; the four groups' sums meet in LDS.  The chip is full with a quarter of the rows, nothing leaves for
// memory between the shares, and no launch joins them.  Where even that leaves CUs idle, keys are shared out over `splits` workgroups too, and a second launch joins the shares.
// What bounds it: the keys' way through LDS, the softmax's issue and the matrix instructions, about as long each; few rows: latency of launch, loads and barriers (15 us with one round of keys and with five;
// loads two rounds ahead changed nothing).  us, bfloat16, 32 tokens, 8 heads of 128 over 2, context 512, before (tiles of 128 rows, keys shared out over up to three workgroups) / now: 64 rows
// 30.2 / 20.6, 32 27.1 / 19.0, 16 23.8 / 18.1, one 16.7 / 16.1; context 4000, one row 42.7 / 25.4, 8 rows 45.4 / 30.7; 32 rows, 14 heads of 64 over 2, context 1000 27.7 / 18.2.  Many rows (scores scaled
// in the exponent's own instruction; rows whose scores are beyond 2^24 apart, ar_factor): 128 rows 35.4 / 30.2; 64 rows of 64, 16 heads over 2, context 1500 111.8 / 93.2; 64 rows, 28 heads of 128 over 4,
// context 1000 79.6 / 67.3; 96 rows of the first, two shares, context 1500 55 / 52.
// Sums scaled only when a maximum has grown by 2^8 would give 4 to 7 % more, but the greatest weight is then no longer 1 but a rounded one: errors against 64 bits of peaked rows grew by 12 %.
// The library's attention with a mask tensor and the copy that its output needs: the first 47, the one row 40, the 14 heads 89, the last two 182 and 199.
#include "jl_attn.h"

// two tiles of KT keys and values per key group and their rows; the groups' sums are joined in the same place
constexpr size_t ab_lds_bytes(int KU, int WM, int KG, int KT) { return (size_t)KG * (2 * 2 * KT * KU * 16 + (KG > 1 && 32 * WM > KT ? 32 * WM : KT) * 8); }

template <int KU, int WM, int KG, int KT>                           // D <= 8 * KU; WM wavefronts of 32 rows, KG groups of them that take every KG-th tile of KT keys
__global__ __launch_bounds__(64 * WM * KG, KG == 1 ? 2 : 1) void attn_block_kernel(jl_block_args a, int row_tiles) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int THREADS = 64 * WM, NHF = KT / 32, NDV = KU / 4, BUF = 2 * KT * KU, PF = KT * KU / THREADS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, kg = wave / WM, tid = threadIdx.x - kg * THREADS, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    const int D = a.D, T = a.T, GT = a.G * T, S = a.splits;
    // workgroups that read the same keys lie eight apart, on one XCD
    const int rt = blockIdx.x / 8 % row_tiles, unit = blockIdx.x / (8 * row_tiles) * 8 + blockIdx.x % 8, c = unit % a.nkv, split = unit / a.nkv % S, r = unit / (a.nkv * S);
    if (r >= a.R) return;
    uint4 *buf0 = (uint4 *)smem + kg * 2 * BUF;
    int *tokS = (int *)((uint4 *)smem + KG * 2 * BUF) + kg * 2 * KT;      // [2][KT] rows of D elements in the cache, or ~ rows in the scratch
    const int cand = a.cand_rows > 0 ? a.row_cand[r] : -1, page_size = a.page_size;
    int kv = a.kv_len[r], len = a.row_len[r];
    kv = kv < 0 ? 0 : kv < a.max_keys ? kv : a.max_keys;
    len = len < 0 ? 0 : len < T ? len : T;
    const int n_keys = kv + len < a.max_keys ? kv + len : a.max_keys;
    const int n_kt = (n_keys + KT - 1) / KT, share = (n_kt + S - 1) / S, t_lo = split * share, t_hi = t_lo + share < n_kt ? t_lo + share : n_kt;
    int first_block = 0;
    if (!a.tables) {
        first_block = a.row_prompt[r];
        first_block = first_block < 0 ? 0 : first_block < a.blocks ? first_block : a.blocks - 1;
    }
    const int cand_row = cand < a.cand_rows ? cand : a.cand_rows - 1;
    const bf16_t *K = (const bf16_t *)a.k, *V = (const bf16_t *)a.v, *CK = (const bf16_t *)a.ck, *CV = (const bf16_t *)a.cv;

    const int R = 32 * WM * rt + 32 * wm + l32, t = R % T;            // this lane's row: head R / T of the group, token t; both half-wavefronts hold it
    const bool ok = R < GT;
    const int last = kv + (t + 1 < len ? t + 1 : len) - 1 < n_keys - 1 ? kv + (t + 1 < len ? t + 1 : len) - 1 : n_keys - 1;      // its last key
    const bool scaled = !ar_one_by_one(a.scale);
    ar_bf16x8 qf[KU / 2];
#pragma unroll
    for (int x = 0; x < KU / 2; ++x) {
        ar_s16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
        if (ok && 16 * x + 8 * hi < D) w = *(const ar_s16x8 *)((const bf16_t *)a.q + (((int64_t)r * a.nkv + c) * GT + R) * D + 16 * x + 8 * hi);
        if (scaled && a.scale < 0.f) w ^= (short)0x8000;
        qf[x] = __builtin_bit_cast(ar_bf16x8, w);
    }
    const float c2 = scaled ? fabsf(a.scale * AR_LOG2E) : AR_LOG2E;
    float m_run = -INFINITY, l_run = 0.f, entry = -INFINITY;
    ar_f32x16 acc[NDV];
#pragma unroll
    for (int y = 0; y < NDV; ++y)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[y][i] = 0.f;
    const bool wave_live = 32 * (WM * rt + wm) < GT, wave_full = 32 * (WM * rt + wm) + 31 < GT;

    ar_s16x8 kreg[PF], vreg[PF];
    int tok_next = 0;
    auto look_up = [&](int kt) {
        const int j = kt * KT + tid;
        if (tid >= KT || kt >= t_hi || j >= n_keys) return;
        if (cand >= 0 && j >= kv) { tok_next = ~((cand_row * a.nkv + c) * a.cand_max + (j - kv)); return; }
        int block = first_block, off = j;
        if (a.tables) {
            const int pg = j / page_size;
            block = pg < a.table_cols ? a.tables[(int64_t)r * a.table_ld + pg] : 0;
            block = block < 0 ? 0 : block < a.blocks ? block : a.blocks - 1;
            off = j - pg * page_size;
        }
        tok_next = (block * a.nkv + c) * page_size + off;
    };
    auto tokens_out = [&](int sel) { if (tid < KT) tokS[sel * KT + tid] = tok_next; };
    auto fetch = [&](int kt, const int *tok) {
        const int nk = n_keys - kt * KT < KT ? n_keys - kt * KT : KT;
#pragma unroll
        for (int it = 0; it < PF; ++it) {
            const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) {
                const int x = tok[jj];
                const int64_t at = (int64_t)(x < 0 ? ~x : x) * D + 8 * u;
                kreg[it] = *(const ar_s16x8 *)((x < 0 ? CK : K) + at);
                vreg[it] = *(const ar_s16x8 *)((x < 0 ? CV : V) + at);
            }
        }
    };
    auto stash = [&](int kt, uint4 *Ks) {                           // columns beyond D and rows beyond the last key as zeros
        const int nk = n_keys - kt * KT < KT ? n_keys - kt * KT : KT;
        const ar_s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int it = 0; it < PF; ++it) {
            const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
            const bool in = jj < nk && 8 * u < D;
            Ks[jj * KU + ar_key_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, in ? kreg[it] : zero);
            Ks[KT * KU + jj * KU + ar_value_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, in ? vreg[it] : zero);
        }
    };
    const int first = t_lo + kg;                                    // this group's first tile
    look_up(first);
    tokens_out(0);
    look_up(first + KG);
    tokens_out(1);
    __syncthreads();
    if (first < t_hi) {
        fetch(first, tokS);
        stash(first, buf0);
    }
    __syncthreads();
    for (int kt = first, sel = 0; kt - kg < t_hi; kt += KG, sel ^= 1) {      // as many rounds for every group
        if (kt + KG < t_hi) fetch(kt + KG, tokS + (sel ^ 1) * KT);
        look_up(kt + 2 * KG);
        const uint4 *Ks = buf0 + sel * BUF;
        const int j0 = kt * KT;
        if (wave_live && kt < t_hi) {
            ar_f32x16 sc[NHF];
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[hf][i] = 0.f;
#pragma unroll
            for (int x = 0; x < KU / 2; ++x)
#pragma unroll
                for (int hf = 0; hf < NHF; ++hf) {
                    const int row = 32 * hf + l32;
                    sc[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ar_bf16x8, Ks[row * KU + ar_key_unit<KU>(row, 2 * x + hi)]), qf[x], sc[hf], 0, 0, 0);
                }
            if (!scaled)
#pragma unroll
                for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                    for (int i = 0; i < 16; ++i) sc[hf][i] *= a.scale;
            if (!wave_full || j0 + KT > kv) {                       // not committed keys only, which every row sees
                const int upto = ok ? last - j0 : -1;
#pragma unroll
                for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                    for (int i = 0; i < 16; ++i) sc[hf][i] = 32 * hf + 8 * (i >> 2) + 4 * hi + (i & 3) <= upto ? sc[hf][i] : -INFINITY;
            }
            float mx = sc[0][0];
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                for (int i = hf == 0 ? 1 : 0; i < 16; ++i) mx = fmaxf(mx, sc[hf][i]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run, mx * c2);
            float factor = c2;
            if (__any(m_new > entry)) {                             // after the first tiles a row's maximum seldom moves (a stale one would leave the greatest weight inexact)
                const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new > -INFINITY ? m_new : 0.f));
                m_run = m_new;
                entry = ar_entry(m_run);
                factor = ar_factor(sc, c2, m_run);
                l_run *= alpha;
#pragma unroll
                for (int y = 0; y < NDV; ++y)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[y][i] *= alpha;
            }
            const float m_sub = m_run > -INFINITY ? m_run : 0.f;
            float sum = 0.f;
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                for (int i = 0; i < 16; ++i) { sc[hf][i] = __builtin_amdgcn_exp2f(fmaf(sc[hf][i], factor, -m_sub)); sum += sc[hf][i]; }
            l_run += sum;
            const char *Vs = (const char *)(Ks + KT * KU);
            const int vk = 4 * hi + ((lane & 15) >> 2), vc8 = 8 * (lane & 1), vu = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);      // this lane's key, half unit and unit of a turned block
#pragma unroll
            for (int hf = 0; hf < NHF; ++hf)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    ar_f32x8 pf;
#pragma unroll
                    for (int x = 0; x < 8; ++x) pf[x] = sc[hf][8 * s + x];
                    const ar_bf16x8 pb = __builtin_convertvector(pf, ar_bf16x8);
#pragma unroll
                    for (int y = 0; y < NDV; ++y) {
                        ar_s16x4 half[2];
#pragma unroll
                        for (int z = 0; z < 2; ++z) {
                            const int key = 32 * hf + 16 * s + 8 * z + vk;
                            half[z] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ar_lds_s16x4 *)(Vs + 16 * (key * KU + ar_value_unit<KU>(key, 4 * y + vu)) + vc8));
                        }
                        const ar_s16x8 va = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
                        acc[y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ar_bf16x8, va), pb, acc[y], 0, 0, 0);
                    }
                }
        }
        if (kt + KG < t_hi) stash(kt + KG, buf0 + (sel ^ 1) * BUF);
        tokens_out(sel);
        __syncthreads();
    }
    l_run += __shfl_xor(l_run, 32, 64);
    if constexpr (KG > 1) {                                         // the groups' sums meet in LDS: a wavefront joins its rows' columns 32 kg .. 32 kg + 31
        ar_f32x4 *sums = (ar_f32x4 *)smem;                          // [KG][WM][NDV][4][64]
        float *ml = (float *)((uint4 *)smem + KG * 2 * BUF);        // [KG][WM][32] greatest exponents, then the weights' sums
        static_assert(KG * WM * NDV * 4 * 64 <= KG * 2 * BUF && NDV <= KG);
        const int mine = kg * WM + wm;
#pragma unroll
        for (int y = 0; y < NDV; ++y)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                ar_f32x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = acc[y][4 * g + x];
                sums[((mine * NDV + y) * 4 + g) * 64 + lane] = v;
            }
        if (hi == 0) {
            ml[mine * 32 + l32] = m_run;
            ml[(KG * WM + mine) * 32 + l32] = l_run;
        }
        __syncthreads();
        float w[KG];
        bool any[KG];
        m_run = -INFINITY;
        l_run = 0.f;
#pragma unroll
        for (int g = 0; g < KG; ++g) m_run = fmaxf(m_run, ml[(g * WM + wm) * 32 + l32]);
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            const float l = ml[(KG * WM + g * WM + wm) * 32 + l32];
            any[g] = l != 0.f;                                      // an empty share's sums are not read
            w[g] = any[g] ? __builtin_amdgcn_exp2f(ml[(g * WM + wm) * 32 + l32] - m_run) : 0.f;
            l_run += w[g] * l;
        }
        if (kg >= NDV) return;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            ar_f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                const ar_f32x4 x = sums[(((g * WM + wm) * NDV + kg) * 4 + q) * 64 + lane];
                if (any[g]) v += w[g] * x;
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[0][4 * q + x] = v[x];
        }
    }
    if (!ok) return;
    const float inv = l_run != 0.f ? 1.0f / l_run : 0.f;
    const int64_t width = (int64_t)a.nkv * a.G * D, row = ((int64_t)r * T + t) * width + (int64_t)(c * a.G + R / T) * D;
    const int64_t rows = (int64_t)a.R * T * a.nkv * a.G;            // a split's (token, head) rows
    if (S > 1 && hi == 0 && (KG == 1 || kg == 0)) {
        float *ml = a.scratch + S * rows * D + (split * rows + row / D) * 2;
        ml[0] = m_run;
        ml[1] = l_run;
    }
    if (S > 1 && l_run == 0.f) return;                             // an empty share is not read
#pragma unroll
    for (int y = 0; y < (KG > 1 ? 1 : NDV); ++y)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = 32 * (KG > 1 ? kg : y) + 8 * g + 4 * hi;      // registers 4g .. 4g + 3: four consecutive columns
            if (col >= D) continue;
            float v[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) v[x] = acc[y][4 * g + x] * (S > 1 ? 1.0f : inv);
            if (S > 1) st4_f(a.scratch + split * rows * D + row + col, v);
            else st4_f((bf16_t *)a.out + row + col, v);
        }
}

// a (token, head) row's shares joined: 32 lanes per row, four columns each
__global__ __launch_bounds__(256) void attn_block_join_kernel(jl_block_args a, int64_t rows) {
    const int64_t row = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    if (row >= rows) return;
    const int S = a.splits, D = a.D, lane = threadIdx.x & 31;
    const float *ml = a.scratch + S * rows * D + row * 2;
    float M = -INFINITY, L = 0.f;
    for (int s = 0; s < S; ++s) M = fmaxf(M, ml[s * rows * 2]);
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < S; ++s) {
        const float m = ml[s * rows * 2], l = ml[s * rows * 2 + 1];
        if (l == 0.f) continue;
        const float w = __builtin_amdgcn_exp2f(m - M);
        L += w * l;
        if (4 * lane < D) {
            const float4 p = *(const float4 *)(a.scratch + (s * rows + row) * D + 4 * lane);
            v[0] += w * p.x; v[1] += w * p.y; v[2] += w * p.z; v[3] += w * p.w;
        }
    }
    const float inv = L != 0.f ? 1.0f / L : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= inv;
    if (4 * lane < D) st4_f((bf16_t *)a.out + row * D + 4 * lane, v);
}

// where the block's keys go: token t of row r at position p to row_prompt * S_max + p of the cache, or (row_cand not negative) to row_cand * T_max + t of the scratch; -1: nowhere
__global__ __launch_bounds__(256) void block_slots_kernel(const int32_t *__restrict__ positions, const int32_t *__restrict__ row_prompt, const int32_t *__restrict__ row_cand,
                                                          const int32_t *__restrict__ row_len, int64_t n, int T, int64_t S_max, int64_t T_max, int64_t *__restrict__ slot_main,
                                                          int64_t *__restrict__ slot_cand) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int r = (int)(e / T), t = (int)(e - (int64_t)r * T), cand = row_cand[r];
    const bool valid = t < row_len[r];
    slot_main[e] = valid && cand < 0 ? row_prompt[r] * S_max + positions[e] : -1;
    if (slot_cand) slot_cand[e] = valid && cand >= 0 ? cand * T_max + t : -1;
}

extern "C" int jl_block_slots(const int32_t *positions, const int32_t *row_prompt, const int32_t *row_cand, const int32_t *row_len, int64_t R, int32_t T, int64_t S_max, int64_t T_max,
                              int64_t *slot_main, int64_t *slot_cand, void *stream) {
    if (R <= 0 || T <= 0) return JL_OK;
    if (!positions || !row_prompt || !row_cand || !row_len || !slot_main) return jl_fail(JL_E_INVALID, "jl_block_slots: null pointer");
    if (R * T / 256 >= INT32_MAX) return jl_fail(JL_E_INVALID, "jl_block_slots: too many rows");
    block_slots_kernel<<<dim3((unsigned)((R * T + 255) / 256)), 256, 0, (hipStream_t)stream>>>(positions, row_prompt, row_cand, row_len, R * T, T, S_max, T_max, slot_main, slot_cand);
    return jl_check_launch("block_slots_kernel");
}

extern "C" int jl_attn_block_ok(int dtype, int32_t D) { return dtype == JL_BF16 && D > 0 && D % 8 == 0 && D <= 128; }
extern "C" int64_t jl_attn_block_scratch_floats(int64_t R, int32_t T, int32_t nkv, int32_t G, int32_t D, int32_t splits) { return splits > 1 ? splits * R * T * nkv * G * (D + 2) : 0; }

template <int KU, int WM, int KG, int KT> static int ab_launch(const jl_block_args &a, hipStream_t st) {
    constexpr size_t lds = ab_lds_bytes(KU, WM, KG, KT);
    auto kern = attn_block_kernel<KU, WM, KG, KT>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_attn_block: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    const int row_tiles = (a.G * a.T + 32 * WM - 1) / (32 * WM);
    const int64_t units = ((int64_t)a.R * a.nkv * a.splits + 7) / 8 * 8;
    if (units * row_tiles > INT32_MAX) return jl_fail(JL_E_INVALID, "jl_attn_block: more rows than 32 bits count");
    kern<<<dim3((unsigned)(units * row_tiles)), 64 * WM * KG, lds, st>>>(a, row_tiles);
    if (a.splits > 1) {
        const int64_t rows = (int64_t)a.R * a.T * a.nkv * a.G;
        attn_block_join_kernel<<<dim3((unsigned)((rows + 7) / 8)), 256, 0, st>>>(a, rows);
    }
    return jl_check_launch("attn_block_kernel");
}

extern "C" int jl_attn_block(const jl_block_args *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_attn_block: null arguments");
    const jl_block_args &a = *ap;
    if (a.R <= 0 || a.T <= 0) return JL_OK;
    if (!a.q || !a.k || !a.v || !a.out || !a.kv_len || !a.row_len || (!a.tables && !a.row_prompt) || (a.cand_rows > 0 && (!a.ck || !a.cv || !a.row_cand)) || (a.splits > 1 && !a.scratch))
        return jl_fail(JL_E_INVALID, "jl_attn_block: null pointer");
    if (!jl_attn_block_ok(JL_BF16, a.D) || a.nkv <= 0 || a.G <= 0 || a.page_size <= 0 || a.blocks <= 0 || a.max_keys < 0 || a.splits <= 0 || (a.cand_rows > 0 && a.cand_max < a.T) ||
        (a.tables ? a.table_cols <= 0 || a.table_ld < a.table_cols : a.max_keys > a.page_size) ||
        (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.ck | (uintptr_t)a.cv | (uintptr_t)a.out | (uintptr_t)a.scratch) & 15))
        return jl_fail(JL_E_INVALID, "jl_attn_block: sizes or alignment (ask jl_attn_block_ok)");
    if ((int64_t)a.blocks * a.nkv * a.page_size > INT32_MAX || (int64_t)(a.cand_rows > 0 ? a.cand_rows : 0) * a.nkv * a.cand_max > INT32_MAX || a.G * (int64_t)a.T > INT32_MAX - 128 ||
        (int64_t)a.R * a.splits * a.nkv > INT32_MAX)
        return jl_fail(JL_E_INVALID, "jl_attn_block: more rows than 32 bits count");
    hipStream_t st = (hipStream_t)stream;
    if (a.grouped) return a.D <= 64 ? ab_launch<8, 2, 4, 32>(a, st) : ab_launch<16, 2, 4, 32>(a, st);
    return a.D <= 64 ? ab_launch<8, 4, 1, 64>(a, st) : ab_launch<16, 4, 1, 64>(a, st);
}
