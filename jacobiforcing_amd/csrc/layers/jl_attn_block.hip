// jl_attn_block.hip — attention of a draft block: R rows of T new tokens over a cache (one row per prompt, or pages), each token seeing the row's committed keys and
// the block up to itself; a candidate row's block lies in a scratch of its own.
// The structure is jl_attn_rows.hip's (32 (head, token) rows per wavefront, S^T = K Q^T, weights straight into the second product, V^T through ds_read_b64_tr_b16).  Lengths, cache
// rows, pages and scratch rows are read by the kernel, so the host builds no mask and gathers no prefix, and the outputs leave token by token as the next product reads them.
// A key head's rows (heads of a group times tokens) go in tiles of 128; keys are shared out over `splits` workgroups where there are fewer of them than CUs, and a second launch
// joins the shares (384 workgroups to aim at: one row of 32 tokens, 8 heads over 2, context 512, 28 us whole, 17 shared out; 64 rows 32 and 30).
// What bounds it: the keys' way through LDS and the softmax's issue at two workgroups per CU, and launches below 20 us.  us against the library's attention with a mask tensor and the
// copy that its output needs (bfloat16): 64 rows of 32 tokens, 8 heads of 128 over 2, context 512 47 -> 30; one row 40 -> 17; 64 rows of 64, 16 over 2, context 1500 182 -> 96;
// 32 rows, 14 heads of 64 over 2, context 1000 89 -> 27; 64 rows, 28 heads of 128 over 4, context 1000 199 -> 68.
#include "jl_attn.h"

constexpr int AB_THREADS = 256, AB_KT = 64;
constexpr size_t ab_lds_bytes(int KU) { return 2 * ((size_t)2 * AB_KT * KU * 16 + AB_KT * 4); }

template <int KU>                                                                       // D <= 8 * KU
__global__ __launch_bounds__(AB_THREADS, 2) void attn_block_kernel(jl_block_args a, int row_tiles) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int KT = AB_KT, NDV = KU / 4, BUF = 2 * KT * KU, PF = KT * KU / AB_THREADS;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    const int D = a.D, T = a.T, GT = a.G * T, S = a.splits;
    const int c = blockIdx.x % a.nkv, split = blockIdx.x / a.nkv % S, rt = blockIdx.x / (a.nkv * S) % row_tiles, r = blockIdx.x / (a.nkv * S * row_tiles);
    uint4 *buf0 = (uint4 *)smem;
    int *tokS = (int *)(buf0 + 2 * BUF);                            // [2][KT] rows of D elements in the cache, or ~ rows in the scratch
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
    for (int e = tid; e < 2 * BUF; e += AB_THREADS) buf0[e] = make_uint4(0, 0, 0, 0);      // columns beyond D and rows beyond the last key stay zero or finite

    const int R = 128 * rt + 32 * wave + l32, t = R % T;            // this lane's row: head R / T of the group, token t; both half-wavefronts hold it
    const bool ok = R < GT;
    const int last = kv + (t + 1 < len ? t + 1 : len) - 1 < n_keys - 1 ? kv + (t + 1 < len ? t + 1 : len) - 1 : n_keys - 1;      // its last key
    ar_bf16x8 qf[KU / 2];
#pragma unroll
    for (int x = 0; x < KU / 2; ++x) {
        ar_s16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
        if (ok && 16 * x + 8 * hi < D) w = *(const ar_s16x8 *)((const bf16_t *)a.q + (((int64_t)r * a.nkv + c) * GT + R) * D + 16 * x + 8 * hi);
        qf[x] = __builtin_bit_cast(ar_bf16x8, w);
    }
    constexpr float LOG2E = 1.44269504088896341f;
    const float c2 = a.scale * LOG2E;
    float m_run = -INFINITY, l_run = 0.f;
    ar_f32x16 acc[NDV];
#pragma unroll
    for (int y = 0; y < NDV; ++y)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[y][i] = 0.f;
    const bool wave_live = 128 * rt + 32 * wave < GT, wave_full = 128 * rt + 32 * wave + 31 < GT;

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
            const int e = tid + it * AB_THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) {
                const int x = tok[jj];
                const int64_t at = (int64_t)(x < 0 ? ~x : x) * D + 8 * u;
                kreg[it] = *(const ar_s16x8 *)((x < 0 ? CK : K) + at);
                vreg[it] = *(const ar_s16x8 *)((x < 0 ? CV : V) + at);
            }
        }
    };
    auto stash = [&](int kt, uint4 *Ks) {
        const int nk = n_keys - kt * KT < KT ? n_keys - kt * KT : KT;
#pragma unroll
        for (int it = 0; it < PF; ++it) {
            const int e = tid + it * AB_THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) {
                Ks[jj * KU + ar_key_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, kreg[it]);
                Ks[KT * KU + jj * KU + ar_value_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, vreg[it]);
            }
        }
    };
    look_up(t_lo);
    tokens_out(0);
    look_up(t_lo + 1);
    tokens_out(1);
    __syncthreads();
    if (t_lo < t_hi) {
        fetch(t_lo, tokS);
        stash(t_lo, buf0);
    }
    __syncthreads();
    for (int kt = t_lo, sel = 0; kt < t_hi; ++kt, sel ^= 1) {
        if (kt + 1 < t_hi) fetch(kt + 1, tokS + (sel ^ 1) * KT);
        look_up(kt + 2);
        const uint4 *Ks = buf0 + sel * BUF;
        const int j0 = kt * KT;
        if (wave_live) {
            ar_f32x16 sc[2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[hf][i] = 0.f;
#pragma unroll
            for (int x = 0; x < KU / 2; ++x)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    const int row = 32 * hf + l32;
                    sc[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ar_bf16x8, Ks[row * KU + ar_key_unit<KU>(row, 2 * x + hi)]), qf[x], sc[hf], 0, 0, 0);
                }
            const bool inside = wave_full && j0 + KT <= kv;         // committed keys only: every row sees them
            const int upto = ok ? last - j0 : -1;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float s = sc[hf][i] * c2;
                    sc[hf][i] = inside || 32 * hf + 8 * (i >> 2) + 4 * hi + (i & 3) <= upto ? s : -INFINITY;
                }
            float mx = sc[0][0];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int i = hf == 0 ? 1 : 0; i < 16; ++i) mx = fmaxf(mx, sc[hf][i]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run, mx), m_sub = m_new > -INFINITY ? m_new : 0.f;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_sub);
            float sum = 0.f;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int i = 0; i < 16; ++i) { sc[hf][i] = __builtin_amdgcn_exp2f(sc[hf][i] - m_sub); sum += sc[hf][i]; }
            l_run = l_run * alpha + sum;
            m_run = m_new;
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int y = 0; y < NDV; ++y)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[y][i] *= alpha;
            }
            const char *Vs = (const char *)(Ks + KT * KU);
            const int vk = 4 * hi + ((lane & 15) >> 2), vc8 = 8 * (lane & 1), vu = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);      // this lane's key, half unit and unit of a turned block
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
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
        if (kt + 1 < t_hi) stash(kt + 1, buf0 + (sel ^ 1) * BUF);
        tokens_out(sel);
        __syncthreads();
    }
    l_run += __shfl_xor(l_run, 32, 64);
    if (!ok) return;
    const float inv = l_run != 0.f ? 1.0f / l_run : 0.f;
    const int64_t width = (int64_t)a.nkv * a.G * D, row = ((int64_t)r * T + t) * width + (int64_t)(c * a.G + R / T) * D;
    const int64_t rows = (int64_t)a.R * T * a.nkv * a.G;            // a split's (token, head) rows
    if (S > 1 && hi == 0) {
        float *ml = a.scratch + S * rows * D + (split * rows + row / D) * 2;
        ml[0] = m_run;
        ml[1] = l_run;
    }
    if (S > 1 && l_run == 0.f) return;                             // an empty share is not read
#pragma unroll
    for (int y = 0; y < NDV; ++y)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = 32 * y + 8 * g + 4 * hi;                // registers 4g .. 4g + 3: four consecutive columns
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

template <int KU> static int ab_launch(const jl_block_args &a, hipStream_t st) {
    constexpr size_t lds = ab_lds_bytes(KU);
    auto kern = attn_block_kernel<KU>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_attn_block: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    const int row_tiles = (a.G * a.T + 127) / 128;
    kern<<<dim3((unsigned)(a.R * row_tiles * a.splits * a.nkv)), AB_THREADS, lds, st>>>(a, row_tiles);
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
    if ((int64_t)a.blocks * a.nkv * a.page_size > INT32_MAX || (int64_t)(a.cand_rows > 0 ? a.cand_rows : 0) * a.nkv * a.cand_max > INT32_MAX ||
        (int64_t)a.R * ((a.G * (int64_t)a.T + 127) / 128) * a.splits * a.nkv > INT32_MAX)
        return jl_fail(JL_E_INVALID, "jl_attn_block: more rows than 32 bits count");
    return a.D <= 64 ? ab_launch<8>(a, (hipStream_t)stream) : ab_launch<16>(a, (hipStream_t)stream);
}
