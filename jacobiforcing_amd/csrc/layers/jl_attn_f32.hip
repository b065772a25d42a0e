// jl_attn_f32.hip — the one-sweep attention of jl_attn_sweep.hip / jl_attn_rows.hip for float activations, on the float matrix instructions.
#include "jl_attn.h"

// Same decomposition as the 128-row form: a wavefront keeps its 32 (query, head) rows to itself, forms S^T = K Q^T of 32 keys at a time, so that a lane
// holds keys of ONE row, and hands the weights over as the B operand of O^T = V^T P^T straight from the accumulators.  v_mfma_f32_32x32x2_f32: lane l supplies
// row (A) or column (B) l % 32 at depth l / 32.  A lane's 16-byte unit is four depths of four instructions (both operands agree on the order); accumulator
// register r of S^T is key 8 (r / 4) + 4 (l / 32) + r % 4, so register r is the B operand of the r-th product with the values, whose A operand is the value column
// 32 t + l % 32 of that key.  Every product and sum is a 32-bit one, the exponentials are expf.
// Prompts: four wavefronts share the key and value tiles (two LDS buffers, the next tile leaves memory while this one is multiplied).  Few tiles with many keys
// (decoding, short portions): one wavefront per workgroup, the keys of a tile shared out over workgroups and joined by attn_sweep_join_kernel.
// What bounds it: the float matrix rate (a tile's 128 products of 64 cycles at widths of 128; everything else hides behind them).  Measured against the float
// multiply-adds from LDS before it (jl_attn.hip, where other sizes, biases and mixed heads still go), 8 heads of 128 over 2 key heads, causal:
//   prompts of 1021, 851 and 681 tokens     4371 -> 160 us          one prompt of 4096        30.1 -> 0.81 ms (43 TFLOP/s)
//   16 decoded tokens at a context of 1000  1441 -> 49 us           one at 4000               7.8 ms -> 50 us
constexpr int AF_KT = 32;

typedef float af_f32x16 __attribute__((ext_vector_type(16)));
template <int U> __device__ __forceinline__ int af_unit(int r, int u) { return U % 16 == 0 ? u ^ (r & 15) : u ^ ((r >> 1) & 7); }      // 16-byte unit u of key row r

constexpr size_t af_lds_bytes(int KU, int NDV, int NW) { return (NW > 1 ? 2 : 1) * (size_t)AF_KT * (KU + 8 * NDV) * 16 + 2 * AF_KT * 4; }

template <int KU, int NDV, int NW, int SRC>                                             // D <= 4 * KU, Dv <= 32 * NDV
__global__ __launch_bounds__(64 * NW) void attn_f32_kernel(jl_attn_args a, int HF, int TQ, int HB) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr bool V_IN_K = SRC == AR_V_IN_K, BUILT = SRC == AR_BUILT;
    constexpr int THREADS = 64 * NW, VU = 8 * NDV, BUF = AF_KT * (KU + VU), KPF = AF_KT * KU / THREADS, VPF = AF_KT * VU / THREADS;
    const int H = a.H, D = a.D, Dv = a.Dv, per_group = H / a.G;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    const int groups = a.G * HB, group = blockIdx.x % groups, tile_i = blockIdx.x / groups;
    const int *tile = a.tiles + 4 * (int64_t)tile_i;
    const int b = tile[0], i0 = tile[1], cnt = tile[2], row0 = tile[3];
    if (b < 0 || cnt <= 0) return;
    const int c = group / HB;
    const int h0 = c * per_group + (group - c * HB) * HF, h_end = (c + 1) * per_group;
    uint4 *buf0 = (uint4 *)smem;
    int *tokS = (int *)(buf0 + (NW > 1 ? 2 : 1) * BUF);             // [2][32] pool tokens of a tile's keys
    const int window = a.window > 0 ? a.window : 0x3fffffff, chunk = a.chunk, i_max = i0 + cnt - 1;
    const int lo = chunk > 0 ? i0 - i0 % chunk : (i0 - window + 1 > 0 ? i0 - window + 1 : 0);      // lowest key the tile's first row sees
    const int n_keys = i_max + 1 - lo;
    const int *bt = BUILT ? nullptr : a.block_tables + (int64_t)b * a.bt_stride;
    const int key_base = BUILT ? a.key_base[b] : 0, Dh = BUILT ? D - a.k_tail_cols : D;
    const float *kc = (const float *)a.k_cache + (int64_t)c * Dh, *kt = (const float *)a.k_tail, *vc = (const float *)a.v_cache + (int64_t)(c % a.Gv) * Dv;
    for (int e = tid; e < (NW > 1 ? 2 : 1) * BUF; e += THREADS) buf0[e] = make_uint4(0, 0, 0, 0);      // columns beyond D / Dv stay zero, rows beyond the last key finite

    const int R = 32 * wave + l32, ii = R / HF, hh = h0 + R % HF;
    const bool ok = R < TQ * HF && ii < cnt && hh < h_end;
    const int qi = i0 + ii, q_lo = chunk > 0 ? qi - qi % chunk : qi - window + 1;                 // the row's keys: q_lo .. qi
    float4 qf[KU / 2];
    {
        const float *qp = (const float *)a.q + (int64_t)(row0 + ii) * a.q_ld + hh * D + 4 * hi;
#pragma unroll
        for (int x = 0; x < KU / 2; ++x) {
            qf[x] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (ok && 8 * x + 4 * hi < D) qf[x] = *(const float4 *)(qp + 8 * x);
        }
    }
    float m_run = -INFINITY, l_run = 0.f;                           // each half-wavefront sums its own keys; the halves meet at the end
    if (a.sink && ok && blockIdx.z == 0) { m_run = a.sink[hh]; l_run = hi ? 0.f : 1.f; }
    af_f32x16 acc[NDV];
#pragma unroll
    for (int t = 0; t < NDV; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    const int wq_first = (32 * wave) / HF, wq_last = (32 * wave + 31) / HF < cnt - 1 ? (32 * wave + 31) / HF : cnt - 1;
    const int wlo_first = chunk > 0 ? (i0 + wq_first) - (i0 + wq_first) % chunk : i0 + wq_first - window + 1;       // lowest key of the wavefront's first query
    const bool wave_live = 32 * wave < TQ * HF && wq_first < cnt;

    int tok_next = 0;
    auto look_up = [&](int u0) {
        if (tid >= AF_KT || u0 + tid >= n_keys) return;
        const int j = lo + u0 + tid;
        if (BUILT) { tok_next = key_base + j; return; }
        const int pg = j / a.page_size;
        tok_next = bt[pg] * a.page_size + (j - pg * a.page_size);
    };
    auto tokens_out = [&](int sel) { if (tid < AF_KT) tokS[sel * AF_KT + tid] = tok_next; };
    auto k_ptr = [&](int tok, int u) -> const float * {
        return BUILT && 4 * u >= Dh ? kt + (int64_t)tok * a.k_tail_ld + (4 * u - Dh) : kc + (int64_t)tok * a.k_ld + 4 * u;
    };
    auto multiply = [&](const uint4 *Ks, int j0, int nk) {
        // wavefront-uniform: keys all behind its last query, or all before its first query's window
        if (!(wave_live && j0 <= i0 + wq_last && j0 + nk - 1 >= wlo_first)) return;
        af_f32x16 sc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.f;
#pragma unroll
        for (int x = 0; x < KU / 2; ++x) {
            const float4 k4 = __builtin_bit_cast(float4, Ks[l32 * KU + af_unit<KU>(l32, 2 * x + hi)]);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.x, qf[x].x, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.y, qf[x].y, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.z, qf[x].z, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.w, qf[x].w, sc, 0, 0, 0);
        }
        const int first = ok ? (q_lo - j0 > 0 ? q_lo - j0 : 0) : AF_KT, last = qi - j0 < nk - 1 ? qi - j0 : nk - 1;     // the row's keys within the tile
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int kk = 8 * (r >> 2) + 4 * hi + (r & 3);
            float s = sc[r] * a.scale;
            if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
            sc[r] = kk >= first && kk <= last ? s : -INFINITY;
            mx = fmaxf(mx, sc[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx), m_sub = m_new > -INFINITY ? m_new : 0.f;
        const float alpha = expf(m_run - m_sub);                    // m_run = -inf: 0, and nothing has been accumulated yet
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) { sc[r] = expf(sc[r] - m_sub); sum += sc[r]; }
        l_run = l_run * alpha + sum;
        m_run = m_new;
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int t = 0; t < NDV; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][r] *= alpha;
        }
        const float *Vf = (const float *)(V_IN_K ? Ks : Ks + AF_KT * KU);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = 8 * (r >> 2) + 4 * hi + (r & 3);
#pragma unroll
            for (int t = 0; t < NDV; ++t) {
                const int col = 32 * t + l32;
                const float v = V_IN_K ? Vf[4 * (key * KU + af_unit<KU>(key, col >> 2)) + (col & 3)] : Vf[key * 4 * VU + col];
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, sc[r], acc[t], 0, 0, 0);
            }
        }
    };
    const int S = a.splits > 1 ? a.splits : 1, split = blockIdx.z, per = ((n_keys + AF_KT - 1) / AF_KT + S - 1) / S;       // key tiles per share
    const int key_lo = split * per * AF_KT, key_hi = (split + 1) * per * AF_KT < n_keys ? (split + 1) * per * AF_KT : n_keys;
    look_up(key_lo);
    tokens_out(0);
    if (NW > 1) {
        look_up(key_lo + AF_KT);
        tokens_out(1);
        float4 kreg[KPF], vreg[VPF];
        auto fetch = [&](int u0, const int *tok) {
            const int nk = key_hi - u0 < AF_KT ? key_hi - u0 : AF_KT;
#pragma unroll
            for (int it = 0; it < KPF; ++it) {
                const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
                if (jj < nk && 4 * u < D) kreg[it] = *(const float4 *)k_ptr(tok[jj], u);
            }
            if (V_IN_K) return;
#pragma unroll
            for (int it = 0; it < VPF; ++it) {
                const int e = tid + it * THREADS, jj = e / VU, u = e % VU;
                if (jj < nk && 4 * u < Dv) vreg[it] = *(const float4 *)(vc + (int64_t)tok[jj] * a.v_ld + 4 * u);
            }
        };
        auto stash = [&](int u0, uint4 *Ks) {
            const int nk = key_hi - u0 < AF_KT ? key_hi - u0 : AF_KT;
#pragma unroll
            for (int it = 0; it < KPF; ++it) {
                const int e = tid + it * THREADS, jj = e / KU, u = e % KU;
                if (jj < nk && 4 * u < D) Ks[jj * KU + af_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, kreg[it]);
            }
            if (V_IN_K) return;
#pragma unroll
            for (int it = 0; it < VPF; ++it) {
                const int e = tid + it * THREADS, jj = e / VU, u = e % VU;
                if (jj < nk && 4 * u < Dv) Ks[AF_KT * KU + jj * VU + u] = __builtin_bit_cast(uint4, vreg[it]);
            }
        };
        __syncthreads();
        fetch(key_lo, tokS);
        stash(key_lo, buf0);
        __syncthreads();
        for (int u0 = key_lo, sel = 0; u0 < key_hi; u0 += AF_KT, sel ^= 1) {
            if (u0 + AF_KT < key_hi) fetch(u0 + AF_KT, tokS + (sel ^ 1) * AF_KT);
            look_up(u0 + 2 * AF_KT);
            multiply(buf0 + sel * BUF, lo + u0, key_hi - u0 < AF_KT ? key_hi - u0 : AF_KT);
            if (u0 + AF_KT < key_hi) stash(u0 + AF_KT, buf0 + (sel ^ 1) * BUF);
            tokens_out(sel);
            __syncthreads();
        }
    } else {
        __syncthreads();
        for (int u0 = key_lo, sel = 0; u0 < key_hi; u0 += AF_KT, sel ^= 1) {
            const int nk = key_hi - u0 < AF_KT ? key_hi - u0 : AF_KT, *tok = tokS + sel * AF_KT;
            look_up(u0 + AF_KT);
            constexpr int BATCH = 8;                                // rows on their way at once: the registers are the query's and the outputs'
#pragma unroll
            for (int part = 0; part < (V_IN_K ? 1 : 2); ++part) {
                const int U = part ? VU : KU, width = part ? Dv : D;
#pragma unroll
                for (int i0_ = 0; i0_ < (part ? VPF : KPF); i0_ += BATCH) {
                    float4 r[BATCH];
#pragma unroll
                    for (int i = 0; i < BATCH; ++i) {
                        const int e = tid + (i0_ + i) * THREADS, jj = e / U, u = e % U;
                        if (jj < nk && 4 * u < width) r[i] = part ? *(const float4 *)(vc + (int64_t)tok[jj] * a.v_ld + 4 * u) : *(const float4 *)k_ptr(tok[jj], u);
                    }
#pragma unroll
                    for (int i = 0; i < BATCH; ++i) {
                        const int e = tid + (i0_ + i) * THREADS, jj = e / U, u = e % U;
                        if (jj < nk && 4 * u < width) buf0[part ? AF_KT * KU + jj * VU + u : jj * KU + af_unit<KU>(jj, u)] = __builtin_bit_cast(uint4, r[i]);
                    }
                }
            }
            __syncthreads();
            multiply(buf0, lo + u0, nk);
            tokens_out(sel ^ 1);
            __syncthreads();
        }
    }
    l_run += __shfl_xor(l_run, 32, 64);
    if (S > 1) {                                                    // this share's rows: [Dv] unnormalised outputs, maximum, sum
        float *part = a.scratch + ((((int64_t)split * a.n_tiles + tile_i) * groups + group) * 32 + l32) * (int64_t)(Dv + 2);
        if (hi == 0) { part[Dv] = m_run; part[Dv + 1] = l_run; }
#pragma unroll
        for (int t = 0; t < NDV; ++t) {
            if (32 * t >= Dv) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) part[32 * t + 8 * (r >> 2) + 4 * hi + (r & 3)] = acc[t][r];
        }
        return;
    }
    if (!ok) return;
    const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
    const float *gate = (const float *)a.gate;
    float gh = a.out_scale;
    if (gate && a.gate_heads) gh *= 1.0f / (1.0f + expf(-gate[(int64_t)(row0 + ii) * a.gate_ld + hh]));
    const int64_t obase = (int64_t)(row0 + ii) * a.out_ld + hh * Dv;
#pragma unroll
    for (int t = 0; t < NDV; ++t) {
        if (32 * t >= Dv) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = 32 * t + 8 * g + 4 * hi;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                float v = acc[t][4 * g + x] * inv * gh;
                if (gate && !a.gate_heads) v *= 1.0f / (1.0f + expf(-gate[(int64_t)(row0 + ii) * a.gate_ld + hh * Dv + col + x]));
                ((float *)a.out)[obase + col + x] = v;
            }
        }
    }
}

bool jl_attn_f32_fits(int H, int G, int Gv, int D, int Dv, int64_t k_ld, int64_t v_ld, bool v_in_k) {
    if (!(H >= 1 && G >= 1 && H % G == 0 && Gv >= 1 && G % Gv == 0 && D >= 4 && D % 4 == 0 && D <= 256 && Dv >= 32 && Dv % 32 == 0 && Dv <= 128 && k_ld % 4 == 0 && v_ld % 4 == 0 &&
          k_ld >= (int64_t)G * D))
        return false;
    return v_in_k ? G == 1 && Dv <= D : v_ld >= (int64_t)Gv * Dv;
}

template <int KU, int NDV, int NW, int SRC> static int af_launch(const jl_attn_args &a, int hf, int hb, hipStream_t st) {
    constexpr size_t lds = af_lds_bytes(KU, NDV, NW);
    auto kern = attn_f32_kernel<KU, NDV, NW, SRC>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_attn_sweep: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    kern<<<dim3((unsigned)(a.n_tiles * a.G * hb), 1, (unsigned)(a.splits > 1 ? a.splits : 1)), 64 * NW, lds, st>>>(a, hf, a.TQ, hb);
    return jl_check_launch("attn_f32_kernel");
}

int jl_attn_f32_launch(const jl_attn_args &a, int hf, int hb, int src, bool wide, hipStream_t st) {
    if (!jl_attn_grid_fits(a, hb)) return jl_fail(JL_E_INVALID, "jl_attn_sweep: too many tiles");
    if (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)a.k_tail) & 15) return jl_fail(JL_E_INVALID, "jl_attn_sweep: float rows start at 16-byte borders");
    const int ku = a.D <= 64 ? 16 : a.D <= 128 ? 32 : a.D <= 192 ? 48 : 64, ndv = a.Dv <= 64 ? 2 : 4;
#define AF_CASE(K, V)                                                                               \
    if (ku == K && ndv == V) {                                                                      \
        if (src == AR_BUILT) return af_launch<K, V, 4, AR_BUILT>(a, hf, hb, st);                    \
        if (src == AR_PAGED) return wide ? af_launch<K, V, 4, AR_PAGED>(a, hf, hb, st) : af_launch<K, V, 1, AR_PAGED>(a, hf, hb, st);        \
        return wide ? af_launch<K, V, 4, AR_V_IN_K>(a, hf, hb, st) : af_launch<K, V, 1, AR_V_IN_K>(a, hf, hb, st);                           \
    }
    AF_CASE(16, 2) AF_CASE(16, 4) AF_CASE(32, 2) AF_CASE(32, 4) AF_CASE(48, 2) AF_CASE(48, 4) AF_CASE(64, 2) AF_CASE(64, 4)
#undef AF_CASE
    return jl_fail(JL_E_INVALID, "jl_attn_sweep: sizes");
}
