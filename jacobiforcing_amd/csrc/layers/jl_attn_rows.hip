// jl_attn_rows.hip — the one-sweep attention of jl_attn_sweep.hip for long portions: 128 (query, head) rows per workgroup.
#include "jl_attn.h"

constexpr int AR_THREADS = 256;

// ---- the same sweep for tiles of up to 128 rows: every wavefront keeps ITS 32 rows to itself ----------------------------------------
// Long portions (prefill) fill 128 (query, head) rows per workgroup; then no partial sums or weights have to meet in LDS.  Per tile of
// 64 (32 for wide keys) keys in LDS, shared by the four wavefronts, a wavefront forms the TRANSPOSED scores S^T = K Q^T (A = the key
// rows, one 16-byte read per lane and v_mfma_f32_32x32x16_bf16; B = its query fragments, in registers for the whole launch), so that a
// lane holds keys of ONE row (query l32; the other half of them in lane l32 + 32): maximum, sum and rescale factor are per-lane numbers
// plus one exchange with the other half-wavefront.  The order of the keys inside the 16 depths of the second product is free as long as
// both operands agree: accumulator registers 8s .. 8s + 7 of S^T (keys 16s + 4 (l / 32) + {0 .. 3, 8 .. 11}) are handed over as the B
// operand as they are, and the A operand V^T is read in the same order by ds_read_b64_tr_b16 (sixteen lanes turn four keys x sixteen
// columns), so weights never touch LDS and no value is packed by hand.  In O^T = V^T P^T a lane again holds one row's values: the rescale
// is one multiply per register, and four consecutive value columns of a row leave as one store.  A wavefront skips the key tiles none of
// its rows can see.
// LDS rows are whole multiples of 64 columns; their 16-byte units are permuted by the row (ar_key_unit, ar_value_unit) so that 8 .. 16 lanes
// of neighbouring rows meet different banks.  The next tile's rows travel from memory (16 bytes per lane) while this one is multiplied.
// What bounds it: issue of the softmax (about 30 cycles per key and lane against 32 of matrix work at widths of 128) at two workgroups per
// CU.  Measured, causal, bfloat16, against the form before it (32-key tiles, 8-deep products, values packed by hand from 2-byte reads):
//   4 x 2048 tokens, 16 heads of 128 over 4 key heads      582 -> 137 us (503 TFLOP/s)
//   1 x 8192 tokens, the same heads                        1728 -> 434 us (633 TFLOP/s)
//   4 x 2048 tokens, 16 heads of 192 / 128 apart           806 -> 180 us (479 TFLOP/s)
//   4 x 2048 tokens, 8 heads of 128 over 2, window 1024    180 -> 66 us
// Scores scaled in the exponent's multiply-add behind their maximum (queries take a negative scale's sign) instead of one by one: the first 129 -> 124, the second 393 -> 383; rows whose
// maximum is beyond 2^24, which would go wrong so, are multiplied one by one in the branch that scales the sums (ar_factor; the look at every tile instead: 2 to 5 %).

constexpr int ar_tile_keys(int KU) { return KU <= 16 ? 64 : 32; }
constexpr size_t ar_lds_bytes(int KU, int VU) { return 2 * (size_t)ar_tile_keys(KU) * (KU + VU) * 16 + 2 * ar_tile_keys(KU) * 4; }

template <int KU, int VU, int SRC>                                                      // D <= 8 * KU, Dv <= 8 * VU
__global__ __launch_bounds__(AR_THREADS, 2) void attn_rows_kernel(jl_attn_args a, int HF, int TQ, int HB) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr bool V_IN_K = SRC == AR_V_IN_K, BUILT = SRC == AR_BUILT;
    constexpr int KT = ar_tile_keys(KU), HALVES = KT / 32, NDV = VU / 4, VROWS = V_IN_K ? 0 : KT * VU;
    constexpr int KPF = KT * KU / AR_THREADS, VPF = KT * VU / AR_THREADS;
    const int H = a.H, D = a.D, Dv = a.Dv, per_group = H / a.G;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    // groups side by side: neighbouring workgroups go to different XCDs, so each keeps few groups' keys in its L2
    const int groups = a.G * HB, group = blockIdx.x % groups;
    const int *tile = a.tiles + 4 * (int64_t)(blockIdx.x / groups);
    const int b = tile[0], i0 = tile[1], cnt = tile[2], row0 = tile[3];
    if (b < 0 || cnt <= 0) return;
    const int c = group / HB;
    const int h0 = c * per_group + (group - c * HB) * HF, h_end = (c + 1) * per_group;
    constexpr int BUF = KT * KU + VROWS;                            // one buffer in 16-byte units: the keys, then the values (or none: the keys' own rows)
    uint4 *buf0 = (uint4 *)smem;
    int *tokS = (int *)(buf0 + 2 * (KT * KU + KT * VU));            // [2][KT] pool tokens of a tile's keys
    const int window = a.window > 0 ? a.window : 0x3fffffff;
    const int i_max = i0 + cnt - 1;
    const int chunk = a.chunk;
    const int lo = chunk > 0 ? i0 - i0 % chunk : (i0 - window + 1 > 0 ? i0 - window + 1 : 0);      // lowest key the tile's first row sees
    const int n_keys = i_max + 1 - lo;
    const int *bt = BUILT ? nullptr : a.block_tables + (int64_t)b * a.bt_stride;
    const int key_base = BUILT ? a.key_base[b] : 0;
    const int Dh = BUILT ? D - a.k_tail_cols : D;                   // columns of a key head that are its own
    const bf16_t *kc = (const bf16_t *)a.k_cache + (int64_t)c * Dh, *kt = (const bf16_t *)a.k_tail;
    const bf16_t *vc = (const bf16_t *)a.v_cache + (int64_t)(c % a.Gv) * Dv;
    const int page_shift = !BUILT && (a.page_size & (a.page_size - 1)) == 0 ? __builtin_ctz(a.page_size) : -1;
    for (int e = tid; e < 2 * BUF; e += AR_THREADS) buf0[e] = make_uint4(0, 0, 0, 0);      // columns beyond D / Dv and rows beyond the last key stay zero or finite
    __syncthreads();

    // this lane's row: (query R / HF, head h0 + R % HF), R = 32 * wave + l32; both half-wavefronts hold it
    const int R = 32 * wave + l32, ii = R / HF, hh = h0 + R % HF;
    const bool ok = R < TQ * HF && ii < cnt && hh < h_end;
    const int qi = i0 + ii, q_lo = chunk > 0 ? qi - qi % chunk : qi - window + 1;                 // the row's keys: q_lo .. qi
    const bool capped = a.softcap > 0.f;
    ar_bf16x8 qf[KU / 2];
    {
        const uint32_t sign = !capped && a.scale < 0.f ? 0x80008000u : 0u;      // scores are scaled behind their maximum: by a factor above zero
        const bf16_t *qp = (const bf16_t *)a.q + (int64_t)(row0 + ii) * a.q_ld + hh * D + 8 * hi;
#pragma unroll
        for (int x = 0; x < KU / 2; ++x) {
            uint2 w[2] = {make_uint2(0, 0), make_uint2(0, 0)};
            if (ok && 16 * x + 8 * hi < D) { w[0] = *(const uint2 *)(qp + 16 * x); w[1] = *(const uint2 *)(qp + 16 * x + 4); }
            qf[x] = __builtin_bit_cast(ar_bf16x8, make_uint4(w[0].x ^ sign, w[0].y ^ sign, w[1].x ^ sign, w[1].y ^ sign));
        }
    }
    // scores are kept times log2(e): weights are 2 ** (s - max)
    float m_run = -INFINITY, l_run = 0.f;
    if (a.sink && ok) { m_run = a.sink[hh] * AR_LOG2E; l_run = 1.f; }   // the sink: an extra score that attends to nothing
    if (m_run == INFINITY) m_run = NAN;                             // such a row is none: its first tile scales its sums by NaN
    float entry = ar_entry(m_run);
    if (hi) l_run = 0.f;                                            // each half-wavefront sums its own keys; the halves meet at the end
    const float c2 = capped ? AR_LOG2E : fabsf(a.scale * AR_LOG2E);
    ar_f32x16 acc[NDV];
#pragma unroll
    for (int t = 0; t < NDV; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    // the queries this wavefront's rows belong to (none: it only helps to load)
    const int wq_first = (32 * wave) / HF, wq_last = (32 * wave + 31) / HF < cnt - 1 ? (32 * wave + 31) / HF : cnt - 1;
    const int wlo_first = chunk > 0 ? (i0 + wq_first) - (i0 + wq_first) % chunk : i0 + wq_first - window + 1;       // lowest keys of the first and the last of them
    const int wlo_last = chunk > 0 ? (i0 + wq_last) - (i0 + wq_last) % chunk : i0 + wq_last - window + 1;
    const bool wave_live = 32 * wave < TQ * HF && wq_first < cnt;
    const bool wave_full = 32 * wave + 31 < TQ * HF && (32 * wave + 31) / HF < cnt && h0 + HF <= h_end;     // all 32 rows are rows of the tile

    // 16-byte loads where rows and columns start at 16-byte borders, else two of 8
    const bool wide = ((uintptr_t)a.k_cache & 15) == 0 && ((uintptr_t)a.v_cache & 15) == 0 && a.k_ld % 8 == 0 && a.v_ld % 8 == 0 &&
                      (!BUILT || (((uintptr_t)a.k_tail & 15) == 0 && a.k_tail_ld % 8 == 0));
    uint4 kreg[KPF], vreg[VPF];
    auto load16 = [&](const bf16_t *p) -> uint4 {
        if (wide) return *(const uint4 *)p;
        const uint2 x = *(const uint2 *)p, y = *(const uint2 *)(p + 4);
        return make_uint4(x.x, x.y, y.x, y.y);
    };
    // thread t < KT looks up the pool token of key t of a tile, two tiles ahead of the products
    int tok_next = 0;
    auto look_up = [&](int u0) {
        if (tid >= KT || u0 + tid >= n_keys) return;
        const int j = lo + u0 + tid;
        if (BUILT) { tok_next = key_base + j; return; }
        const int pg = page_shift >= 0 ? j >> page_shift : j / a.page_size;
        tok_next = bt[pg] * a.page_size + (j - pg * a.page_size);
    };
    auto tokens_out = [&](int sel) { if (tid < KT) tokS[sel * KT + tid] = tok_next; };
    auto fetch = [&](int u0, const int *tok) {
        const int nk = n_keys - u0 < KT ? n_keys - u0 : KT;
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * AR_THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D)
                kreg[it] = load16(BUILT && 8 * u >= Dh ? kt + (int64_t)tok[jj] * a.k_tail_ld + (8 * u - Dh) : kc + (int64_t)tok[jj] * a.k_ld + 8 * u);
        }
        if (V_IN_K) return;
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * AR_THREADS, jj = e / VU, u = e % VU;
            if (jj < nk && 8 * u < Dv) vreg[it] = load16(vc + (int64_t)tok[jj] * a.v_ld + 8 * u);
        }
    };
    auto stash = [&](int u0, uint4 *Ks) {
        const int nk = n_keys - u0 < KT ? n_keys - u0 : KT;
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * AR_THREADS, jj = e / KU, u = e % KU;
            if (jj < nk && 8 * u < D) Ks[jj * KU + ar_key_unit<KU>(jj, u)] = kreg[it];
        }
        if (V_IN_K) return;
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * AR_THREADS, jj = e / VU, u = e % VU;
            if (jj < nk && 8 * u < Dv) Ks[KT * KU + jj * VU + ar_value_unit<VU>(jj, u)] = vreg[it];
        }
    };
    // tile t is multiplied out of buffer t % 2 while tile t + 1 and the page numbers of tile t + 2 leave memory; both are written to LDS behind the
    // products: one barrier per tile (a buffer is written again only after the barrier that follows its last reader)
    look_up(0);
    tokens_out(0);
    look_up(KT);
    tokens_out(1);
    __syncthreads();
    fetch(0, tokS);
    stash(0, buf0);
    __syncthreads();
    for (int u0 = 0, tsel = 0; u0 < n_keys; u0 += KT, tsel ^= 1) {
        const int nk = n_keys - u0 < KT ? n_keys - u0 : KT;
        if (u0 + KT < n_keys) fetch(u0 + KT, tokS + (tsel ^ 1) * KT);
        look_up(u0 + 2 * KT);
        const uint4 *Ks = buf0 + tsel * BUF;
        const int j0 = lo + u0;                                     // position of the tile's first key
        // wavefront-uniform: keys all behind its last query, or all before its first query's window
        if (wave_live && j0 <= i0 + wq_last && j0 + nk - 1 >= wlo_first) {
            ar_f32x16 sc[HALVES];
#pragma unroll
            for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[hf][r] = 0.f;
#pragma unroll
            for (int x = 0; x < KU / 2; ++x)
#pragma unroll
                for (int hf = 0; hf < HALVES; ++hf) {
                    const int row = 32 * hf + l32;
                    const ar_bf16x8 ka = __builtin_bit_cast(ar_bf16x8, Ks[row * KU + ar_key_unit<KU>(row, 2 * x + hi)]);
                    sc[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka, qf[x], sc[hf], 0, 0, 0);
                }
            if (capped) {
                float big = 0.f;
#pragma unroll
                for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                    for (int r = 0; r < 16; ++r) { sc[hf][r] *= a.scale; big = fmaxf(big, fabsf(sc[hf][r])); }
                if (__any(big > 0.25f * a.softcap)) {               // wavefront-uniform: most tiles' scores are far below the cap
#pragma unroll
                    for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                        for (int r = 0; r < 16; ++r) sc[hf][r] = soft_cap_fast(sc[hf][r], a.softcap);
                } else {
                    const float inv_cap = 1.0f / a.softcap;
#pragma unroll
                    for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                        for (int r = 0; r < 16; ++r) sc[hf][r] = soft_cap_small(sc[hf][r], inv_cap);
                }
            }
            // wavefront-uniform: a full tile whose keys every row of the wavefront sees needs no mask
            const bool inside = nk == KT && wave_full && j0 + KT - 1 <= i0 + wq_first && j0 >= wlo_last;
            if (!inside) {
                const int first = ok ? (q_lo - j0 > 0 ? q_lo - j0 : 0) : KT, last = qi - j0 < nk - 1 ? qi - j0 : nk - 1;     // the row's keys within the tile
#pragma unroll
                for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int kk = 32 * hf + 8 * (r >> 2) + 4 * hi + (r & 3);
                        sc[hf][r] = kk >= first && kk <= last ? sc[hf][r] : -INFINITY;
                    }
            }
            float mx = sc[0][0];
#pragma unroll
            for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                for (int r = hf == 0 ? 1 : 0; r < 16; ++r) mx = fmaxf(mx, sc[hf][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run, mx * c2);
            float factor = c2;
            if (__any(!(m_new <= entry))) {                         // after the first tiles a row's maximum seldom moves (a stale one would leave the greatest weight inexact)
                const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new > -INFINITY ? m_new : 0.f));      // m_run = -inf: 0, and nothing has been accumulated yet
                m_run = m_new;
                entry = ar_entry(m_run);
                factor = ar_factor(sc, c2, m_run);
                l_run *= alpha;
#pragma unroll
                for (int t = 0; t < NDV; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[t][r] *= alpha;
            }
            const float m_sub = m_run > -INFINITY ? m_run : 0.f;   // a row that has seen no key yet: all weights are 2 ** -inf
            float sum = 0.f;
#pragma unroll
            for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                for (int r = 0; r < 16; ++r) { sc[hf][r] = __builtin_amdgcn_exp2f(fmaf(sc[hf][r], factor, -m_sub)); sum += sc[hf][r]; }
            l_run += sum;
            const char *Vs = (const char *)(V_IN_K ? Ks : Ks + KT * KU);
            const int vk = 4 * hi + ((lane & 15) >> 2), vc8 = 8 * (lane & 1), vu = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);      // this lane's key, half unit and unit of a turned block
#pragma unroll
            for (int hf = 0; hf < HALVES; ++hf)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    ar_f32x8 pf;
#pragma unroll
                    for (int x = 0; x < 8; ++x) pf[x] = sc[hf][8 * s + x];
                    const ar_bf16x8 pb = __builtin_convertvector(pf, ar_bf16x8);
#pragma unroll
                    for (int t = 0; t < NDV; ++t) {
                        ar_s16x4 half[2];
#pragma unroll
                        for (int y = 0; y < 2; ++y) {
                            const int key = 32 * hf + 16 * s + 8 * y + vk, u = 4 * t + vu;
                            const int at = V_IN_K ? key * KU + ar_key_unit<KU>(key, u) : key * VU + ar_value_unit<VU>(key, u);
                            half[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ar_lds_s16x4 *)(Vs + 16 * at + vc8));
                        }
                        const ar_s16x8 va = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ar_bf16x8, va), pb, acc[t], 0, 0, 0);
                    }
                }
        }
        if (u0 + KT < n_keys) stash(u0 + KT, buf0 + (tsel ^ 1) * BUF);
        tokens_out(tsel);
        __syncthreads();
    }
    l_run += __shfl_xor(l_run, 32, 64);
    if (!ok) return;
    const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
    const bf16_t *gate = (const bf16_t *)a.gate;
    float gh = 1.0f;
    if (gate && a.gate_heads) gh = 1.0f / (1.0f + __expf(-ld_f(gate + (int64_t)(row0 + ii) * a.gate_ld + hh)));
    const int64_t obase = (int64_t)(row0 + ii) * a.out_ld + hh * Dv;
    gh *= a.out_scale;
#pragma unroll
    for (int t = 0; t < NDV; ++t) {
        if (32 * t >= Dv) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = 32 * t + 8 * g + 4 * hi;                // registers 4g .. 4g + 3: four consecutive value columns
            float v[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                v[x] = acc[t][4 * g + x] * inv * gh;
                if (gate && !a.gate_heads) v[x] *= 1.0f / (1.0f + __expf(-ld_f(gate + (int64_t)(row0 + ii) * a.gate_ld + hh * Dv + col + x)));
            }
            if (a.out_dtype == JL_OUT_F32) st4_f((float *)a.out + obase + col, v);
            else st4_f((bf16_t *)a.out + obase + col, v);
        }
    }
}

template <int KU, int VU, int SRC> static int ar_launch(const jl_attn_args &args, int hf, int hb, hipStream_t st) {
    jl_attn_args a = args;
    if (!(a.softcap > 0.f) && ar_one_by_one(a.scale)) a.softcap = INFINITY;      // a cap's scores are multiplied one by one, and come out of an infinite one as they are
    constexpr size_t lds = ar_lds_bytes(KU, VU);
    auto kern = attn_rows_kernel<KU, VU, SRC>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_attn_sweep: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    kern<<<dim3((unsigned)(a.n_tiles * a.G * hb)), AR_THREADS, lds, st>>>(a, hf, a.TQ, hb);
    return jl_check_launch("attn_rows_kernel");
}
template <int KU, int VU> static int ar_launch_v(const jl_attn_args &a, int hf, int hb, bool v_in_k, hipStream_t st) {
    return v_in_k ? ar_launch<KU, VU, AR_V_IN_K>(a, hf, hb, st) : ar_launch<KU, VU, AR_PAGED>(a, hf, hb, st);
}

int jl_attn_rows_launch(const jl_attn_args &args, int hf, int hb, bool v_in_k, hipStream_t st) {
    jl_attn_args a = args;
    a.q_ld = (int64_t)a.H * a.D;
    if (!jl_attn_grid_fits(a, hb)) return jl_fail(JL_E_INVALID, "jl_attn_sweep: too many tiles");
    const int ku = 8 * ((a.D + 63) / 64), vu = a.Dv <= 64 ? 8 : 16;      // 16-byte units of a row in LDS
#define AR_CASE(K, V) if (ku == K && vu == V) return ar_launch_v<K, V>(a, hf, hb, v_in_k, st)
    AR_CASE(8, 8); AR_CASE(8, 16);
    AR_CASE(16, 8); AR_CASE(16, 16);
    AR_CASE(24, 8); AR_CASE(24, 16);
    AR_CASE(32, 8); AR_CASE(32, 16);
#undef AR_CASE
    return jl_fail(JL_E_INVALID, "jl_attn_sweep: 128-row tiles take key widths up to 256, value widths up to 128");
}

extern "C" int jl_attn_expanded_tile_rows(void) { return AR_ROWS; }

extern "C" int jl_attn_expanded(const jl_attn_args *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_attn_expanded: null arguments");
    const jl_attn_args &a = *ap;
    if (a.n_tiles <= 0) return JL_OK;
    if (!a.q || !a.k_cache || !a.v_cache || !a.out || !a.tiles || !a.key_base || (a.k_tail_cols > 0 && !a.k_tail)) return jl_fail(JL_E_INVALID, "jl_attn_expanded: null pointer");
    const int64_t own = a.D - a.k_tail_cols;
    if ((a.dtype != JL_BF16 && a.dtype != JL_F32) || a.H <= 0 || a.G != a.H || (a.Gv > 0 && a.Gv != a.H) || a.D <= 0 || a.D % 8 || a.D > 256 || a.k_tail_cols < 0 || a.k_tail_cols % 8 || own < 0 ||
        a.Dv < 32 || a.Dv % 32 || a.Dv > 128 || a.TQ != AR_ROWS || !jl_attn_grid_fits(a, 1))
        return jl_fail(JL_E_INVALID, "jl_attn_expanded: a key and a value head per query head, key widths in multiples of 8 up to 256, value widths in multiples of 32 up to 128");
    if (a.k_ld < a.H * own || a.v_ld < (int64_t)a.H * a.Dv || a.q_ld < (int64_t)a.H * a.D || a.out_ld < (int64_t)a.H * a.Dv || (a.k_tail_cols > 0 && a.k_tail_ld < a.k_tail_cols) ||
        a.k_ld % 4 || a.v_ld % 4 || a.q_ld % 4 || a.out_ld % 4 || a.k_tail_ld % 4)
        return jl_fail(JL_E_INVALID, "jl_attn_expanded: row strides hold a row and are multiples of four");
    if (a.out_dtype != JL_OUT_SAME && a.out_dtype != JL_OUT_F32) return jl_fail(JL_E_INVALID, "jl_attn_expanded: unknown out_dtype");
    if (a.chunk > 0 && a.window > 0) return jl_fail(JL_E_INVALID, "jl_attn_expanded: chunks exclude a window");
    hipStream_t st = (hipStream_t)stream;
    if (a.dtype == JL_F32) return jl_attn_f32_launch(a, 1, 1, AR_BUILT, true, st);
    const int ku = 8 * ((a.D + 63) / 64), vu = a.Dv <= 64 ? 8 : 16;
#define AR_CASE(K, V) if (ku == K && vu == V) return ar_launch<K, V, AR_BUILT>(a, 1, 1, st)
    AR_CASE(8, 8); AR_CASE(8, 16);
    AR_CASE(16, 8); AR_CASE(16, 16);
    AR_CASE(24, 8); AR_CASE(24, 16);
    AR_CASE(32, 8); AR_CASE(32, 16);
#undef AR_CASE
    return jl_fail(JL_E_INVALID, "jl_attn_expanded: sizes");
}
