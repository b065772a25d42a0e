// jl_retention.hip — retention: linear attention with a fixed decay per head and a float state per (request slot, head),
// scanned token by token for prompt portions and decoded tokens alike.
#include "jl_common.h"
#include <type_traits>

// One workgroup per (request, head); thread (p, j) owns rows DPER p .. of column j of the state S [D, Dv] in registers, PARTS threads per column.  Tokens are taken TT at a
// time: the rotated queries / keys of a group go through LDS, each thread runs the recurrence for its rows, the parts' sums meet in LDS, and part p finishes every PARTS-th token (unit norm over the
// head's Dv outputs).  What bounds single tokens is the state's way in and out, so as many loads as fit are on the way: one thread per column took 34.7 us for 32 tokens of 8 heads of 128 x 128 (33.6 MB),
// four take 12.7; a step of 32 decoding requests 516 -> 503 us, which then waits for the host.
constexpr int RET_TT = 8;

// MAXT: the largest workgroup the instantiation is launched with (1 024 threads leave 128 registers per lane: one thread per column keeps up to 64 rows in them).
// WHOLE: D is DMAX.  Else rows beyond D, zeros times a v that may not be finite, stay out of the sums: a branch per RB rows (fewer rows where a part has few; 32 tokens of 8 heads of 96: 9.8 -> 8.5 us, with its
// bound of registers; 300 of 4 heads of 192 in chunks 276 -> 393).
template <typename T, int DMAX, int PARTS, int MAXT, bool WHOLE>
__global__ __launch_bounds__(MAXT, !WHOLE && PARTS == 4 && DMAX <= 128 ? 4 : 1) void retention_kernel(const T *__restrict__ proj, int64_t ld, int q_col, int k_col, int v_col, int g_col,
                                 const int32_t *__restrict__ seq, int H, int D, int Dv, int rot_dims,
                                 const float *__restrict__ cos_t, const float *__restrict__ sin_t, int64_t table_len,
                                 const float *__restrict__ decay, float eps, float *__restrict__ state, T *__restrict__ out, int mode) {
    constexpr int DPER = DMAX / PARTS, RB = WHOLE || PARTS == 4 ? 4 : 16;
    extern __shared__ float lds[];
    float *qs = lds;                                   // [TT][DMAX]
    float *ks = qs + RET_TT * DMAX;                    // [TT][DMAX]
    float *red = ks + RET_TT * DMAX;                   // [TT][16]
    float *sums = red + RET_TT * 16;                   // [TT][threads]: the parts' sums
    const int b = blockIdx.x / H, h = blockIdx.x - b * H;
    const int row0 = seq[4 * b], cnt = seq[4 * b + 1], pos0 = seq[4 * b + 2], slot = seq[4 * b + 3];
    if (cnt <= 0) return;
    const int tid = threadIdx.x, width = blockDim.x / PARTS, part = PARTS > 1 ? tid / width : 0, j = PARTS > 1 ? tid - part * width : tid, wave = j >> 6, nw = width >> 6, d0 = part * DPER;
    const bool live = j < Dv;
    const int mine = __builtin_amdgcn_readfirstlane(D - d0);       // rows of this part that exist (the same for a wavefront)
    const float gamma = decay[h], kscale = 1.0f / sqrtf((float)D);
    const int half = rot_dims >> 1;
    float *sp = state + ((int64_t)slot * H + h) * D * Dv;
    float S[DPER];
    const bool old = live && (mode == JL_RET_FROM_SLOT || (mode == JL_RET_SCAN && pos0 > 0));
#pragma unroll
    for (int i = 0; i < DPER; ++i) S[i] = old && d0 + i < D ? sp[(int64_t)(d0 + i) * Dv + j] : 0.f;

    for (int t0 = 0; t0 < cnt; t0 += RET_TT) {
        const int nt = cnt - t0 < RET_TT ? cnt - t0 : RET_TT;
        __syncthreads();
        for (int e = tid; e < nt * DMAX; e += blockDim.x) {
            const int tt = e / DMAX, d = e - tt * DMAX;
            if (d >= D) { qs[e] = ks[e] = 0.f; continue; }      // rows beyond D stay zero
            const T *row = proj + (int64_t)(row0 + t0 + tt) * ld + h * D;
            float qv, kv;
            if (d < rot_dims) {
                const int i = d < half ? d : d - half;
                int64_t p = pos0 + t0 + tt;
                if (p >= table_len) p = table_len - 1;
                const float c = cos_t[p * half + i], s = sin_t[p * half + i];
                const float qu = ld_f(row + q_col + i), qw = ld_f(row + q_col + i + half);
                const float ku = ld_f(row + k_col + i), kw = ld_f(row + k_col + i + half);
                qv = d < half ? qu * c - qw * s : qw * c + qu * s;
                kv = d < half ? ku * c - kw * s : kw * c + ku * s;
            } else {
                qv = ld_f(row + q_col + d);
                kv = ld_f(row + k_col + d);
            }
            qs[e] = qv;
            ks[e] = kv * kscale;
        }
        __syncthreads();
        float o[RET_TT];
#pragma unroll
        for (int tt = 0; tt < RET_TT; ++tt) {
            o[tt] = 0.f;
            if (tt < nt) {
                const float v = live ? ld_f(proj + (int64_t)(row0 + t0 + tt) * ld + v_col + h * Dv + j) : 0.f;
                const float *qp = qs + tt * DMAX + d0, *kp = ks + tt * DMAX + d0;
                float acc = 0.f;
#pragma unroll
                for (int i0 = 0; i0 < DPER; i0 += RB) {
                    float4 q4[RB / 4];
#pragma unroll
                    for (int y = 0; y < RB / 4; ++y) {
                        const int i = i0 + 4 * y;
                        const float4 k4 = *(const float4 *)(kp + i);
                        q4[y] = *(const float4 *)(qp + i);
                        S[i] = gamma * S[i] + k4.x * v;
                        S[i + 1] = gamma * S[i + 1] + k4.y * v;
                        S[i + 2] = gamma * S[i + 2] + k4.z * v;
                        S[i + 3] = gamma * S[i + 3] + k4.w * v;
                    }
                    if (WHOLE || i0 + RB <= mine)
#pragma unroll
                        for (int y = 0; y < RB / 4; ++y) {
                            const int i = i0 + 4 * y;
                            acc += S[i] * q4[y].x;
                            acc += S[i + 1] * q4[y].y;
                            acc += S[i + 2] * q4[y].z;
                            acc += S[i + 3] * q4[y].w;
                        }
                    else
#pragma unroll
                        for (int i = 0; i < RB; ++i)
                            if (i0 + i < mine) acc += S[i0 + i] * qp[i0 + i];
                }
                o[tt] = acc;
                if (PARTS > 1 && mode != JL_RET_LOCAL_STATE) sums[tt * blockDim.x + tid] = acc;
            }
        }
        if (mode == JL_RET_LOCAL_STATE) continue;
        if (PARTS > 1) __syncthreads();
#pragma unroll
        for (int y = 0; y < RET_TT / PARTS; ++y) {                  // this part's tokens: part, part + PARTS, ..
            const int tt = y * PARTS + part;
            if (tt >= nt) continue;
            if (PARTS > 1) {
                float acc = sums[tt * blockDim.x + j];
#pragma unroll
                for (int p = 1; p < PARTS; ++p) acc += sums[tt * blockDim.x + p * width + j];
                o[y] = acc;
            }
            const float ss = wave_sum_f32(o[y] * o[y]);
            if ((j & 63) == 0) red[tt * 16 + wave] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int y = 0; y < RET_TT / PARTS; ++y) {
            const int tt = y * PARTS + part;
            if (tt >= nt || !live) continue;
            float ss = 0.f;
            for (int w = 0; w < nw; ++w) ss += red[tt * 16 + w];
            const float r = 1.0f / sqrtf(ss / (float)Dv + eps);
            const int64_t n = row0 + t0 + tt;
            const float g = ld_f(proj + n * ld + g_col + h * Dv + j);
            st_f(out + n * ((int64_t)H * Dv) + h * Dv + j, o[y] * r * (g / (1.0f + expf(-g))));
        }
    }
    if (live && mode != JL_RET_FROM_SLOT)
#pragma unroll
        for (int i = 0; i < DPER; ++i)
            if (d0 + i < D) sp[(int64_t)(d0 + i) * Dv + j] = S[i];
}

template <typename T, int DMAX>
static int ret_launch(const void *proj, int64_t ld, int q_col, int k_col, int v_col, int g_col, const int32_t *seq, int B, int H, int D,
                      int Dv, int rot_dims, const float *cos_t, const float *sin_t, int64_t table_len, const float *decay, float eps,
                      float *state, void *out, int mode, hipStream_t st) {
    const int width = (Dv + 63) / 64 * 64, parts = width <= 128 ? 4 : width <= 256 ? 2 : 1;
    const size_t lds = (size_t)(2 * RET_TT * DMAX + RET_TT * 16 + (parts > 1 ? RET_TT * width * parts : 0)) * 4;
#define RET_LAUNCH(PARTS, MAXT)                                                                                                                          \
    (D == DMAX ? retention_kernel<T, DMAX, PARTS, MAXT, true> : retention_kernel<T, DMAX, PARTS, MAXT, false>)<<<dim3((unsigned)(B * H)), width * PARTS, lds, st>>>((const T *)proj, ld, q_col, k_col, v_col, g_col, seq, H, D, Dv, \
                                                                                               rot_dims, cos_t, sin_t, table_len, decay, eps, state, (T *)out, mode)
    if (parts == 4) RET_LAUNCH(4, 512);
    else if (parts == 2) RET_LAUNCH(2, 512);
    else RET_LAUNCH(1, 1024);
#undef RET_LAUNCH
    return jl_check_launch("retention_kernel");
}

extern "C" int jl_retention(const void *proj, int dtype, int64_t ld, int32_t q_col, int32_t k_col, int32_t v_col, int32_t g_col,
                            const int32_t *seq, int32_t B, int32_t H, int32_t D, int32_t Dv, int32_t rot_dims, const float *cos_t,
                            const float *sin_t, int64_t table_len, const float *decay, float eps, float *state, void *out,
                            int32_t mode, void *stream) {
    if (B <= 0) return JL_OK;
    if (!proj || !seq || !decay || !state || (!out && mode != JL_RET_LOCAL_STATE)) return jl_fail(JL_E_INVALID, "jl_retention: null pointer");
    if (mode < JL_RET_SCAN || mode > JL_RET_FROM_SLOT) return jl_fail(JL_E_INVALID, "jl_retention: unknown mode %d", mode);
    if (H <= 0 || D <= 0 || D > 256 || Dv <= 0 || Dv > 1024) return jl_fail(JL_E_INVALID, "jl_retention: D must be <= 256 and Dv <= 1024");
    if (rot_dims < 0 || rot_dims > D || rot_dims % 2 || (rot_dims && (!cos_t || !sin_t || table_len <= 0)))
        return jl_fail(JL_E_INVALID, "jl_retention: rot_dims must be even and <= D, with tables");
    hipStream_t st = (hipStream_t)stream;
#define RET_CASE(N) JL_DISPATCH(dtype, return (ret_launch<T, N>(proj, ld, q_col, k_col, v_col, g_col, seq, B, H, D, Dv, rot_dims, cos_t, \
                                                                 sin_t, table_len, decay, eps, state, out, mode, st)))
    if (D <= 32) RET_CASE(32);
    else if (D <= 64) RET_CASE(64);
    else if (D <= 128) RET_CASE(128);
    else RET_CASE(256);
#undef RET_CASE
    return JL_OK;
}

// Joins the chunks of long portions.  Per (request, head): S = the request's state (zero when it starts at position 0); for each of
// its chunks in order: the chunk's local state in `scratch` is replaced by S (the state the chunk starts from), then
// S = decay^len S + local.  The final S is the request's new state.  req [B, 4] = {first chunk, chunks, pos0, slot},
// chunk_len [chunks] int32.
__global__ __launch_bounds__(256) void retention_join_kernel(const int32_t *__restrict__ req, const int32_t *__restrict__ chunk_len, int H,
                                                              int64_t DDv, const float *__restrict__ decay, float *__restrict__ state,
                                                              float *__restrict__ scratch) {
    const int b = blockIdx.x / H, h = blockIdx.x - b * H;
    const int c0 = req[4 * b], nc = req[4 * b + 1], pos0 = req[4 * b + 2], slot = req[4 * b + 3];
    const float gamma = decay[h];
    float *sp = state + ((int64_t)slot * H + h) * DDv;
    for (int64_t e = (int64_t)blockIdx.y * 256 + threadIdx.x; e < DDv; e += (int64_t)gridDim.y * 256) {
        float S = pos0 > 0 ? sp[e] : 0.f;
        for (int c = c0; c < c0 + nc; ++c) {
            float *lp = scratch + ((int64_t)c * H + h) * DDv + e;
            const float local = *lp;
            *lp = S;
            float gp = 1.f;
            for (int t = 0; t < chunk_len[c]; ++t) gp *= gamma;
            S = gp * S + local;
        }
        sp[e] = S;
    }
}

extern "C" int jl_retention_join(const int32_t *req, int32_t B, const int32_t *chunk_len, int32_t H, int32_t D, int32_t Dv,
                                 const float *decay, float *state, float *scratch, void *stream) {
    if (B <= 0) return JL_OK;
    if (!req || !chunk_len || !decay || !state || !scratch || H <= 0 || D <= 0 || Dv <= 0) return jl_fail(JL_E_INVALID, "jl_retention_join: null pointer or bad sizes");
    const int64_t ddv = (int64_t)D * Dv;
    const unsigned gy = (unsigned)((ddv + 255) / 256 < 64 ? (ddv + 255) / 256 : 64);
    retention_join_kernel<<<dim3((unsigned)(B * H), gy), 256, 0, (hipStream_t)stream>>>(req, chunk_len, H, ddv, decay, state, scratch);
    return jl_check_launch("retention_join_kernel");
}

// ---- long portions on the float matrix instructions: pieces side by side, 64 tokens at a time -------------------------------------------------
// With g = the head's decay, a group of n tokens is three products on the state S the group starts from:
//   o_i = g^(i+1) S^T q_i + sum_{j <= i} g^(i-j) (q_i . k_j) v_j,          S <- g^n S + sum_j g^(n-1-j) k_j v_j^T.
// A portion is cut into pieces (whole groups, except the last) that run side by side: every piece's own contribution to the state (RM_LOCAL, not for a
// request's last piece), the state every piece starts from (retention_pieces_join_kernel), outputs (RM_OUT; the last piece leaves the final state in its slot).
// A workgroup owns one head of one piece; wavefront w holds columns 32 w .. + 31 of S [D, Dv] in accumulators.  v_mfma_f32_32x32x2_f32: lane l supplies
// row (A) or column (B) l % 32 at depth l / 32, accumulator r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 — so the state's accumulators are the B operand of
// S^T q as they are (register r against the query's element of the same row), and never cross LDS.  Everything is a 32-bit number from the projection on, as in
// the scan: no operand is split or rounded.  q, k (rotated, scaled), v and the pairs' weights of the group lie in LDS as floats; the next group's rows
// are on their way meanwhile.
// What bounds it: 368 matrix instructions of 64 cycles per wavefront and group of 64 tokens at 128 x 128, and the phases of a group at one workgroup per CU.
// Values that are not finite reach the tokens from their own on and the state, as in the scan, though products run over whole groups (a second pass over a group that holds one).
// Outputs leave as floats and are normed and gated by rows in a launch of their own: in this one, a wavefront's sums over its 32 columns cost 160 exchanges per group and the gates
// came two bytes at a time, four on their way (outputs 211 us then, 119 and 18 now).
// Measured at 8 heads of 128 x 128, bfloat16, against the scan (chunks of 64 tokens side by side): 4 x 2048 tokens 1157 -> 182 us, one prompt of 128
// 985 -> 53, 8 x 8 tokens 84 -> 34; float, 1021 + 851 + 681 tokens: 1091 -> 105.
constexpr int RM_T = 64, RM_OUT = 0, RM_LOCAL = 1;
typedef float rm_f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ rm_f32x16 rm_mma(float a, float b, rm_f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
static constexpr size_t rm_lds_bytes(int DP, bool out) { return ((size_t)RM_T * DP * (out ? 2 : 1) + RM_T * 128 + (out ? RM_T * RM_T : 0) + 2 * RM_T) * 4; }

template <typename T, int DP, int MODE>
__global__ __launch_bounds__(256, 1) void retention_pieces_kernel(jl_retention_pieces a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr bool OUT = MODE == RM_OUT;
    constexpr int U = DP / 4, KPF = RM_T * U / 256, VPF = RM_T * 32 / 256, NS = DP / 32;
    const int piece = blockIdx.x, h = blockIdx.y, H = a.H, D = a.D, Dv = a.Dv;
    const int row0 = a.piece_rec[4 * piece], cnt = a.piece_rec[4 * piece + 1], slot = a.piece_rec[4 * piece + 2], last = a.piece_rec[4 * piece + 3];
    if (cnt <= 0 || (!OUT && last)) return;
    float4 *Ks = (float4 *)smem, *Qs = Ks + RM_T * U;               // [64][D], 16-byte units permuted by the row
    float *Vs = (float *)(OUT ? Qs + RM_T * U : Qs);                // [64][128]
    float4 *Ps = (float4 *)(Vs + RM_T * 128);                       // [64][64] decayed q . k of the pairs, permuted likewise
    float *gp = (float *)Ps + (OUT ? RM_T * RM_T : 0);              // g^0 .. g^64
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5, nw = (Dv + 31) / 32, col = 32 * wave + l32;
    const float gamma = a.decay[h], kscale = 1.0f / sqrtf((float)D);
    if (wave == 0) {                                                // powers by doubling, which doubles a rounding error too: in 64 bits.  Lane l holds g^(l+1)
        double p = gamma;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double y = __shfl_up(p, off, 64);
            if (lane >= off) p *= y;
        }
        gp[lane + 1] = (float)p;
        if (lane == 0) gp[0] = 1.0f;
    }
    auto at = [](int row, int u) { return u ^ (row & 15); };        // U is a multiple of 16
    const T *src = (const T *)a.proj + (int64_t)row0 * a.ld;
    const int half = a.rot_dims >> 1, hu = half / 4;

    rm_f32x16 S[NS];
    float *sp = a.scratch + ((int64_t)piece * H + h) * D * Dv;
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int d = 32 * t + 8 * (r >> 2) + 4 * hi + (r & 3);
            S[t][r] = (OUT && d < D && col < Dv) ? sp[(int64_t)d * Dv + col] : 0.f;
        }
    // a group's rows on their way: four elements of a row per unit
    typedef typename std::conditional<sizeof(T) == 2, uint2, float4>::type unit_t;
    unit_t rq[KPF], rk[KPF], rv[VPF];
    auto to_float = [](const unit_t &w) -> float4 {
        float v[4];
        ld4_f((const T *)&w, v);
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    auto fetch = [&](int t0) {
        const int nt = cnt - t0;
        const T *base = src + (int64_t)t0 * a.ld;
        const unit_t zero = {};
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * 256, tt = e / U, u = e % U;
            rk[it] = rq[it] = zero;
            if (tt < nt && 4 * u < D) {
                const T *row = base + (int64_t)tt * a.ld + h * D + 4 * u;
                rk[it] = *(const unit_t *)(row + a.k_col);
                if (OUT) rq[it] = *(const unit_t *)(row + a.q_col);
            }
        }
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * 256, tt = e >> 5, u = e & 31;
            rv[it] = zero;
            if (tt < nt && 4 * u < Dv) rv[it] = *(const unit_t *)(base + (int64_t)tt * a.ld + a.v_col + h * Dv + 4 * u);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < cnt; t0 += RM_T) {
        const int nt = cnt - t0 < RM_T ? cnt - t0 : RM_T;
        __syncthreads();                                            // the group before has been read
#pragma unroll
        for (int it = 0; it < KPF; ++it) {
            const int e = tid + it * 256, tt = e / U, u = e % U;
            const float4 k = to_float(rk[it]);
            Ks[tt * U + at(tt, u)] = make_float4(k.x * kscale, k.y * kscale, k.z * kscale, k.w * kscale);
            if (OUT) Qs[tt * U + at(tt, u)] = to_float(rq[it]);
        }
#pragma unroll
        for (int it = 0; it < VPF; ++it) {
            const int e = tid + it * 256;
            ((float4 *)Vs)[e] = to_float(rv[it]);                   // rows of 128 columns, those beyond Dv and tokens beyond the portion zero
        }
        __syncthreads();
        int broken = RM_T;                                          // the group's first token whose value in this lane's column is not finite
        if (t0 + RM_T < cnt) fetch(t0 + RM_T);                      // in flight while this group is multiplied
        for (int e = tid; e < nt * hu; e += 256) {                  // rotation in place: units u and u + half / 4 of a row
            const int tt = e / hu, u = e - tt * hu;
            int64_t p = a.pos[row0 + t0 + tt];
            if (p >= a.table_len) p = a.table_len - 1;
            const float4 c = *(const float4 *)(a.cos_t + p * half + 4 * u), s = *(const float4 *)(a.sin_t + p * half + 4 * u);
            auto turn = [&](float4 *rows) {
                float4 *x = rows + tt * U + at(tt, u), *y = rows + tt * U + at(tt, u + hu);
                const float4 v = *x, w = *y;
                *x = make_float4(v.x * c.x - w.x * s.x, v.y * c.y - w.y * s.y, v.z * c.z - w.z * s.z, v.w * c.w - w.w * s.w);
                *y = make_float4(w.x * c.x + v.x * s.x, w.y * c.y + v.y * s.y, w.z * c.z + v.z * s.z, w.w * c.w + v.w * s.w);
            };
            turn(Ks);
            if (OUT) turn(Qs);
        }
        __syncthreads();
        if (OUT) {
            for (int part = wave; part < 3; part += 4) {            // quadrants (queries, keys) of the pairs: (0, 0), (1, 0), (1, 1)
                const int qi = part > 0, qj = part > 1;
                rm_f32x16 s;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 0.f;
                const int ki = 32 * qj + l32, ii = 32 * qi + l32;
#pragma unroll 4
                for (int x = 0; x < U / 2; ++x) {
                    const float4 k = Ks[ki * U + at(ki, 2 * x + hi)], q = Qs[ii * U + at(ii, 2 * x + hi)];
                    s = rm_mma(k.x, q.x, s);
                    s = rm_mma(k.y, q.y, s);
                    s = rm_mma(k.z, q.z, s);
                    s = rm_mma(k.w, q.w, s);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int j0 = 32 * qj + 8 * g + 4 * hi;
                    float v[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = j0 + x <= ii ? s[4 * g + x] * gp[ii - j0 - x > 0 ? ii - j0 - x : 0] : 0.f;
                    Ps[ii * 16 + at(ii, j0 >> 2)] = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
            __syncthreads();
            rm_f32x16 o[2];
            if (wave < nw) {
                for (bool first_time = true;; first_time = false) {
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[rt][r] = 0.f;
                    }
#pragma unroll
                    for (int x = 0; x < U / 2; ++x) {
                        if (x % 2 == 0) __builtin_amdgcn_sched_barrier(0);      // all operands at once would not fit the registers
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) {
                            const int i = 32 * rt + l32;
                            const float4 q = Qs[i * U + at(i, 2 * x + hi)];
                            o[rt] = rm_mma(q.x, S[x >> 2][4 * (x & 3)], o[rt]);
                            o[rt] = rm_mma(q.y, S[x >> 2][4 * (x & 3) + 1], o[rt]);
                            o[rt] = rm_mma(q.z, S[x >> 2][4 * (x & 3) + 2], o[rt]);
                            o[rt] = rm_mma(q.w, S[x >> 2][4 * (x & 3) + 3], o[rt]);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[rt][r] *= gp[32 * rt + 8 * (r >> 2) + 4 * hi + (r & 3) + 1];
                    auto pairs = [&](int x, int first) {                // eight keys; no key of the second half is visible to the first half's queries
                        float v[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = Vs[(8 * x + 4 * hi + i) * 128 + col];
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) {
                            if (rt < first) continue;
                            const int i = 32 * rt + l32;
                            const float4 p = Ps[i * 16 + at(i, 2 * x + hi)];
                            o[rt] = rm_mma(p.x, v[0], o[rt]);
                            o[rt] = rm_mma(p.y, v[1], o[rt]);
                            o[rt] = rm_mma(p.z, v[2], o[rt]);
                            o[rt] = rm_mma(p.w, v[3], o[rt]);
                        }
                    };
#pragma unroll 2
                    for (int x = 0; x < 4; ++x) pairs(x, 0);
#pragma unroll 2
                    for (int x = 4; x < 8; ++x) pairs(x, 1);
                    // A value that is not finite makes every sum of its column none, through weights of zero also those of tokens in front of it.  Then, once more without it: what it
                    // reaches is set below.  (All keys enter a row of the second half.)
                    if (!first_time || !__any(!__builtin_isfinite(o[1][0]))) break;
                    for (int j = RM_T - 1; j >= 0; --j)
                        if (!__builtin_isfinite(Vs[j * 128 + col])) {
                            broken = j;
                            if (hi) Vs[j * 128 + col] = 0.f;        // the column's other lane looks at it in the same instruction
                        }
                    if (!__any(broken < RM_T)) break;
                }
                if (col < Dv) {                                     // as they are: the norm over a head's Dv columns spans wavefronts, and a gate's bytes are better read in rows
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int i = 32 * rt + 8 * (r >> 2) + 4 * hi + (r & 3);
                            if (i < nt) a.raw[(int64_t)(row0 + t0 + i) * ((int64_t)H * Dv) + h * Dv + col] = i < broken ? o[rt][r] : NAN;
                        }
                }
            }
        }
        if (wave < nw && (!OUT || last || t0 + RM_T < cnt)) {       // the state behind the group
            const float gn = gp[nt];
#pragma unroll
            for (int t = 0; t < NS; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) S[t][r] *= gn;
#pragma unroll 1
            for (int x = 0; 8 * x < nt; ++x) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = 8 * x + 4 * hi + i;
                    const float v = Vs[j * 128 + col] * gp[nt - 1 - j > 0 ? nt - 1 - j : 0];
#pragma unroll
                    for (int t = 0; t < NS; ++t) {
                        const int d = 32 * t + l32;
                        S[t] = rm_mma(((const float *)(Ks + j * U + at(j, d >> 2)))[d & 3], v, S[t]);
                    }
                }
            }
            if (OUT && broken < RM_T)
#pragma unroll
                for (int t = 0; t < NS; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) S[t][r] = NAN;
        }
    }
    float *dst = OUT ? a.state + ((int64_t)slot * H + h) * D * Dv : sp;
    if (col < Dv && (!OUT || last))
#pragma unroll
        for (int t = 0; t < NS; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int d = 32 * t + 8 * (r >> 2) + 4 * hi + (r & 3);
                if (d < D) dst[(int64_t)d * Dv + col] = S[t][r];
            }
}

// The state every piece of a request starts from, in place of the piece's own contribution: S = the slot's state (zero at position 0), then for every piece but
// the last S <- g^tokens S + contribution.  Every piece but the last of a request is `tokens` long.
__global__ __launch_bounds__(256) void retention_pieces_join_kernel(jl_retention_pieces a) {
    const int b = blockIdx.x / a.H, h = blockIdx.x - b * a.H;
    const int p0 = a.req[4 * b], np = a.req[4 * b + 1], pos0 = a.req[4 * b + 2], slot = a.req[4 * b + 3];
    const int64_t ddv = (int64_t)a.D * a.Dv;
    double power = 1.0, g2 = a.decay[h];
    for (int n = a.piece_tokens; n; n >>= 1) {
        if (n & 1) power *= g2;
        g2 *= g2;
    }
    const float gn = (float)power;
    const float *sp = a.state + ((int64_t)slot * a.H + h) * ddv;
    for (int64_t e = (int64_t)blockIdx.y * 256 + threadIdx.x; e < ddv; e += (int64_t)gridDim.y * 256) {
        float S = pos0 > 0 ? sp[e] : 0.f;
        float next = np > 1 ? a.scratch[((int64_t)p0 * a.H + h) * ddv + e] : 0.f;
        for (int p = p0; p < p0 + np; ++p) {
            float *lp = a.scratch + ((int64_t)p * a.H + h) * ddv + e;
            const float local = next;
            next = p + 2 < p0 + np ? lp[(int64_t)a.H * ddv] : 0.f;  // the last piece has none
            *lp = S;
            S = gn * S + local;
        }
    }
}

extern "C" int jl_retention_pieces_ok(int dtype, int32_t D, int32_t Dv, int32_t rot_dims) {
    return (dtype == JL_BF16 || dtype == JL_F32) && D > 0 && D <= 128 && D % 4 == 0 && Dv > 0 && Dv <= 128 && Dv % 4 == 0 && rot_dims >= 0 && rot_dims <= D && rot_dims % 8 == 0;
}

template <typename T, int DP> static int rm_launch(const jl_retention_pieces &a, hipStream_t st) {
    auto local = retention_pieces_kernel<T, DP, RM_LOCAL>;
    auto outs = retention_pieces_kernel<T, DP, RM_OUT>;
    constexpr size_t l0 = rm_lds_bytes(DP, false), l1 = rm_lds_bytes(DP, true);
    hipError_t e = hipFuncSetAttribute((const void *)local, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l0);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)outs, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l1);
    if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_retention_pieces_run: cannot get %zu bytes of LDS: %s", l1, hipGetErrorString(e));
    const dim3 grid((unsigned)a.pieces, (unsigned)a.H);
    if (a.pieces > a.B) local<<<grid, 256, l0, st>>>(a);
    const int64_t ddv = (int64_t)a.D * a.Dv;
    retention_pieces_join_kernel<<<dim3((unsigned)(a.B * a.H), (unsigned)((ddv + 255) / 256 < 64 ? (ddv + 255) / 256 : 64)), 256, 0, st>>>(a);
    outs<<<grid, 256, l1, st>>>(a);
    const int rc = jl_check_launch("retention_pieces_kernel");
    return rc != JL_OK ? rc : jl_heads_out(a.raw, a.proj, a.dtype, a.ld, a.g_col, nullptr, a.N * a.H, a.H, a.Dv, a.eps, a.out, st);
}

extern "C" int jl_retention_pieces_run(const jl_retention_pieces *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_retention_pieces_run: null arguments");
    const jl_retention_pieces &a = *ap;
    if (a.B <= 0 || a.pieces <= 0) return JL_OK;
    if (!a.proj || !a.decay || !a.state || !a.out || !a.scratch || !a.raw || a.N <= 0 || !a.piece_rec || !a.req || !a.pos || (a.rot_dims && (!a.cos_t || !a.sin_t || a.table_len <= 0)))
        return jl_fail(JL_E_INVALID, "jl_retention_pieces_run: null pointer");
    if (!jl_retention_pieces_ok(a.dtype, a.D, a.Dv, a.rot_dims) || a.H <= 0 || a.H > 65535 || a.piece_tokens <= 0 || a.piece_tokens % RM_T || a.ld % 4 || (a.q_col | a.k_col | a.v_col) % 4 ||
        ((uintptr_t)a.proj % (a.dtype == JL_BF16 ? 8 : 16)) || ((uintptr_t)a.cos_t % 16) || ((uintptr_t)a.sin_t % 16))
        return jl_fail(JL_E_INVALID, "jl_retention_pieces_run: sizes, columns or alignment (ask jl_retention_pieces_ok)");
    hipStream_t st = (hipStream_t)stream;
    if (a.D <= 64) JL_DISPATCH(a.dtype, return (rm_launch<T, 64>(a, st)));
    JL_DISPATCH(a.dtype, return (rm_launch<T, 128>(a, st)));
    return JL_OK;
}
