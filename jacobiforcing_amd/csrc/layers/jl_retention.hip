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

// ---- long portions in pieces side by side, 32 tokens at a time on the bfloat16 matrix instructions ----------------------------------------------
// With g = the head's decay, a group of n tokens is three products on the state S the group starts from:
//   o_i = g^(i+1) S^T q_i + sum_{j <= i} g^(i-j) (q_i . k_j) v_j,          S <- g^n S + sum_j g^(n-1-j) k_j v_j^T.
// A portion is cut into pieces (whole groups, except the last) that run side by side: every piece's own contribution to the state (RM_LOCAL, not for a
// request's last piece), the state every piece starts from (retention_pieces_join_kernel), outputs (RM_OUT; the last piece leaves the final state in its slot).
// q and k are 32-bit numbers behind their rotation, as are the state, the pairs' weights and the decayed values: each enters the products as the sum of three bfloat16 numbers, of whose nine products six are
// formed (jl_split8; bfloat16 values are one number).  The terms of q and k are made once per group, on the way into LDS, the others in the registers that hold them: a workgroup owns one head of one
// piece, wavefront w columns 32 w .. + 31 of S [D, Dv] in accumulators.  Accumulator r of lane l of a 32 x 32 product is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32, so registers 8s .. 8s + 7 are an operand
// over the depths 16s + 4 (l / 32) + {0 .. 3, 8 .. 11} as they are: the state as B of S^T q, the weights of the pairs (formed turned, K Q^T, by every wavefront for itself) as A of the sum over values.
// q and k rows are read in that order as two 8-byte halves; k (for the state) and v are turned by ds_read_b64_tr_b16.  Two barriers per group.
// What bounds it: issue and latency at two workgroups per CU; 150 products of 32 cycles per group and wavefront (4 800 cycles) beside splits, rotations and
// LDS reads, where a group takes 14 us with all of them.
// Before, 64 tokens at a time on the float matrix instructions (368 products of 64 cycles per wavefront, rotated in LDS behind a barrier of their own, the pairs' weights through LDS, one workgroup per CU).
// us, 8 heads of 128 x 128, bfloat16, 4 x 2048 tokens, outputs / contributions: 121 / 54 then, 58 / 26 now; the whole layer 188 / 117, one portion of 128 51 / 36, of 1000 60 / 47, 8 of 8 33 / 24; 8 heads of 64 109 / 70;
// float, 1021 + 851 + 681 tokens 105 / 80.  Error of the states against 64 bits 2.1e-7 then, 1.7e-7 now.
// Values that are not finite reach the tokens from their own on and the state, as in the scan, though products run over whole groups: they are left out of them, and their columns' outputs and state set behind.
// Numbers that no bfloat16 number comes near (infinities, and floats between the two types' ends) have no terms: groups whose outputs are not all finite, and contributions of keys or values like that, are
// formed on the float instructions from the numbers themselves, so that sums of one sign stay infinite and finite ones finite (looking for them takes 2 %: 4 x 2048 tokens 104 / 106 us).  Numbers below
// 2^-118 lose the digits of their terms that lie below bfloat16's last place, 2^-133.
// The instructions cut what they add to a sum towards minus infinity, which would make all states and outputs lean one way (states by 0.1e-7 of their root mean square at decays of 0.97, 0.4e-7 at 0.9998, and
// with them all tokens to come); so states and queries have a minus sign in half of the groups, which leaves 0.01e-7 and 0.09e-7.  us of the whole layer, without / with: 4 x 2048 tokens 100.6 / 103.8, of 64 62.9 / 65.0,
// the float ones 77.1 / 79.6, one portion of 128 33.9 / 35.6.
// Outputs leave as floats and are normed and gated by rows in a launch of their own.
constexpr int RM_T = 64, RC_T = 32, RM_OUT = 0, RM_LOCAL = 1, RC_VROW = 128 + 16;      // RM_T: pieces come in multiples of it
typedef float rm_f32x16 __attribute__((ext_vector_type(16)));
typedef float rm_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 rm_bf16x4 __attribute__((ext_vector_type(4)));
typedef short rm_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) rm_s16x4 rm_lds_s16x4;
constexpr int RM_TERMS = JL_SPLIT_TERMS;
__device__ __forceinline__ float rm_signed(float v, uint32_t sign) { return __uint_as_float(__float_as_uint(v) ^ sign); }
constexpr float RM_BEYOND = 3.395e38f;                               // bfloat16 ends at 3.3895e38; from 3.3953e38 on a float is rounded to infinity
template <typename T> static constexpr size_t rm_lds_bytes(int DP, bool out) {
    return 2 * RC_T * ((out ? 2 : 1) * (size_t)RM_TERMS * (DP + 8) + (sizeof(T) == 4 ? RM_TERMS : 1) * RC_VROW) + (RC_T + 4 * RC_T + 4 * RC_T + 4) * 4;
}

template <typename T, int DP, int MODE>
__global__ __launch_bounds__(256, sizeof(T) == 4 && DP > 64 ? 1 : 2) void retention_pieces_kernel(jl_retention_pieces a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr bool OUT = MODE == RM_OUT;
    constexpr int QROW = DP + 8, SLOTS = DP / 8, QIT = RC_T * SLOTS / 256, VIT = RC_T * 32 / 256, NS = DP / 32, VT = sizeof(T) == 4 ? RM_TERMS : 1;
    const int piece = blockIdx.x, h = blockIdx.y, H = a.H, D = a.D, Dv = a.Dv;
    const int row0 = a.piece_rec[4 * piece], cnt = a.piece_rec[4 * piece + 1], slot = a.piece_rec[4 * piece + 2], last = a.piece_rec[4 * piece + 3];
    if (cnt <= 0 || (!OUT && last)) return;
    bf16_t *Ks = (bf16_t *)smem, *Vs = Ks + RM_TERMS * RC_T * QROW, *Qs = Vs + VT * RC_T * RC_VROW;      // [terms][32][..]
    float *g1 = (float *)(Qs + (OUT ? RM_TERMS * RC_T * QROW : 0)), *powers = g1 + RC_T;     // g^(i+1); g^(31-m), none from 32 on, and all that with a minus sign
    int *brokenS = (int *)(powers + 4 * RC_T), *flawS = brokenS + 4 * RC_T;                     // per column: the group's first token whose value is not finite; whether this group, the one before, has one
    int *beyondS = flawS + 2;                                                                // RM_LOCAL: whether this group, the one before, has a key or value that no bfloat16 number comes near
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hi = lane >> 5, col = 32 * wave + l32;
    const bool busy = 32 * wave < Dv;
    const float gamma = a.decay[h], kscale = 1.0f / sqrtf((float)D);
    if (wave == 0) {                                                // powers by doubling, which doubles a rounding error too: in 64 bits.  Lane l holds g^(l+1)
        double p = gamma;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double y = __shfl_up(p, off, 64);
            if (lane >= off) p *= y;
        }
        if (lane < RC_T) g1[lane] = (float)p;
        const double q = __shfl(p, lane < 31 ? 30 - lane : 0, 64);
        const float d = lane < 31 ? (float)q : lane == 31 ? 1.0f : 0.f;
        powers[lane] = d;
        powers[2 * RC_T + lane] = -d;
        if (lane < 4) flawS[lane] = 0;
    }
    const T *src = (const T *)a.proj + (int64_t)row0 * a.ld;
    const int half = a.rot_dims >> 1, hu = half / 4;
    const int64_t pos0 = half ? a.pos[row0] : 0;                    // a portion's positions follow each other

    rm_f32x16 S[NS];
    float *sp = a.scratch + ((int64_t)piece * H + h) * D * Dv;
    // f(row of the state, byte offset in it, register): one address that moves on, not sixty-four in registers
    auto each_state = [&](auto &&f) {
        uint32_t off = (uint32_t)(4 * hi * Dv + col) * 4;
#pragma unroll
        for (int t = 0; t < NS; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                asm volatile("" : "+v"(off));
                S[t][r] = f(32 * t + 8 * (r >> 2) + 4 * hi + (r & 3), off, S[t][r]);
                off += ((r & 3) == 3 ? 5 : 1) * Dv * 4;
            }
    };
    each_state([&](int d, uint32_t off, float) { return (OUT && d < D && col < Dv) ? *(const float *)((const char *)sp + off) : 0.f; });
    // a group's rows on their way.  A thread's share of q and k: pairs of units of four dimensions that are rotated together (or two that are not)
    typedef typename std::conditional<sizeof(T) == 2, uint2, rm_f32x4>::type unit_t;
    unit_t rq[QIT][2], rk[QIT][2], rv[VIT];
    rm_f32x4 rc[QIT], rs[QIT];
    const int pair = tid % SLOTS, ua = pair < hu ? pair : 2 * pair, ub = pair < hu ? pair + hu : 2 * pair + 1;
    const bool turns = pair < hu, in_a = 4 * ua < D, in_b = 4 * ub < D;
    auto fetch = [&](int t0) {
        const int nt = cnt - t0;
        const T *base = src + (int64_t)t0 * a.ld;
        const unit_t zero = {};
#pragma unroll
        for (int it = 0; it < QIT; ++it) {
            const int tt = tid / SLOTS + it * (256 / SLOTS);
            rk[it][0] = rk[it][1] = rq[it][0] = rq[it][1] = zero;
            if (tt < nt) {
                const T *k = base + (int64_t)tt * a.ld + h * D + a.k_col, *q = base + (int64_t)tt * a.ld + h * D + a.q_col;
                if (in_a) rk[it][0] = *(const unit_t *)(k + 4 * ua);
                if (in_b) rk[it][1] = *(const unit_t *)(k + 4 * ub);
                if (OUT && in_a) rq[it][0] = *(const unit_t *)(q + 4 * ua);
                if (OUT && in_b) rq[it][1] = *(const unit_t *)(q + 4 * ub);
                if (turns) {
                    const int64_t p = pos0 + t0 + tt < a.table_len ? pos0 + t0 + tt : a.table_len - 1;
                    rc[it] = *(const rm_f32x4 *)(a.cos_t + p * half + 4 * ua);
                    rs[it] = *(const rm_f32x4 *)(a.sin_t + p * half + 4 * ua);
                }
            }
        }
#pragma unroll
        for (int it = 0; it < VIT; ++it) {
            const int e = tid + it * 256, tt = e >> 5, u = e & 31;
            rv[it] = zero;
            if (tt < nt && 4 * u < Dv) rv[it] = *(const unit_t *)(base + (int64_t)tt * a.ld + a.v_col + h * Dv + 4 * u);
        }
    };
    auto to_float = [](const unit_t &w, const unit_t &x) {
        float v[4], u[4];
        ld4_f((const T *)&w, v);
        ld4_f((const T *)&x, u);
        return jl_f32x8{v[0], v[1], v[2], v[3], u[0], u[1], u[2], u[3]};
    };
    auto put = [](bf16_t *to, const jl_bf16x8 &v, int part) {       // four of the eight
        *(rm_bf16x4 *)to = part ? __builtin_shufflevector(v, v, 4, 5, 6, 7) : __builtin_shufflevector(v, v, 0, 1, 2, 3);
    };
    // turned operands: column (or row) l % 32 of 32 columns from c on, tokens 16 s + 4 hi + {0 .. 3, 8 .. 11}
    const int tr_row = 4 * hi + ((lane & 15) >> 2), tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto turned = [&](const bf16_t *tile, int row_len, int c, int s) {
        rm_s16x4 part[2];
#pragma unroll
        for (int y = 0; y < 2; ++y) part[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((rm_lds_s16x4 *)(tile + (16 * s + 8 * y + tr_row) * row_len + c + tr_col));
        return __builtin_bit_cast(jl_bf16x8, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto row_of = [&](const bf16_t *tile, int s) {                  // row l % 32, depths 16 s + 4 hi + {0 .. 3, 8 .. 11}
        const rm_bf16x4 x = *(const rm_bf16x4 *)(tile + l32 * QROW + 16 * s + 4 * hi), y = *(const rm_bf16x4 *)(tile + l32 * QROW + 16 * s + 8 + 4 * hi);
        return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto acc8 = [](const rm_f32x16 &v, int s) {
        jl_f32x8 f;
#pragma unroll
        for (int x = 0; x < 8; ++x) f[x] = v[8 * s + x];
        return f;
    };
    // what the terms stand for, from memory: the value of token t of a group at depth d of q or k, turned and scaled, and of v at this lane's column
    auto whole = [&](int from, float scale, int t0, int nt, int t, int d) {
        asm volatile("" : "+v"(t), "+v"(d));                        // nothing of it is worth a register in the loop around
        if (t >= nt || d >= D) return 0.f;
        const T *x = src + (int64_t)(t0 + t) * a.ld + h * D + from;
        const float u = ld_f(x + d) * scale;
        if (d >= 2 * half) return u;
        const int64_t p = (pos0 + t0 + t < a.table_len ? pos0 + t0 + t : a.table_len - 1) * half + (d < half ? d : d - half);
        const float w = ld_f(x + (d < half ? d + half : d - half)) * scale, c = a.cos_t[p], s = a.sin_t[p];
        return d < half ? u * c - w * s : u * c + w * s;
    };
    auto value = [&](int t0, int nt, int t) {                       // (one that is not finite is left out of outputs and set behind them, as in the terms)
        asm volatile("" : "+v"(t));
        const float v = t < nt && col < Dv ? ld_f(src + (int64_t)(t0 + t) * a.ld + a.v_col + h * Dv + col) : 0.f;
        return OUT && !__builtin_isfinite(v) ? 0.f : v;
    };
    fetch(0);
    uint32_t held = 0u;
    for (int t0 = 0; t0 < cnt; t0 += RC_T) {
        const int nt = cnt - t0 < RC_T ? cnt - t0 : RC_T;
        // the signs that this group's queries have (+ - + -) and the state behind it is held with (+ - - +), a group whose products go with either in turn
        const uint32_t asked = (uint32_t)(t0 / RC_T) << 31, next = (uint32_t)((t0 / RC_T + 1) >> 1) << 31;
        const float *dec = powers + (held ? 2 * RC_T : 0);
        uint32_t given = asked ^ held;                              // and its outputs
        __syncthreads();                                            // the group before has been read
        float big = 0.f;                                            // of keys and values, where no outputs tell (NaN passes: it reaches the same sums either way)
#pragma unroll
        for (int it = 0; it < QIT; ++it) {
            const int tt = tid / SLOTS + it * (256 / SLOTS);
            auto stage = [&](bf16_t *rows, jl_f32x8 v, bool key, uint32_t sign) {
                if (turns && tt < nt) {
                    const jl_f32x8 w = v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) { v[i] = w[i] * rc[it][i] - w[4 + i] * rs[it][i]; v[4 + i] = w[4 + i] * rc[it][i] + w[i] * rs[it][i]; }
                }
                if (!OUT && key)
#pragma unroll
                    for (int i = 0; i < 8; ++i) big = fmaxf(big, fabsf(v[i]));
                if (!key)
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = rm_signed(v[i], sign);
                jl_bf16x8 part[RM_TERMS];
                jl_split8(v, part);
#pragma unroll
                for (int x = 0; x < RM_TERMS; ++x) {
                    put(rows + (x * RC_T + tt) * QROW + 4 * ua, part[x], 0);
                    put(rows + (x * RC_T + tt) * QROW + 4 * ub, part[x], 1);
                }
            };
            stage(Ks, to_float(rk[it][0], rk[it][1]) * kscale, true, 0u);
            if (OUT) stage(Qs, to_float(rq[it][0], rq[it][1]), false, asked);
        }
        float zero = 0.f;                                           // not a number with a value that is not finite
#pragma unroll
        for (int it = 0; it < VIT; it += 2) {                       // rows of 128 columns, those beyond Dv and tokens beyond the portion zero
            const jl_f32x8 v = to_float(rv[it], rv[it + 1]);
            if (OUT)
#pragma unroll
                for (int i = 0; i < 8; ++i) zero = __builtin_fmaf(v[i], 0.f, zero);
            if (!OUT)
#pragma unroll
                for (int i = 0; i < 8; ++i) big = fmaxf(big, fabsf(v[i]));
            jl_bf16x8 part[RM_TERMS];
            if (VT > 1) jl_split8(v, part);
            else part[0] = __builtin_convertvector(v, jl_bf16x8);
#pragma unroll
            for (int x = 0; x < VT; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const int e = tid + (it + y) * 256;
                    put(Vs + (x * RC_T + (e >> 5)) * RC_VROW + 4 * (e & 31), part[x], y);
                }
        }
        if (OUT && zero != 0.f) flawS[t0 / RC_T & 1] = 1;
        if (!OUT && big >= RM_BEYOND) beyondS[t0 / RC_T & 1] = 1;
        __syncthreads();
        bool beyond = false;                                        // the group takes the float instructions
        if (!OUT) {
            beyond = __builtin_amdgcn_readfirstlane(beyondS[t0 / RC_T & 1]);
            if (tid == 0) beyondS[~(t0 / RC_T) & 1] = 0;
        }
        bool flawed = false;
        if (OUT) {
            flawed = __builtin_amdgcn_readfirstlane(flawS[t0 / RC_T & 1]);
            if (tid == 0) flawS[~(t0 / RC_T) & 1] = 0;
            if (flawed && busy) {                                   // such values are left out of the products; what they reach is set behind them
                int broken = RC_T;
                for (int t = 16 * hi; t < 16 * hi + 16; ++t) {
                    float v = 0.f;
                    for (int x = 0; x < VT; ++x) v += ld_f(Vs + (x * RC_T + t) * RC_VROW + col);
                    if (__builtin_isfinite(v)) continue;
                    broken = min(broken, t);
                    for (int x = 0; x < VT; ++x) Vs[(x * RC_T + t) * RC_VROW + col] = 0;
                }
                broken = min(broken, __shfl_xor(broken, 32, 64));
                brokenS[32 * wave + l32] = broken;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (t0 + RC_T < cnt) fetch(t0 + RC_T);                      // in flight while this group is multiplied
        if (!busy) continue;
        jl_bf16x8 vf[VT][2];
#pragma unroll
        for (int x = 0; x < VT; ++x)
#pragma unroll
            for (int s = 0; s < 2; ++s) vf[x][s] = turned(Vs + x * RC_T * RC_VROW, RC_VROW, 32 * wave, s);
        if (OUT) {
            rm_f32x16 o, p;                                         // outputs; weights of the pairs, turned
#pragma unroll
            for (int r = 0; r < 16; ++r) o[r] = p[r] = 0.f;
#pragma unroll
            for (int s = 0; s < DP / 16; ++s) {
                jl_bf16x8 qf[RM_TERMS], kf[RM_TERMS], sf[RM_TERMS];
#pragma unroll
                for (int x = 0; x < RM_TERMS; ++x) { qf[x] = row_of(Qs + x * RC_T * QROW, s); kf[x] = row_of(Ks + x * RC_T * QROW, s); }
                jl_split8(acc8(S[s >> 1], s & 1), sf);
#pragma unroll
                for (int d = RM_TERMS - 1; d >= 0; --d)             // the terms whose numbers add up to d
#pragma unroll
                    for (int x = 0; x <= d; ++x) {
                        p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[x], qf[d - x], p, 0, 0, 0);
                        o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[x], sf[d - x], o, 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);       // all operands at once would not fit the registers
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const rm_f32x4 g4 = *(const rm_f32x4 *)(g1 + 8 * x + 4 * hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[4 * x + i] *= g4[i];
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                jl_f32x8 w = acc8(p, s);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int j = 16 * s + 4 * hi + (i & 3) + 8 * (i >> 2);
                    const float f = w[i] * dec[31 - l32 + j];
                    w[i] = j <= l32 ? f : 0.f;
                }
                jl_bf16x8 wf[RM_TERMS];
                jl_split8(w, wf);
#pragma unroll
                for (int d = RM_TERMS - 1; d >= 0; --d)
#pragma unroll
                    for (int x = 0; x <= d; ++x)
                        if (d - x < VT) o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[x], vf[d - x < VT ? d - x : 0][s], o, 0, 0, 0);
            }
            float odd = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) odd = __builtin_fmaf(o[r], 0.f, odd);
            beyond = __ballot(odd != 0.f) != 0;                     // not a number in some lane (a key or value like that is in its own token's output)
            if (beyond) {
#pragma unroll
                for (int r = 0; r < 16; ++r) o[r] = p[r] = 0.f;
#pragma unroll
                for (int t = 0; t < NS; ++t)
#pragma unroll 1
                    for (int r = 0; r < 16; ++r) {
                        const int d = 32 * t + 8 * (r >> 2) + 4 * hi + (r & 3);
                        const float q = whole(a.q_col, 1.0f, t0, nt, l32, d), k = whole(a.k_col, kscale, t0, nt, l32, d);
                        p = __builtin_amdgcn_mfma_f32_32x32x2f32(k, q, p, 0, 0, 0);
                        o = __builtin_amdgcn_mfma_f32_32x32x2f32(q, S[t][r], o, 0, 0, 0);
                    }
#pragma unroll
                for (int r = 0; r < 16; ++r) o[r] *= rm_signed(g1[8 * (r >> 2) + 4 * hi + (r & 3)], held);
                given = 0u;
#pragma unroll 1
                for (int r = 0; r < 16; ++r) {
                    const int j = 8 * (r >> 2) + 4 * hi + (r & 3);
                    o = __builtin_amdgcn_mfma_f32_32x32x2f32(j <= l32 ? p[r] * powers[31 - l32 + j] : 0.f, value(t0, nt, j), o, 0, 0, 0);
                }
            }
            const int broken = flawed ? brokenS[32 * wave + l32] : RC_T;
            if (col < Dv) {                                         // as they are: the norm over a head's Dv columns spans wavefronts, and a gate's bytes are better read in rows
                const uint32_t o_row = (uint32_t)(H * Dv) * 4;
                char *to = (char *)(a.raw + (int64_t)(row0 + t0) * ((int64_t)H * Dv) + h * Dv);
                uint32_t off = 4 * hi * o_row + 4 * col;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    asm volatile("" : "+v"(off));
                    const int i = 8 * (r >> 2) + 4 * hi + (r & 3);
                    if (i < nt) *(float *)(to + off) = i < broken ? rm_signed(o[r], given) : NAN;
                    off += (r & 3) == 3 ? 5 * o_row : o_row;
                }
            }
        }
        if (!OUT || last || t0 + RC_T < cnt) {                      // the state behind the group
            const float gn = rm_signed(g1[nt - 1], held ^ next);
            held = next;
            dec = powers + (held ? 2 * RC_T : 0);
#pragma unroll
            for (int t = 0; t < NS; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) S[t][r] *= gn;
            if (beyond) {
#pragma unroll
                for (int t = 0; t < NS; ++t)
#pragma unroll 1
                    for (int r = 0; r < 16; ++r) {
                        const int j = 8 * (r >> 2) + 4 * hi + (r & 3);
                        S[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(whole(a.k_col, kscale, t0, nt, j, 32 * t + l32), value(t0, nt, j) * dec[RC_T - nt + j], S[t], 0, 0, 0);
                    }
            } else
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                jl_f32x8 v;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int j = 16 * s + 4 * hi + (i & 3) + 8 * (i >> 2);
                    float f = (float)vf[VT - 1][s][i];
#pragma unroll
                    for (int x = VT - 2; x >= 0; --x) f += (float)vf[x][s][i];
                    v[i] = f * dec[RC_T - nt + j];
                }
                jl_bf16x8 vd[RM_TERMS];
                jl_split8(v, vd);
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    jl_bf16x8 kf[RM_TERMS];
#pragma unroll
                    for (int x = 0; x < RM_TERMS; ++x) kf[x] = turned(Ks + x * RC_T * QROW, QROW, 32 * t, s);
#pragma unroll
                    for (int d = RM_TERMS - 1; d >= 0; --d)
#pragma unroll
                        for (int x = 0; x <= d; ++x) S[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[x], vd[d - x], S[t], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (OUT && flawed && brokenS[32 * wave + l32] < RC_T)
#pragma unroll
                for (int t = 0; t < NS; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) S[t][r] = NAN;
        }
    }
    char *dst = (char *)(OUT ? a.state + ((int64_t)slot * H + h) * D * Dv : sp);
    if (col < Dv && (!OUT || last)) each_state([&](int d, uint32_t off, float v) { if (d < D) *(float *)(dst + off) = rm_signed(v, held); return v; });
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
    constexpr size_t l0 = rm_lds_bytes<T>(DP, false), l1 = rm_lds_bytes<T>(DP, true);
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
