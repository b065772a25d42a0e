// jl_linear.hip — dense products of a few rows (decoding): out[n] = W x[n] (+ bias), W [O, K] read once.
#include "jl_small.h"
#include "jl_split.h"

// What bounds such a product is W's bytes when W is large and the way there when it is small (a launch alone is 3 us, a trip to memory 2 us).  So a workgroup's NW wavefronts
// share the depth of 16 * OT rows of W, every lane has LS_AHEAD pairs of 16-byte units of each of its rows of W and x (which comes from L2) on the way at once, straight into the
// operands of 16 x 16 products — no LDS in between, no barrier before the end.  The order of the depths is free as long as both operands agree: lane l supplies units l / 16 and
// 4 + l / 16 of each 128 bytes of row l % 16, so that a load takes 64 neighbouring bytes of every row.  The shares meet in LDS; a lane ends with four neighbouring columns of a row.
//
// The split (us of GPU time for 16 * OT rows of W and NW wavefronts, bfloat16, W from memory: 1 x 8 / 1 x 4 / 2 x 4 / 4 x 4):
//   W 1024 x 1024, 32 rows:  5.7 / 5.6 /  6.7 /  9.3     W 5120 x 2048, 32 rows: 16.3 / 15.8 / 12.8 / 18.0     W 32000 x 1024, 32 rows: 29.4 / 30.5 / 23.6 / 21.5
//   W 2048 x 4096, 16 rows: 11.3 / 11.4 / 16.2 / 25.8    W 5120 x 2048,  1 row:   8.7 /  9.0 /  9.2 / 13.4     W 32000 x 1024,  1 row:  17.7 / 14.5 / 16.3 / 17.4
// As long as 16 rows of W per workgroup come to no more workgroups than the chip has CUs, that is the best; beyond, x is read again by every workgroup that a CU runs, and more rows
// of W per workgroup pay (not for one row of x).  Library products of the same shapes take 8.2, 12.4, 24.0 / 14.9, 12.2, 18.7 us, and 11 us more of host time per call (19.5 / 8.6).
// Rows beyond 16 cost x's reads: the caller's rule (layer_ops.linear) leaves products to the library where a CU would read more than 128 KB of x.
template <typename TX, typename T, int NT, int OT, int NW>          // N <= 16 * NT rows of x, 16 * OT rows of W, NW wavefronts
__global__ __launch_bounds__(64 * NW) void linear_small_kernel(const TX *__restrict__ x, int64_t x_ld, const T *__restrict__ w, const T *__restrict__ bias, void *__restrict__ out,
                                                               int64_t out_ld, int N, int K, int O, int out_mode) {
    __shared__ ls_f32x4 part[NW][OT][NT][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, o0 = blockIdx.x * 16 * OT;
    ls_f32x4 acc[OT][NT];
    ls_products<TX, T, NT, OT, NW>(acc, x, x_ld, w, N, K, o0, O, wave, lane);
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
        for (int t = 0; t < NT; ++t) part[wave][o][t][lane] = acc[o][t];
    __syncthreads();
    for (int e = threadIdx.x; e < OT * NT * 64; e += 64 * NW) {
        const int l = e & 63, t = (e >> 6) % NT, ot = (e >> 6) / NT, n = 16 * t + (l & 15), o = o0 + 16 * ot + 4 * (l >> 4);
        if (n >= N || o >= O) continue;
        ls_f32x4 s = part[0][ot][t][l];
#pragma unroll
        for (int i = 1; i < NW; ++i) s += part[i][ot][t][l];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (o + i >= O) continue;
            float v = s[i];
            if (bias) v += ld_f(bias + o + i);
            if (out_mode == JL_LINEAR_FLOAT) ((float *)out)[n * out_ld + o + i] = v;
            else if (out_mode == JL_LINEAR_ROUNDED_FLOAT) {
                TX r;
                st_f(&r, v);
                ((float *)out)[n * out_ld + o + i] = ld_f(&r);
            } else st_f((TX *)out + n * out_ld + o + i, v);
        }
    }
}

template <typename TX, typename T, int NT>
static void linear_small_launch(const void *x, int64_t x_ld, const void *w, const void *bias, void *out, int64_t out_ld, int N, int K, int O, int out_mode, hipStream_t st) {
#define LS_LAUNCH(OT, NW) linear_small_kernel<TX, T, NT, OT, NW><<<dim3((unsigned)((O + 16 * OT - 1) / (16 * OT))), 64 * NW, 0, st>>>((const TX *)x, x_ld, (const T *)w, (const T *)bias, out, \
                                                                                                                                 out_ld, N, K, O, out_mode)
    if (O <= JL_LINEAR_ONE_TILE) LS_LAUNCH(1, 8);
    else if (N == 1) LS_LAUNCH(1, 4);
    else if (O <= 4 * JL_LINEAR_ONE_TILE) LS_LAUNCH(2, 4);
    else LS_LAUNCH(4, 4);
#undef LS_LAUNCH
}

// ---- one row (or a few) that every workgroup makes for itself ------------------------------------------------------------------------------
// A token alone waits for launches: a norm, an activation or a gate in front of a product takes a launch of 4 us of the GPU and 5 of the host for a few KB.  Here each workgroup of 16 rows of W makes the
// product's operand itself, in LDS: what the rows are made of leaves memory first, this wavefront's weights right behind it, and the operand is made while they travel, all rows at once: their sums go
// through two barriers together.  Up to JL_LINEAR_ONE_TILE rows of W the product's sums are those of linear_small_kernel.  us of the GPU, launch and product / so, one, two and four rows (by 1024 values and 4096):
// norm 7.1 / 5.1, 7.2 / 5.7, 7.3 / 7.5 and 8.1 / 5.9, 7.9 / 6.6, 8.1 / 8.6; unit 6.3 / 3.6, 6.5 / 4.5, 6.7 / 5.9 and 7.2 / 4.5, 7.4 / 5.1, 7.7 / 6.5; gated norm 6.3 / 4.7, 6.5 / 5.2, 6.7 / 6.8 and
// 7.2 / 5.5, 7.4 / 5.9, 7.5 / 7.9; and the two calls take the host 9.5 us, the one 5.  (Rows one behind the other, two barriers a sum: norm, 1024 by 1024, 5.6, 7.0 and 9.7.)  Every workgroup repeats the
// rows' work: see jl_linear_after_ok.
// sums of the rows' values over the workgroup's eight wavefronts, all rows at once: one barrier
template <int R> __device__ __forceinline__ void la_sums(float (&v)[R], float (*red)[8], int wave, int lane) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] += __shfl_xor(v[r], off, 64);
    if (lane == 0)
#pragma unroll
        for (int r = 0; r < R; ++r) red[r][wave] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        v[r] = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) v[r] += red[r][w];
    }
}
template <int MODE, int VI, int R>                                  // R: rows, or one more than there are
__global__ __launch_bounds__(512) void linear_after_kernel(jl_linear_after a) {
    constexpr int NW = 8, STEP = 64 * NW * 4;
    __shared__ ls_f32x4 part[NW][64];
    __shared__ float red[2][R][8];
    extern __shared__ __attribute__((aligned(16))) bf16_t xs[];     // [N][K]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g4 = lane >> 4, o0 = blockIdx.x * 16, K = a.K, O = a.O, N = a.N;
    const int steps = (K + 63) / 64, s0 = steps * wave / NW, s1 = steps * (wave + 1) / NW, k_lane = 8 * g4;
    const bf16_t *wp = (const bf16_t *)a.w + (int64_t)(o0 + r16 < O ? o0 + r16 : O - 1) * K + k_lane;      // rows that do not exist repeat the last one and are not stored
    uint4 wr[LS_AHEAD][2];
    auto load = [&](int s) {
#pragma unroll
        for (int i = 0; i < LS_AHEAD; ++i)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int k = (s + i) * 64 + 32 * y;
                wr[i][y] = s + i < s1 && k + k_lane < K ? *(const uint4 *)(wp + k) : make_uint4(0, 0, 0, 0);
            }
    };
    const bool with = MODE == JL_AFTER_NORM && a.y, row = MODE == JL_AFTER_NORM && a.add_row;
    float x[R][VI][4], y[R][VI][4], post[VI][4], add[VI][4], next[VI][4];       // y: what is added, the gate, the linear branch
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int c = i * STEP + 4 * tid, n = R == 1 || r < N ? r : N - 1;
            if (c >= K) continue;
            if (MODE == JL_AFTER_ACT) {
                const bf16_t *z = (const bf16_t *)a.x + n * a.x_ld + c;
                ld4_f(z + a.g_col, x[r][i]);
                if (a.u_col >= 0) ld4_f(z + a.u_col, y[r][i]);
            } else {
                ld4_f((const float *)a.x + (int64_t)n * K + c, x[r][i]);
                if (MODE == JL_AFTER_GATED_NORM) ld4_f((const bf16_t *)a.y + n * a.y_ld + c, y[r][i]);
                else if (with) {
                    if (a.y_dtype == JL_BF16) ld4_f((const bf16_t *)a.y + (int64_t)n * K + c, y[r][i]);
                    else ld4_f((const float *)a.y + (int64_t)n * K + c, y[r][i]);
                }
            }
        }
    if (MODE != JL_AFTER_ACT)
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int c = i * STEP + 4 * tid;
            if (c >= K) continue;
            if (with) ld4_f(a.w_post + c, post[i]);
            if (row) ld4_f(a.add_row + c, add[i]);
            ld4_f(a.w_next + c, next[i]);
        }
    __builtin_amdgcn_sched_barrier(0);
    load(s0);
    __builtin_amdgcn_sched_barrier(0);
    float ss[R], scale[R];
    if (with) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ss[r] = 0.f;
#pragma unroll
            for (int i = 0; i < VI; ++i)
                if (i * STEP + 4 * tid < K) ss[r] += y[r][i][0] * y[r][i][0] + y[r][i][1] * y[r][i][1] + y[r][i][2] * y[r][i][2] + y[r][i][3] * y[r][i][3];
        }
        la_sums<R>(ss, red[0], wave, lane);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float f = 1.0f / sqrtf(ss[r] / (float)K + a.eps);
#pragma unroll
            for (int i = 0; i < VI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[r][i][e] += y[r][i][e] * f * post[i][e];
        }
    }
    if (MODE != JL_AFTER_ACT) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ss[r] = 0.f;
#pragma unroll
            for (int i = 0; i < VI; ++i) {
                if (i * STEP + 4 * tid >= K) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (row) x[r][i][e] += add[i][e];
                    if (MODE == JL_AFTER_GATED_NORM) {
                        y[r][i][e] = gate_act_f(y[r][i][e], a.kind);
                        if (a.gate_first) x[r][i][e] *= y[r][i][e];
                    }
                }
                if (MODE == JL_AFTER_NORM && blockIdx.x == 0 && (R == 1 || r < N)) st4_f(a.x_out + (int64_t)r * K + i * STEP + 4 * tid, x[r][i]);
                ss[r] += x[r][i][0] * x[r][i][0] + x[r][i][1] * x[r][i][1] + x[r][i][2] * x[r][i][2] + x[r][i][3] * x[r][i][3];
            }
        }
        la_sums<R>(ss, red[1], wave, lane);
#pragma unroll
        for (int r = 0; r < R; ++r) scale[r] = (MODE == JL_AFTER_GATED_NORM ? a.scale : 1.0f) / sqrtf(ss[r] / (float)K + a.eps);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            const int c = i * STEP + 4 * tid;
            if (c >= K || (R > 1 && r >= N)) continue;
            float to[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                to[e] = MODE == JL_AFTER_ACT ? gated_unit_f<true>(x[r][i][e], a.u_col >= 0 ? y[r][i][e] : 1.0f, a.kind, a.limit, a.alpha, a.shift)
                        : MODE == JL_AFTER_NORM ? next[i][e] * (x[r][i][e] * scale[r]) : next[i][e] * (x[r][i][e] * scale[r] * (a.gate_first ? 1.0f : y[r][i][e]));
            st4_f(xs + (int64_t)r * K + c, to);
        }
    __syncthreads();
    const bf16_t *xp = xs + (r16 < N ? r16 : N - 1) * K + k_lane;
    ls_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += LS_AHEAD) {
        if (s > s0) load(s);
#pragma unroll
        for (int i = 0; i < LS_AHEAD; ++i)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int k = (s + i) * 64 + 32 * y;
                acc = ls_mma((const bf16_t *)nullptr, wr[i][y], s + i < s1 && k + k_lane < K ? *(const uint4 *)(xp + k) : make_uint4(0, 0, 0, 0), acc);
            }
    }
    part[wave][lane] = acc;
    __syncthreads();
    const int o = o0 + 4 * g4;
    if (tid >= 64 || r16 >= N || o >= O) return;
    ls_f32x4 sum = part[0][lane];
#pragma unroll
    for (int i = 1; i < NW; ++i) sum += part[i][lane];
    bf16_t *out = (bf16_t *)a.out + (int64_t)r16 * O + o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (o + i < O) st_f(out + i, a.bias ? sum[i] + ld_f((const bf16_t *)a.bias + o + i) : sum[i]);
}

// One and two rows everywhere (us, launch and product / so: norm of one by 4096 values and 8192 23.3 / 18.6, of two 24.0 / 17.9, by 8192 and 8192 48.9 / 42.5; what loses there are units of two by 8192
// values, 4096 18.9 / 21.3).  Three and four, whose time is that of four, where the host's part outweighs what 256 workgroups repeat: norm of four by 512 and 2048 6.6 / 7.1, by 2048 and 4096 11.6 / 11.0,
// by 4096 and 1024 14.4 / 13.3, gated norm 13.0 / 14.0; beyond, by 1024 and 8192 10.2 / 11.0, by 4096 and 4096 gated norm 15.7 / 17.9, unit 13.4 / 15.4, and by 4096 and 8192, two workgroups a CU that
// do not fit, norm 24.3 / 31.8, gated norm 22.3 / 32.8.
extern "C" int jl_linear_after_ok(int64_t N, int64_t K, int64_t O) {
    if (N <= 0 || N > JL_AFTER_ROWS || K <= 0 || K % 8 || K > 8192 || (N > 2 ? 4 : N) * K > JL_AFTER_VALUES || O <= 0 || O > 8192) return 0;
    return N <= 2 || (O <= 4096 && (K <= 2048 || O <= 1024));
}
extern "C" int jl_linear_after_run(const jl_linear_after *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_linear_after_run: null arguments");
    const jl_linear_after &a = *ap;
    if (!a.x || !a.w || !a.out || !jl_linear_after_ok(a.N, a.K, a.O)) return jl_fail(JL_E_INVALID, "jl_linear_after_run: null pointer, or up to %d rows and %d values of theirs", JL_AFTER_ROWS, JL_AFTER_VALUES);
    auto al = [](const void *q, uintptr_t b) { return ((uintptr_t)q % b) == 0; };
    if (!al(a.x, 16) || !al(a.y, 8) || !al(a.w, 16) || !al(a.w_post, 16) || !al(a.add_row, 16) || !al(a.w_next, 16)) return jl_fail(JL_E_INVALID, "jl_linear_after_run: operands at 16-byte borders");
    if (a.mode == JL_AFTER_NORM ? !a.x_out || a.x_out == a.x || !al(a.x_out, 16) || !a.w_next || (a.y && (!a.w_post || (a.y_dtype != JL_BF16 && !al(a.y, 16))))
        : a.mode == JL_AFTER_ACT ? a.g_col < 0 || a.g_col % 4 || (a.u_col >= 0 && a.u_col % 4) || a.x_ld % 4 || a.g_col + (int64_t)a.K > a.x_ld || a.u_col + (int64_t)a.K > a.x_ld ||
                                       a.kind < JL_ACT_GELU_TANH || a.kind > JL_ACT_GELU_ERF
                                 : a.mode != JL_AFTER_GATED_NORM || !a.y || a.y_ld < a.K || a.y_ld % 4 || !a.w_next || (a.kind != JL_ACT_SILU && a.kind != JL_ACT_SIGMOID))
        return jl_fail(JL_E_INVALID, "jl_linear_after_run: bad operands for the mode");
    const dim3 grid((unsigned)((a.O + 15) / 16));
    const int lds = a.N * a.K * 2;
    hipStream_t st = (hipStream_t)stream;
#define LA_ROWS(M, VI)                                                                   \
    do {                                                                                  \
        if (a.N == 1) linear_after_kernel<M, VI, 1><<<grid, 512, lds, st>>>(a);            \
        else if (a.N == 2) linear_after_kernel<M, VI, 2><<<grid, 512, lds, st>>>(a);       \
        else if constexpr (VI <= 2) linear_after_kernel<M, VI, 4><<<grid, 512, lds, st>>>(a); \
    } while (0)
#define LA_MODE(M)                                                                       \
    do {                                                                                  \
        if (a.K <= 2048) LA_ROWS(M, 1);                                                    \
        else if (a.K <= 4096) LA_ROWS(M, 2);                                               \
        else LA_ROWS(M, 4);                                                                \
    } while (0)
    if (a.mode == JL_AFTER_NORM) LA_MODE(JL_AFTER_NORM);
    else if (a.mode == JL_AFTER_ACT) LA_MODE(JL_AFTER_ACT);
    else LA_MODE(JL_AFTER_GATED_NORM);
#undef LA_MODE
#undef LA_ROWS
    return jl_check_launch("linear_after_kernel");
}

// ---- some hundred to a few thousand rows: TM of x by TN of W per workgroup -------------------------------------------------------------------------
// Stages of 128 bytes of every row go from memory straight into a ring of RING buffers in LDS (16 bytes per lane, every lane fetching the unit that the permutation puts into its place).  A wavefront
// reads the next stage's operands into registers while it multiplies this one's, so that one barrier per stage says both that the next stage is there and that this one may be written over, and multiplies
// 16 x 16 tiles, whose sums wait for one another half as long as those of 32 x 32.  W's rows are the A operand and dealt out so that a lane ends with 4 * NT neighbouring columns of a row: 16 bytes a
// store and more.
// What bounds it: with few workgroups a stage's way (0.25 us before, operands read behind the barrier into one 32 x 32 tile; half of it now), with many what a CU takes in from L2, so tiles are as large
// as still give every CU one (linear_mid_tiles).  us of GPU time, operands from memory, library / 64 x 64 with 32 x 32 tiles before / this: 1024 x 1024 by 600 rows 9.2 / 8.1 / 7.0, by 1000 9.6 / 8.3 / 7.4,
// by 2048 11.1 / 10.6 / 9.9; 2048 x 1024 by 200 10.1 / 12.1 / 10.4, 1000 x 4864 by 896 21.9 / 27.3 / 21.3, 1536 x 1536 by 1300 14.3 / 14.0 / 12.4, 1024 x 1536 by 2048 13.9 / 16.1 / 14.1, 2048 x 2048 by
// 2048 22.6 / 32.4 / 23.5, 1024 x 4096 by 2048 22.2 / 33.2 / 23.2; and the call takes the host 5 us, the library's 21.
typedef uint32_t ld_u32x4 __attribute__((ext_vector_type(4)));
// GATED: W's rows are a unit's gates and behind them its O linear branches; a lane's first COLS / 2 columns are gates, the others their linear branches, and the unit leaves
// (2048 rows of 1024 by 2 x 2048: 24.9 us and 5.9 for the unit in a launch of its own, 24.5 so).
struct LinearUnit { int kind; float limit, alpha, shift; };
template <int TM, int TN, int WM, int WN, int RING, bool GATED>
__global__ __launch_bounds__(64 * WM * WN, (WM * WN >= 8 ? 1 : 2) * WM * WN / 4) void linear_mid_kernel(const bf16_t *__restrict__ x, int64_t x_ld, const bf16_t *__restrict__ w, const bf16_t *__restrict__ bias,
                                                                                                   void *__restrict__ out, int64_t out_ld, int N, int K, int O, int out_mode, int row_tiles, int tiles, LinearUnit unit) {
    constexpr int THREADS = 64 * WM * WN, U = 8, UNIT = 8, STAGE = 64, BUF = (TM + TN) * U, XT = TM / WM / 16, NT = TN / WN / 16, XL = TM * U / THREADS, WL = TN * U / THREADS, COLS = 4 * NT;
    static_assert(NT == 2 || NT == 4, "a lane's columns in whole stores");
    extern __shared__ __attribute__((aligned(16))) uint4 ldS[];
    // workgroups with the same remainder by 8 share an XCD; it walks strips of 1024 rows, column by column
    const int per_xcd = (tiles + 7) / 8, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;
    const int cols = tiles / row_tiles, high = 1024 / TM < row_tiles ? 1024 / TM : row_tiles, strip = tile / (high * cols), here = row_tiles - strip * high < high ? row_tiles - strip * high : high;
    const int in_strip = tile - strip * high * cols, n0 = (strip * high + in_strip % here) * TM, o0 = in_strip / here * (GATED ? TN / 2 : TN);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, quad = lane >> 4, wm = wave / WN, wn = wave % WN;
    // unit u of a row of LDS lies at u ^ swap: the sixteen rows that are read at once meet different banks.  Row 16 b + i of a wavefront's rows of W there is row COLS * (i / 4) + 4 b + i % 4 of them
    auto swap = [](int row) { return (row >> 1) & 7; };
    auto w_row = [](int m) { const int p = m % (16 * NT); return m - p + (p % 16 / 4) * COLS + p / 16 * 4 + p % 4; };
    const int lr = tid / U, lu = (tid % U) ^ swap(lr);              // rows step by 32 or 64: the permutation is the same
    uint32_t xo[XL], wo[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {                                  // rows that do not exist repeat the last one
        const int m = lr + THREADS / U * i, n = n0 + m;
        xo[i] = (uint32_t)((n < N ? n : N - 1) * x_ld + lu * UNIT) * 2;
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int r = w_row(lr + THREADS / U * i), linear = GATED && r % COLS >= COLS / 2, o = o0 + (GATED ? r / COLS * (COLS / 2) + r % (COLS / 2) : r);
        wo[i] = (uint32_t)(((o < O ? o : O - 1) + (linear ? O : 0)) * (int64_t)K + lu * UNIT) * 2;
    }
    const char *xb = (const char *)x, *wb = (const char *)w;
    const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)(ldS + wave * 64));
    const int full = K / STAGE;
    auto issue = [&](int s, int sel) {                              // behind the last stage, stage 0 again (never used): the number of loads on their way stays the same
        const int64_t k = s < full ? (int64_t)s * 128 : 0;
#pragma unroll
        for (int i = 0; i < XL; ++i) jl_load_lds(xb + k, xo[i], lds + (sel * BUF + i * THREADS) * 16);
#pragma unroll
        for (int i = 0; i < WL; ++i) jl_load_lds(wb + k, wo[i], lds + (sel * BUF + (XL + i) * THREADS) * 16);
    };
    ls_f32x4 acc[XT][NT];
#pragma unroll
    for (int a = 0; a < XT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = (ls_f32x4){0.f, 0.f, 0.f, 0.f};
    uint4 xf[2][2][XT], wf[2][2][NT];
    const int xs = (wm * (TM / WM) + l16) * U, ws = (TM + wn * (TN / WN) + l16) * U, p = swap(l16);
    auto read = [&](int sel, int to) {
        const uint4 *B = ldS + sel * BUF;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int u = (4 * k + quad) ^ p;
#pragma unroll
            for (int b = 0; b < NT; ++b) wf[to][k][b] = B[ws + 16 * b * U + u];
#pragma unroll
            for (int a = 0; a < XT; ++a) xf[to][k][a] = B[xs + 16 * a * U + u];
        }
    };
    auto products = [&](int from) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int a = 0; a < XT; ++a)
#pragma unroll
                for (int b = 0; b < NT; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ls_bf16x8, wf[from][k][b]), __builtin_bit_cast(ls_bf16x8, xf[from][k][a]), acc[a][b], 0, 0, 0);
    };
    if (full > 0) {
#pragma unroll
        for (int s = 0; s < RING; ++s) issue(s, s);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 1) * (XL + WL)) : "memory");
        __syncthreads();
        read(0, 0);
        int sel = 0;
        auto step = [&](int s, int from) {
            const int next = sel == RING - 1 ? 0 : sel + 1;
            // this stage's operands are in registers, the next stage has landed: everybody may write over this one
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((RING - 2) * (XL + WL)) : "memory");
            __builtin_amdgcn_s_barrier();
            issue(s + RING, sel);
            read(next, from ^ 1);
            __builtin_amdgcn_sched_barrier(0);                      // the reads leave before the products
            products(from);
            __builtin_amdgcn_sched_barrier(0);
            sel = next;
        };
        int s = 0;
        for (; s + 1 < full; s += 2) {
            step(s, 0);
            step(s + 1, 1);
        }
        if (s < full) step(s, 0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    if (full * STAGE < K) {                                         // depths beyond K are zero; a lane beyond K reads its row's first unit: a row may be shorter than a stage
        const ld_u32x4 zero = {0, 0, 0, 0};
        const bool in = full * STAGE + lu * UNIT < K;
        const int64_t k = in ? (int64_t)full * 128 : -(int64_t)lu * 16;
        auto last = [&](const char *base, uint32_t off) {
            const ld_u32x4 v = *(const ld_u32x4 *)(base + off + k);
            return __builtin_bit_cast(uint4, in ? v : zero);
        };
#pragma unroll
        for (int i = 0; i < XL; ++i) ldS[i * THREADS + tid] = last(xb, xo[i]);
#pragma unroll
        for (int i = 0; i < WL; ++i) ldS[(XL + i) * THREADS + tid] = last(wb, wo[i]);
        __syncthreads();
        read(0, 0);
        products(0);
    }
    if constexpr (GATED) {
        constexpr int HALF = COLS / 2;
        const int o = o0 + (wn * (TN / WN) + quad * COLS) / 2;
#pragma unroll
        for (int a = 0; a < XT; ++a) {
            const int n = n0 + wm * (TM / WM) + 16 * a + l16;
            if (n >= N || o >= O) continue;
            float v[HALF / 4][4];
#pragma unroll
            for (int e = 0; e < HALF; ++e) v[e >> 2][e & 3] = gated_unit_f<true>(acc[a][e >> 2][e & 3], acc[a][(HALF + e) >> 2][e & 3], unit.kind, unit.limit, unit.alpha, unit.shift);
            bf16_t *p = (bf16_t *)out + n * out_ld + o;
#pragma unroll
            for (int e = 0; e < HALF; e += 4) {
                if (O % 4 == 0 && out_ld % 4 == 0) { if (o + e < O) st4_f(p + e, v[e >> 2]); }
                else
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        if (o + e + y < O) st_f(p + e + y, v[e >> 2][y]);
            }
        }
        return;
    }
    const int o = o0 + wn * (TN / WN) + quad * COLS;                // this lane's COLS columns
    const bool whole = O % 8 == 0 && out_ld % 8 == 0, float_out = out_mode == JL_LINEAR_FLOAT || out_mode == JL_LINEAR_ROUNDED_FLOAT;
    float add[COLS];
#pragma unroll
    for (int e = 0; e < COLS; ++e) add[e] = bias && o + e < O ? ld_f(bias + o + e) : 0.f;
#pragma unroll
    for (int a = 0; a < XT; ++a) {
        const int n = n0 + wm * (TM / WM) + 16 * a + l16;
        if (n >= N) continue;
#pragma unroll
        for (int e0 = 0; e0 < COLS; e0 += 8) {
            if (o + e0 >= O) continue;
            float v[2][4];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e >> 2][e & 3] = acc[a][(e0 + e) >> 2][e & 3] + add[e0 + e];
            if (float_out) {
                float *p = (float *)out + n * out_ld + o + e0;
                if (out_mode == JL_LINEAR_ROUNDED_FLOAT)
#pragma unroll
                    for (int e = 0; e < 8; ++e) { bf16_t r; st_f(&r, v[e >> 2][e & 3]); v[e >> 2][e & 3] = ld_f(&r); }
                if (whole) { st4_f(p, v[0]); st4_f(p + 4, v[1]); }
                else
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (o + e0 + e < O) p[e] = v[e >> 2][e & 3];
                continue;
            }
            bf16_t *p = (bf16_t *)out + n * out_ld + o + e0;
            if (whole) {
                if (out_mode == JL_LINEAR_ADD) {
                    const ld_u32x4 r = *(const ld_u32x4 *)p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e >> 1][2 * (e & 1)] += __uint_as_float(r[e] << 16);
                        v[e >> 1][2 * (e & 1) + 1] += __uint_as_float(r[e] & 0xffff0000u);
                    }
                }
                typedef float f32x8 __attribute__((ext_vector_type(8)));
                const f32x8 all = {v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
                *(ls_bf16x8 *)p = __builtin_convertvector(all, ls_bf16x8);
            } else
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (o + e0 + e < O) st_f(p + e, v[e >> 2][e & 3] + (out_mode == JL_LINEAR_ADD ? ld_f(p + e) : 0.f));
        }
    }
}

// The largest tiles of which there is still about one per CU, since a CU takes in (TM + TN) rows for TM x TN sums: 64 x 64 up to 256 of them, 64 x 128, 128 x 128, and two of those per CU.
// us by 64 x 64 / 64 x 128 / 128 x 128 / two per CU: 1024 x 1024 by 1000 rows (256 of 64 x 64) 7.4 / 9.0 / 11.9 / 13.0, by 2048 (512) 10.6 / 9.9 / 12.9 / 13.5, 2048 x 2048 by 2048 (1024) 32 / 24.4 / 23.5 / 26.9, 1024 x 4096 by
// 2048 (2048) 33 / 27.3 / 27.6 / 23.2.
static int linear_mid_tiles(int64_t N, int64_t O) {
    auto tiles = [&](int tm, int tn) { return ((N + tm - 1) / tm) * ((O + tn - 1) / tn); };
    return tiles(64, 64) <= 256 ? 0 : tiles(64, 128) <= 256 ? 1 : tiles(128, 128) <= 256 ? 2 : 3;
}

// 1: where the launch is the better one; 2: there, and it was so for products that autocast does not see.  Tiles of 64 x 64; two of 128 x 128 per CU (linear_mid_tiles) lose to the library at depths beyond
// 1024, many tiles and very few at depths beyond 2048 (layer_ops.linear_mid has the figures).
extern "C" int jl_linear_mid_ok(int64_t N, int64_t K, int64_t O) {
    if (N <= 0 || K <= 0 || O <= 0) return 0;
    const int64_t tiles = ((N + 63) / 64) * ((O + 63) / 64);
    if ((K <= 1024 && tiles <= 512) || (K <= 2048 && tiles <= 256)) return 2;
    if (N > 2304 || K > 4096 || K * O > (int64_t)32 << 20) return 0;
    if (K > 2048) return N >= 300 && tiles >= 80 && tiles <= 256;
    return ((N + 127) / 128) * ((O + 127) / 128) <= (K <= 1024 ? 512 : 256);
}
template <int TM, int TN, int WM, int WN, int RING, bool GATED = false>
static int linear_mid_launch(const bf16_t *x, int64_t N, int64_t x_ld, const bf16_t *w, int32_t K, int32_t O, const bf16_t *bias, void *out, int64_t out_ld, int32_t out_mode, hipStream_t st, LinearUnit unit = {0, 0.f, 0.f, 0.f}) {
    const int64_t row_tiles = (N + TM - 1) / TM, cols = GATED ? TN / 2 : TN, tiles = row_tiles * ((O + cols - 1) / cols);
    if (tiles > INT32_MAX / (64 * WM * WN)) return jl_fail(JL_E_INVALID, "jl_linear_mid: too many tiles");
    constexpr int lds = (TM + TN) * 128 * RING;
    auto kern = linear_mid_kernel<TM, TN, WM, WN, RING, GATED>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_linear_mid: cannot get %d bytes of LDS: %s", lds, hipGetErrorString(e));
    }
    kern<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 64 * WM * WN, lds, st>>>(x, x_ld, w, bias, out, out_ld, (int)N, K, O, out_mode, (int)row_tiles, (int)tiles, unit);
    return jl_check_launch("linear_mid_kernel");
}
extern "C" int jl_linear_mid(const void *x, int dtype, int64_t N, int64_t x_ld, const void *w, int32_t K, int32_t O, const void *bias, void *out, int64_t out_ld, int32_t out_mode,
                             void *stream) {
    if (N <= 0 || O <= 0) return JL_OK;
    if (!x || !w || !out || K <= 0 || x_ld < K || out_ld < O) return jl_fail(JL_E_INVALID, "jl_linear_mid: null pointer or bad sizes");
    if (dtype != JL_BF16 || K % 8 || x_ld % 8 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15))
        return jl_fail(JL_E_INVALID, "jl_linear_mid: bfloat16, rows of x and W and the result at 16-byte borders");
    if (N > INT32_MAX / 64 || N * x_ld * 2 > UINT32_MAX || (int64_t)O * K * 2 > UINT32_MAX) return jl_fail(JL_E_INVALID, "jl_linear_mid: operands of up to 4 GB");
    if (out_mode < JL_LINEAR_SAME || out_mode > JL_LINEAR_ADD) return jl_fail(JL_E_INVALID, "jl_linear_mid: unknown out_mode");
    const bf16_t *xp = (const bf16_t *)x, *wp = (const bf16_t *)w, *bp = (const bf16_t *)bias;
    hipStream_t st = (hipStream_t)stream;
    switch (linear_mid_tiles(N, O)) {
    case 0: return linear_mid_launch<64, 64, 2, 2, 4>(xp, N, x_ld, wp, K, O, bp, out, out_ld, out_mode, st);
    case 1: return linear_mid_launch<64, 128, 2, 4, 3>(xp, N, x_ld, wp, K, O, bp, out, out_ld, out_mode, st);
    case 2: return linear_mid_launch<128, 128, 2, 4, 4>(xp, N, x_ld, wp, K, O, bp, out, out_ld, out_mode, st);
    }
    return linear_mid_launch<128, 128, 2, 2, 2>(xp, N, x_ld, wp, K, O, bp, out, out_ld, out_mode, st);
}
extern "C" int jl_linear_mid_gated(const void *x, int dtype, int64_t N, int64_t x_ld, const void *w, int32_t K, int32_t F, int32_t kind, float limit, float alpha, float shift, void *out, int64_t out_ld,
                                   void *stream) {
    if (N <= 0 || F <= 0) return JL_OK;
    if (!x || !w || !out || K <= 0 || x_ld < K || out_ld < F || F > INT32_MAX / 2 || kind < JL_ACT_GELU_TANH || kind > JL_ACT_GELU_ERF)
        return jl_fail(JL_E_INVALID, "jl_linear_mid_gated: null pointer, bad sizes or kind");
    if (dtype != JL_BF16 || K % 8 || x_ld % 8 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15))
        return jl_fail(JL_E_INVALID, "jl_linear_mid_gated: bfloat16, rows of x and W and the result at 16-byte borders");
    if (N > INT32_MAX / 64 || N * x_ld * 2 > UINT32_MAX || (int64_t)F * K * 4 > UINT32_MAX) return jl_fail(JL_E_INVALID, "jl_linear_mid_gated: operands of up to 4 GB");
    const bf16_t *xp = (const bf16_t *)x, *wp = (const bf16_t *)w;
    const LinearUnit unit = {kind, limit, alpha, shift};
    hipStream_t st = (hipStream_t)stream;
    switch (linear_mid_tiles(N, 2 * (int64_t)F)) {
    case 0: return linear_mid_launch<64, 64, 2, 2, 4, true>(xp, N, x_ld, wp, K, F, nullptr, out, out_ld, JL_LINEAR_SAME, st, unit);
    case 1: return linear_mid_launch<64, 128, 2, 4, 3, true>(xp, N, x_ld, wp, K, F, nullptr, out, out_ld, JL_LINEAR_SAME, st, unit);
    case 2: return linear_mid_launch<128, 128, 2, 4, 4, true>(xp, N, x_ld, wp, K, F, nullptr, out, out_ld, JL_LINEAR_SAME, st, unit);
    }
    return linear_mid_launch<128, 128, 2, 2, 2, true>(xp, N, x_ld, wp, K, F, nullptr, out, out_ld, JL_LINEAR_SAME, st, unit);
}

// ---- float products of many rows: TM of x by 128 of W per workgroup, on the bfloat16 matrix instructions in three terms per operand (jl_split.h) -----
// Eight wavefronts, so that two share a SIMD where a CU has one tile only: one wavefront issues vector instructions at half their rate and makes its terms while nobody multiplies (64 rows, one tile per
// CU, 1024 depths: 36 us with four, 27 with eight).  Large products reach 184 TFLOP/s, 1100 of the bfloat16 instructions, which is what a large bfloat16 product reaches here; smaller ones
// wait for their stages.  Error against 64 bits of 2553 x 1024 by 1024, 2-norm: 4.9e-7, the library's on the float instructions 5.7e-7 (of 4096 x 4096 by 4096 1.0e-6 / 1.15e-6).
template <int TM, int NW, int WM, int TKU>
__global__ __launch_bounds__(64 * NW, NW / 2) void linear_split_kernel(const float *__restrict__ x, int64_t x_ld, const float *__restrict__ w, const float *__restrict__ bias, float *__restrict__ out,
                                                              int64_t out_ld, int64_t N, int K, int O, int row_tiles, int tiles) {
    constexpr int WR = 128, XT = TM / WM / 32, WN = NW / WM, NT = WR / WN / 32;
    __shared__ uint4 smem[split_units(TM, WR, TKU)];
    // workgroups with the same remainder by 8 share an XCD: neighbouring tiles, which share W's rows
    const int per_xcd = (tiles + 7) / 8, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5, wm = wave / WN, wn = wave % WN;
    const int64_t n0 = (int64_t)(tile % row_tiles) * TM;
    const int o0 = tile / row_tiles * WR;
    auto x_at = [&](int m) { return x + (n0 + m < N ? n0 + m : N - 1) * x_ld; };
    auto w_at = [&](int j) { return w + (int64_t)(o0 + j < O ? o0 + j : O - 1) * K; };
    auto x_row = [&](int t) { return wm * (TM / WM) + 32 * t; };
    auto w_row = [&](int t) { return wn * (WR / WN) + 32 * t; };
    sp_f32x16 acc[XT][NT];
    split_products<TM, WR, NW, WM, TKU>(acc, smem, K, x_at, w_at, x_row, w_row);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int o = o0 + w_row(t) + l32;
        if (o >= O) continue;
        const float add = bias ? bias[o] : 0.f;
#pragma unroll
        for (int xt = 0; xt < XT; ++xt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t n = n0 + x_row(xt) + 8 * (r >> 2) + 4 * hi + (r & 3);
                if (n < N) out[n * out_ld + o] = acc[xt][t][r] + add;
            }
    }
}

// 128 rows per tile as soon as they give about half of the CUs one each.  us, 128 / 64 rows: 2553 x 1024 by 1100 (180 tiles of 128) 47 / 52, by 4096 139 / 150, 1500 x 768 by 1536 (144) 36 / 39;
// below, 512 x 1024 by 4096 (128) 51 / 36, 2553 x 512 by 768 (120) 26 / 18
static bool split_low(int64_t N, int64_t O) { return (N + 127) / 128 * ((O + 127) / 128) < 140; }

// The launch's time goes by rounds of 256 tiles, the library's, which has tiles of more heights and splits depths, more nearly by the product's size, so the line lies where a round is full enough: by the
// product's size in units of 64 x 128 against the tiles it is padded to.  us of GPU time, library / own: 2553 rows of 1024 by 1024 57 / 52, by 3072 135 / 100, 4096 of 4096 by 4096 948 / 747 (184 TFLOP/s; the
// float instructions reach 145), 2049 of 1028 by 1153 69 / 57, 1700 of 1024 by 1024 38 / 37, 128 of 1024 by 16384 39 / 36.  Beyond the line: padded rows, 96 of 1024 by 16384 30 / 35, 160 by 8192 28 / 33,
// 650 by 3072 41 / 53; rounds that have just begun, 513 of 1024 by 4096 49 / 52, 1290 by 3072 68 / 86, 2060 by 1024 49 / 54, 4100 of 2048 by 1024 149 / 160; one round of 64 rows at great depths, 1536
// of 4096 by 1024 111 / 115.  Up to depths of 320 both take 3 us more or less of the GPU, but the library's call 15 more of the host: from 192 tiles of 64 rows on.
extern "C" int jl_linear_split_ok(int64_t N, int64_t K, int64_t O) {
    if (N <= 0 || K <= 0 || O <= 0) return 0;
    const int64_t cols = (O + 127) / 128, tiles = (N + 63) / 64 * cols;
    if (K < 320) return tiles >= 192;
    const double size = (double)N * (double)O / (64 * 128);
    if (split_low(N, O)) return tiles >= 192 && tiles <= 256 && size >= 164 && size >= 0.8 * (double)tiles && (K < 2048 || size >= 200);
    const int64_t high = (N + 127) / 128 * cols, rounds = (high + 255) / 256;
    return rounds == 1 ? size > (high <= 200 ? 288 : 340) : size >= 330.0 * (double)rounds;
}

extern "C" int jl_linear_split(const float *x, int64_t N, int64_t x_ld, const float *w, int32_t K, int32_t O, const float *bias, float *out, int64_t out_ld, void *stream) {
    if (N <= 0 || O <= 0) return JL_OK;
    if (!x || !w || !out || K <= 0 || x_ld < K || out_ld < O) return jl_fail(JL_E_INVALID, "jl_linear_split: null pointer or bad sizes");
    if (K % 4 || x_ld % 4 || (((uintptr_t)x | (uintptr_t)w) & 15)) return jl_fail(JL_E_INVALID, "jl_linear_split: rows of x and W at 16-byte borders");
    const int64_t cols = ((int64_t)O + 127) / 128;
    const bool low = split_low(N, O);
    const int64_t row_tiles = low ? (N + 63) / 64 : (N + 127) / 128, tiles = row_tiles * cols;
    if (tiles > INT32_MAX / 512) return jl_fail(JL_E_INVALID, "jl_linear_split: too many tiles");
    (low ? linear_split_kernel<64, 8, 2, 8> : linear_split_kernel<128, 8, 2, 4>)<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 512, 0, (hipStream_t)stream>>>(x, x_ld, w, bias, out, out_ld, N, K, O,
                                                                                                                                                       (int)row_tiles, (int)tiles);
    return jl_check_launch("linear_split_kernel");
}

extern "C" int jl_linear_small(const void *x, int dtype, int64_t N, int64_t x_ld, const void *w, int w_dtype, int32_t K, int32_t O, const void *bias, void *out, int64_t out_ld,
                               int32_t out_mode, void *stream) {
    if (N <= 0 || O <= 0) return JL_OK;
    if (!x || !w || !out || K <= 0 || x_ld < K || out_ld < O) return jl_fail(JL_E_INVALID, "jl_linear_small: null pointer or bad sizes");
    if ((dtype != JL_BF16 && dtype != JL_F32) || (w_dtype != dtype && w_dtype != JL_F32)) return jl_fail(JL_E_INVALID, "jl_linear_small: W of x's type, or float");
    const int x_unit = dtype == JL_BF16 ? 8 : 4, w_unit = w_dtype == JL_BF16 ? 8 : 4;
    if (N > JL_LINEAR_SMALL_ROWS || K % w_unit || x_ld % x_unit || (((uintptr_t)x | (uintptr_t)w) & 15))
        return jl_fail(JL_E_INVALID, "jl_linear_small: up to %d rows, rows of x and W at 16-byte borders", JL_LINEAR_SMALL_ROWS);
    if (out_mode < JL_LINEAR_SAME || out_mode > JL_LINEAR_ROUNDED_FLOAT) return jl_fail(JL_E_INVALID, "jl_linear_small: unknown out_mode");
#define LS_TYPES(TX, T)                                                                                                                        \
    do {                                                                                                                                       \
        if (N <= 16) linear_small_launch<TX, T, 1>(x, x_ld, w, bias, out, out_ld, (int)N, K, O, out_mode, (hipStream_t)stream);                 \
        else if (N <= 32) linear_small_launch<TX, T, 2>(x, x_ld, w, bias, out, out_ld, (int)N, K, O, out_mode, (hipStream_t)stream);            \
        else linear_small_launch<TX, T, 4>(x, x_ld, w, bias, out, out_ld, (int)N, K, O, out_mode, (hipStream_t)stream);                         \
    } while (0)
    if (dtype == JL_F32) LS_TYPES(float, float);
    else if (w_dtype == JL_F32) LS_TYPES(bf16_t, float);
    else LS_TYPES(bf16_t, bf16_t);
#undef LS_TYPES
    return jl_check_launch("linear_small_kernel");
}
