// jl_scan.hip — linear recurrence with one decay per head (and token): S_t = a_t S_(t-1) + k_t (u_t v_t)^T, o_t = S_t^T q_t + skip v_t.
// Fixed decays are lightning attention, decays and step sizes from a projection (u = softplus, a = exp(-exp(A_log) u)) are the state-space
// duality of Mamba-2; one float state [D, Dv] per (request slot, head).
#include "jl_common.h"
#include <type_traits>

// ---- token by token: decoded tokens, short portions, float activations ----------------------------------------------------------------------
// The columns of S never interact, so a workgroup is ONE wavefront that owns 32 columns of one head's state (grid.y walks the head's
// columns): two adjacent lanes per column, each with DMAX / 2 consecutive rows in registers.  Rows of S are read and written as 128
// consecutive bytes.  Eight tokens at a time go through LDS; the next group's inputs travel while the current one is worked on.
constexpr int SC_TT = 8, SC_COLS = 32, SC_TOKEN_COLS = 16, SC_TOKEN_HEADS = 2048;
// silu in the activations' dtype: both forms of the recurrence see the same q, k and v, however a prompt is cut
template <typename T> __device__ __forceinline__ float silu_as(float z) {
    T t;
    st_f(&t, silu_f(z));
    return ld_f(&t);
}

template <typename T, int DMAX>
__global__ __launch_bounds__(64) void scan_kernel(jl_scan_args a) {
    constexpr int DPER = DMAX / 2, PRE = SC_TT * DMAX / 64, ROW = DMAX + 8;
    __shared__ __attribute__((aligned(16))) float qs[SC_TT * ROW], ks[SC_TT * ROW];
    __shared__ float as[SC_TT], us[SC_TT];
    auto at = [](int tt, int d) { return tt * ROW + d + (d / DPER) * 4; };      // the two lanes of a column read different banks
    const int H = a.H, D = a.D, Dv = a.Dv;
    const int b = blockIdx.x / H, h = blockIdx.x - b * H, kh = h / (H / a.G);
    const int row0 = a.seq[4 * b], cnt = a.seq[4 * b + 1], pos0 = a.seq[4 * b + 2], slot = a.seq[4 * b + 3];
    if (cnt <= 0) return;
    const int lane = threadIdx.x, j = (blockIdx.z * gridDim.y + blockIdx.y) * SC_COLS + (lane >> 1), sub = lane & 1, d0 = sub * DPER;
    const bool live = j < Dv;
    const T *src = (const T *)a.src, *dtp = (const T *)a.dt;
    const bool fixed = a.decay != nullptr, act = a.act == JL_ACT_SILU;
    const float gamma = fixed ? a.decay[h] : 0.f, rate = fixed ? 0.f : -expf(a.A_log[h]), bias = fixed ? 0.f : a.dt_bias[h];
    const float skip = a.skip ? a.skip[h] : 0.f;
    float *sp = a.state + ((int64_t)slot * H + h) * D * Dv;
    float S[DPER];
#pragma unroll
    for (int i = 0; i < DPER; ++i) S[i] = (live && d0 + i < D && pos0 > 0) ? sp[(int64_t)(d0 + i) * Dv + j] : 0.f;
    float pq[PRE], pk[PRE], pv[SC_TT], pd = 0.f;
    auto fetch = [&](int t0) {
        const int nt = cnt - t0 < SC_TT ? cnt - t0 : SC_TT;
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int e = i * 64 + lane, tt = e / DMAX, d = e - tt * DMAX;
            pq[i] = pk[i] = 0.f;
            if (tt < nt && d < D) {
                const T *row = src + (int64_t)(row0 + t0 + tt) * a.ld + kh * D + d;
                pq[i] = ld_f(row + a.q_col);
                pk[i] = ld_f(row + a.k_col);
            }
        }
#pragma unroll
        for (int tt = 0; tt < SC_TT; ++tt) pv[tt] = (tt < nt && live) ? ld_f(src + (int64_t)(row0 + t0 + tt) * a.ld + a.v_col + (int64_t)h * Dv + j) : 0.f;
        if (!fixed && lane < nt) pd = ld_f(dtp + (int64_t)(row0 + t0 + lane) * a.dt_ld + a.dt_col + h);
    };
    fetch(0);
    for (int t0 = 0; t0 < cnt; t0 += SC_TT) {
        const int nt = cnt - t0 < SC_TT ? cnt - t0 : SC_TT;
        __syncthreads();                                        // the group before has been read
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int e = i * 64 + lane, tt = e / DMAX, d = e - tt * DMAX;
            if (tt < nt) {
                qs[at(tt, d)] = act ? silu_as<T>(pq[i]) : pq[i];
                ks[at(tt, d)] = act ? silu_as<T>(pk[i]) : pk[i];
            }
        }
        if (lane < nt) {
            const float u = fixed ? 1.0f : softplus_f(pd + bias);
            us[lane] = u;
            as[lane] = fixed ? gamma : expf(rate * u);
        }
        float v[SC_TT];
#pragma unroll
        for (int tt = 0; tt < SC_TT; ++tt) v[tt] = act ? silu_as<T>(pv[tt]) : pv[tt];
        __syncthreads();
        if (t0 + SC_TT < cnt) fetch(t0 + SC_TT);                // in flight while this group's steps run
#pragma unroll
        for (int tt = 0; tt < SC_TT; ++tt) {
            if (tt < nt) {
                const float *qp = qs + tt * ROW + d0 + sub * 4, *kp = ks + tt * ROW + d0 + sub * 4;
                const float g = as[tt], u = us[tt] * v[tt];
                float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < DPER; i += 4) {
                    const float4 k4 = *(const float4 *)(kp + i), q4 = *(const float4 *)(qp + i);
                    S[i] = g * S[i] + k4.x * u;             acc[0] += S[i] * q4.x;
                    S[i + 1] = g * S[i + 1] + k4.y * u;     acc[1] += S[i + 1] * q4.y;
                    S[i + 2] = g * S[i + 2] + k4.z * u;     acc[2] += S[i + 2] * q4.z;
                    S[i + 3] = g * S[i + 3] + k4.w * u;     acc[3] += S[i + 3] * q4.w;
                }
                float o = (acc[0] + acc[1]) + (acc[2] + acc[3]);
                o += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o), 0xB1, 0xF, 0xF, true));      // quad_perm [1, 0, 3, 2]: the column's other lane
                if (live && sub == 0) a.out[(int64_t)(row0 + t0 + tt) * ((int64_t)H * Dv) + (int64_t)h * Dv + j] = o + skip * v[tt];
            }
        }
    }
    if (live)
#pragma unroll
        for (int i = 0; i < DPER; ++i)
            if (d0 + i < D) sp[(int64_t)(d0 + i) * Dv + j] = S[i];
}

// ---- a decoding step: one token for each request -----------------------------------------------------------------------------------------------
// A token has nothing to walk: what the wavefronts above spend is two lanes' walk through half a column each, 64 dependent sums in a row behind 64 loads, in one wavefront per CU.  Here a workgroup takes
// 16 columns, four per thread in one 16-byte access, and its 64 groups of four threads D / 64 rows each, all on their way at once; the column's sum goes through shuffles and LDS.
// us a launch, wavefronts of two lanes a column / so (bfloat16, D and Dv 128 but as said): 1 request of 8 heads 10.0 / 4.2, 8 10.5 / 5.2, 32 of 16 heads 23.2 / 18.2, 48 32.9 / 28.9, of 64 x 64 11.4 / 10.8, 32 of 8 of 256 x 256 48.7 / 32.6.
template <typename T, int R>
__global__ __launch_bounds__(256) void scan_token_kernel(jl_scan_args a) {
    __shared__ float part[4][16];
    const int H = a.H, D = a.D, Dv = a.Dv;
    const int b = blockIdx.x / H, h = blockIdx.x - b * H, kh = h / (H / a.G);
    const int row0 = a.seq[4 * b], cnt = a.seq[4 * b + 1], pos0 = a.seq[4 * b + 2], slot = a.seq[4 * b + 3];
    if (cnt <= 0) return;
    const int tid = threadIdx.x, c = tid & 3, d0 = tid >> 2, j = (blockIdx.z * gridDim.y + blockIdx.y) * SC_TOKEN_COLS + 4 * c;
    const bool live = j < Dv, fixed = a.decay != nullptr, act = a.act == JL_ACT_SILU;
    float *sp = a.state + ((int64_t)slot * H + h) * D * Dv;
    float S[R][4];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        S[i][0] = S[i][1] = S[i][2] = S[i][3] = 0.f;
        if (live && d0 + 64 * i < D && pos0 > 0) ld4_f(sp + (int64_t)(d0 + 64 * i) * Dv + j, S[i]);
    }
    const float gamma = fixed ? a.decay[h] : 0.f, rate = fixed ? 0.f : -expf(a.A_log[h]), bias = fixed ? 0.f : a.dt_bias[h], skip = a.skip ? a.skip[h] : 0.f;
    for (int t = 0; t < cnt; ++t) {                             // (a request of several tokens beside others of none)
        const T *row = (const T *)a.src + (int64_t)(row0 + t) * a.ld, *qp = row + a.q_col + kh * D, *kp = row + a.k_col + kh * D, *vp = row + a.v_col + (int64_t)h * Dv + j;
        float q[R], k[R], v[4], acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const bool in = d0 + 64 * i < D;
            q[i] = in ? ld_f(qp + d0 + 64 * i) : 0.f;
            k[i] = in ? ld_f(kp + d0 + 64 * i) : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = live ? ld_f(vp + e) : 0.f;
        const float u = fixed ? 1.0f : softplus_f(ld_f((const T *)a.dt + (int64_t)(row0 + t) * a.dt_ld + a.dt_col + h) + bias), g = fixed ? gamma : expf(rate * u);
        if (act) {
#pragma unroll
            for (int i = 0; i < R; ++i) { q[i] = silu_as<T>(q[i]); k[i] = silu_as<T>(k[i]); }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = silu_as<T>(v[e]);
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (d0 + 64 * i < D)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    S[i][e] = g * S[i][e] + k[i] * (u * v[e]);
                    acc[e] += S[i][e] * q[i];
                }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int x = 4; x < 64; x *= 2) acc[e] += __shfl_xor(acc[e], x);
        __syncthreads();                                        // the token before has been read
        if ((tid & 63) < 4)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[tid >> 6][4 * c + e] = acc[e];
        __syncthreads();
        if (tid < 4 && live) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (part[0][4 * c + e] + part[1][4 * c + e]) + (part[2][4 * c + e] + part[3][4 * c + e]) + skip * v[e];
            st4_f(a.out + (int64_t)(row0 + t) * ((int64_t)H * Dv) + (int64_t)h * Dv + j, o);
        }
    }
    if (live)
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (d0 + 64 * i < D) st4_f(sp + (int64_t)(d0 + 64 * i) * Dv + j, S[i]);
}

template <typename T> static int scan_launch(const jl_scan_args &a, hipStream_t st) {
    // no more tokens than requests: a token each (or none); rows of the state and of the result at 16-byte borders; and up to 2048 heads, since beyond that the wavefronts' 128 bytes of a row in one access
    // read memory a little better than these 64 (200 requests of 16 heads of 128 x 128 133.4 / 135.5 us)
    if (a.N > 0 && a.N <= a.B && (int64_t)a.B * a.H <= SC_TOKEN_HEADS && a.Dv % 4 == 0 && (((uintptr_t)a.state | (uintptr_t)a.out) & 15) == 0) {
        const unsigned cols = (unsigned)((a.Dv + SC_TOKEN_COLS - 1) / SC_TOKEN_COLS), y = cols < 65535 ? cols : 65535;
        const dim3 grid((unsigned)(a.B * a.H), y, (cols + y - 1) / y);
        if (a.D <= 64) scan_token_kernel<T, 1><<<grid, 256, 0, st>>>(a);
        else if (a.D <= 128) scan_token_kernel<T, 2><<<grid, 256, 0, st>>>(a);
        else scan_token_kernel<T, 4><<<grid, 256, 0, st>>>(a);
        return jl_check_launch("scan_token_kernel");
    }
    const unsigned cols = (unsigned)((a.Dv + SC_COLS - 1) / SC_COLS), y = cols < 65535 ? cols : 65535;      // (a launch's second dimension ends there)
    const dim3 grid((unsigned)(a.B * a.H), y, (cols + y - 1) / y);
    if (a.D <= 32) scan_kernel<T, 32><<<grid, 64, 0, st>>>(a);
    else if (a.D <= 64) scan_kernel<T, 64><<<grid, 64, 0, st>>>(a);
    else if (a.D <= 128) scan_kernel<T, 128><<<grid, 64, 0, st>>>(a);
    else scan_kernel<T, 256><<<grid, 64, 0, st>>>(a);
    return jl_check_launch("scan_kernel");
}

// ---- long portions on the matrix cores (bfloat16): pieces side by side, 64 tokens at a time --------------------------------------------------
// With L_t the running sum of log a inside a group of 64 tokens (kept to base 2), the recurrence of the group is three products:
//   o_i = exp(L_i) S^T q_i + sum_{j <= i} (q_i . k_j) exp(L_i - L_j) u_j v_j,        S <- exp(L_end) S + sum_j k_j (exp(L_end - L_j) u_j v_j)^T.
// A request's portion is cut into pieces (whole groups, except the last) that run side by side in three launches: every piece's own
// contribution to the state from a zero state (CH_LOCAL, not for a request's last piece), scan_join_kernel (the state every piece starts
// from), outputs (CH_OUT; the last piece leaves the request's final state in its slot).  Where every request has one piece, in one: it starts from the slot (one portion of 64 tokens, 16 heads of
// 128 x 128: 20 -> 16 us, 16 of 100 67 -> 33).
// q, k and v enter the products as bfloat16 (what the projection, the convolution and their activation give); everything else stays float
// and crosses the matrix cores as the sum of THREE bfloat16 numbers, which hold all 24 bits of it: the state, the decayed weights of a pair,
// the decayed values.
// A wavefront keeps 32 columns of one head's state, all rows of it, in accumulators and needs nothing from the others but the rows of q, k and v, which they share in
// LDS: heads that read the same q and k sit in one workgroup (``heads`` of them, NW wavefronts).  Accumulator r of lane l of a 32 x 32 product is row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32; lane l supplies row (A) or column (B) l % 32 with eight depths of a 16-deep step, and which depths these are is free as
// long as both operands agree.  So registers 8s .. 8s + 7 of an accumulator are handed on as an operand over the depths 16s + 4 (l / 32) + {0 .. 3, 8 .. 11}: the state as B of
// S^T q, the weights of the pairs (formed turned, K Q^T) as A of the sum over values, without a trip through LDS.  q and k rows are read in that order as two 8-byte halves; k and v are
// turned by ds_read_b64_tr_b16, and the values' operand, scaled and split in registers, is the state's update too.  One staging of rows and two barriers per group are left.
// What bounds it: latency with two wavefronts per SIMD, all that their registers allow.  Per group and wavefront 1 900 vector instructions (splits, exponentials, silu) and 138 products of 32 cycles
// take 12 000 cycles of issue; two side by side take 40 000.  Loads, stores, splits, weights: leaving out any one of them gives 5 to 15 % of the time.
// Before, 64 columns of one head per workgroup met in LDS five times per group, one workgroup per CU.  us of the three launches, 4 x 2048 tokens, before / now: 16 heads of 128 x 128 with silu
// 212 / 121 (their bytes at the rate of a large copy: 78), 32 heads of 128 x 64 over one key head 201 / 116; 3 x 1000 of 8 heads 74 / 54, 8 x 200 of 16 heads 90 / 47; but one portion of 256 of
// 16 heads 31 / 33: a group alone takes its wavefront 9 us, and three launches' ends show.
typedef __bf16 ch_bf16x4 __attribute__((ext_vector_type(4)));
typedef float ch_f32x4 __attribute__((ext_vector_type(4)));
typedef float ch_f32x16 __attribute__((ext_vector_type(16)));
typedef short ch_s16x4 __attribute__((ext_vector_type(4)));
typedef short ch_s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) ch_s16x4 ch_lds_s16x4;
constexpr int CH_T = 64, CH_TERMS = JL_SPLIT_TERMS, CH_OUT = 0, CH_LOCAL = 1;

__device__ __forceinline__ uint2 ch_silu4(uint2 w) {
    float v[4] = {__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= __builtin_amdgcn_rcpf(1.0f + __expf(-v[i]));          // rounded to bfloat16 next
    const ch_f32x4 f = {v[0], v[1], v[2], v[3]};
    return __builtin_bit_cast(uint2, __builtin_convertvector(f, ch_bf16x4));
}

static constexpr size_t ch_lds_bytes(int DP, int NW, bool out) { return 2 * CH_T * ((out ? 2 : 1) * (size_t)(DP + 8) + 32 * NW + 16) + NW * 4 * CH_T * 4 + (out ? (NW * 32 + 2) * 4 : 0); }

template <int DP, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW == 2 && DP > 64 ? 1 : 2) void scan_chunk_kernel(jl_scan_args a, int heads, int blocks, int alone) {      // alone: every request has one piece
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr bool OUT = MODE == CH_OUT;
    constexpr int THREADS = 64 * NW, QROW = DP + 8, VROW = 32 * NW + 16, UD = DP <= 32 ? 8 : DP <= 64 ? 16 : 32, UV = 8 * NW, NT = DP / 32;
    constexpr int KSTEP = THREADS / UD, KIT = CH_T / KSTEP, VSTEP = THREADS / UV, VIT = CH_T / VSTEP;      // rows the workgroup takes at once, and how often
    const int D = a.D, Dv = a.Dv, H = a.H;
    const int sharing = H / a.G, per_key = (sharing + heads - 1) / heads;                    // heads that read the same q and k, and their workgroups
    const int piece = blockIdx.x, kh = blockIdx.y / per_key, first = (blockIdx.y % per_key) * heads, h0 = kh * sharing + first;
    if (sharing - first < heads) heads = sharing - first;
    const int row0 = a.chunk_rec[4 * piece], cnt = a.chunk_rec[4 * piece + 1], slot = a.chunk_rec[4 * piece + 2], last = a.chunk_rec[4 * piece + 3];
    if (cnt <= 0 || (!OUT && last)) return;
    bf16_t *Ks = (bf16_t *)smem, *Vs = Ks + CH_T * QROW, *Qs = Vs + CH_T * VROW;             // [64][DP + 8] keys, [64][32 NW + 16] values, [64][DP + 8] queries
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    float *tables = (float *)(Vs + CH_T * VROW + (OUT ? CH_T * QROW : 0));
    float *Ls = tables + wave * 4 * CH_T;                                                    // this wavefront's: [64] running log2 decay
    float *us = Ls + CH_T, *es = us + CH_T, *el = es + CH_T;                                 // [64] u; exp(L_end - L) u; exp(L)
    int *brokenS = (int *)(tables + NW * 4 * CH_T) + wave * 32;                              // [32] the first token of a group whose value is not finite, per column (outputs only)
    int *flawS = (int *)(tables + NW * 4 * CH_T) + NW * 32;                                  // [2] whether this group, the one before, has such a value
    // the columns of wavefront w: block w % blocks (of those from blockIdx.z * NW on) of head h0 + w / blocks
    auto head_of = [&](int w) { return h0 + w / blocks; };
    auto col_of = [&](int w) { return 32 * ((int)blockIdx.z * NW + w % blocks); };
    const int h = head_of(wave), c_base = col_of(wave), sc = c_base + l32;
    const bool busy = wave < heads * blocks && c_base < Dv;
    const bf16_t *src = (const bf16_t *)a.src, *dtp = (const bf16_t *)a.dt;
    const bool fixed = a.decay != nullptr, act = a.act == JL_ACT_SILU;
    const float glog = fixed && busy ? fmaxf(log2f(a.decay[h]), -1e30f) : 0.f, rate = fixed || !busy ? 0.f : (float)(-1.4426950408889634 * exp((double)a.A_log[h])), bias = fixed || !busy ? 0.f : a.dt_bias[h];
    const float skip = a.skip && busy ? a.skip[h] : 0.f;

    ch_f32x16 S[NT];                                                // rows 32 x .. 32 x + 31 of the wavefront's columns
    // registers become f(row, byte offset in the state, register): one address that moves on, not sixty-four in registers
    auto each_state = [&](auto &&f) {
        uint32_t off = (uint32_t)(4 * hi * Dv + sc) * 4;
#pragma unroll
        for (int x = 0; x < NT; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                asm volatile("" : "+v"(off));
                S[x][r] = f(32 * x + 8 * (r >> 2) + 4 * hi + (r & 3), off, S[x][r]);
                off += ((r & 3) == 3 ? 5 : 1) * Dv * 4;
            }
    };
#pragma unroll
    for (int x = 0; x < NT; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[x][r] = 0.f;
    bool started = OUT && busy && sc < Dv;
    if (started) {
        const char *sp = (const char *)(a.scratch + ((int64_t)piece * H + h) * D * Dv);
        if (alone) {                                                // from its slot, as there is nothing to join
            int b = piece;
            if (a.req[4 * b] != piece)
                for (b = 0; b + 1 < a.B && a.req[4 * b] != piece;) ++b;
            started = a.req[4 * b + 2] > 0;
            sp = (const char *)(a.state + ((int64_t)slot * H + h) * D * Dv);
        }
        if (started) each_state([&](int d, uint32_t off, float) { return d < D ? *(const float *)(sp + off) : 0.f; });
    }
    uint2 rq[OUT ? KIT : 1], rk[KIT], rv[VIT];
    float rd = 0.f;
    // this thread's unit of four values: of q and k, of v (`w`: whose columns); what does not exist is staged as zeros
    const int kt = tid / UD, kd = (tid % UD) * 4, vt = tid / UV, vc = (tid % UV) * 4, vw = vc >> 5, vcol = col_of(vw) + (vc & 31);
    const bool k_in = kd < D, v_in = vw < heads * blocks && vcol < Dv;
    const uint32_t k_off = k_in ? (uint32_t)(kt * a.ld + kd) : 0u, v_off = v_in ? (uint32_t)(vt * a.ld + (int64_t)(vw / blocks) * Dv + vcol) : 0u;
    auto fetch = [&](int t0) {                                      // rows beyond the portion repeat its last and are cleared on the way to LDS
        const int nt = cnt - t0;
        const bf16_t *base = src + (int64_t)(row0 + t0) * a.ld, *kb = base + a.k_col + kh * D, *qb = base + a.q_col + kh * D, *vb = base + a.v_col + (int64_t)h0 * Dv;
        if (nt >= CH_T) {
#pragma unroll
            for (int it = 0; it < KIT; ++it) {
                rk[it] = *(const uint2 *)(kb + it * KSTEP * a.ld + k_off);
                if (OUT) rq[OUT ? it : 0] = *(const uint2 *)(qb + it * KSTEP * a.ld + k_off);
            }
#pragma unroll
            for (int it = 0; it < VIT; ++it) rv[it] = *(const uint2 *)(vb + it * VSTEP * a.ld + v_off);
        } else {
#pragma unroll
            for (int it = 0; it < KIT; ++it) {
                const int t = kt + it * KSTEP < nt ? kt + it * KSTEP : nt - 1;
                const int64_t o = k_in ? t * a.ld + kd : 0;
                rk[it] = *(const uint2 *)(kb + o);
                if (OUT) rq[OUT ? it : 0] = *(const uint2 *)(qb + o);
            }
#pragma unroll
            for (int it = 0; it < VIT; ++it) {
                const int t = vt + it * VSTEP < nt ? vt + it * VSTEP : nt - 1;
                rv[it] = *(const uint2 *)(vb + (v_in ? t * a.ld + (int64_t)(vw / blocks) * Dv + vcol : 0));
            }
        }
        if (!fixed && busy) rd = lane < nt ? ld_f(dtp + (int64_t)(row0 + t0 + lane) * a.dt_ld + a.dt_col + h) : 0.f;
    };
    // turned operands: column (or row) l % 32 of 32 columns from c on, tokens 16 s + 4 hi + {0 .. 3, 8 .. 11}
    const int tr_row = 4 * hi + ((lane & 15) >> 2), tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto turned = [&](const bf16_t *tile, int row_len, int c, int s) {
        ch_s16x4 half[2];
#pragma unroll
        for (int y = 0; y < 2; ++y) half[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ch_lds_s16x4 *)(tile + (16 * s + 8 * y + tr_row) * row_len + c + tr_col));
        return __builtin_bit_cast(jl_bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto row_of = [&](const bf16_t *tile, int t, int s) {           // row t, depths 16 s + 4 hi + {0 .. 3, 8 .. 11}
        const ch_bf16x4 x = *(const ch_bf16x4 *)(tile + t * QROW + 16 * s + 4 * hi), y = *(const ch_bf16x4 *)(tile + t * QROW + 16 * s + 8 + 4 * hi);
        return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto acc8 = [](const ch_f32x16 &v, int s) {
        jl_f32x8 f;
#pragma unroll
        for (int x = 0; x < 8; ++x) f[x] = v[8 * s + x];
        return f;
    };
    // The outputs of a group leave behind the next group's barrier and the loads of the one after it: loads and stores share a counter, and the wait for those loads, a group
    // later, finds the stores done too.
    ch_f32x16 o[OUT ? 2 : 1];                                       // outputs of queries 0 .. 31, 32 ..
    auto outputs = [&](int t0, int n) {
        const int64_t o_ld = (int64_t)H * Dv;
        char *to = (char *)(a.out + (row0 + t0) * o_ld + (int64_t)h * Dv + c_base);
        const uint32_t o_row = (uint32_t)o_ld * 4;                  // (ch_in_reach)
        uint32_t off = 4 * hi * o_row + 4 * l32;
        auto store = [&](auto whole) {
#pragma unroll
            for (int y = 0; y < (OUT ? 2 : 0); ++y)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    asm volatile("" : "+v"(off));                   // one address that moves on, not thirty-two in registers
                    if (decltype(whole)::value || 32 * y + 8 * (r >> 2) + 4 * hi + (r & 3) < n) *(float *)(to + off) = o[y][r];
                    off += (r & 3) == 3 ? 5 * o_row : o_row;
                }
        };
        if (!busy || sc >= Dv) return;
        if (n >= CH_T) store(std::true_type());
        else store(std::false_type());
    };
    if (OUT && tid < 2) flawS[tid] = 0;
    fetch(0);
    float l_all = 0.f, end = 0.f, g = 1.f;                          // log2 of the piece's decay up to here, of the group's; the group's decay (fixed decays: the same for whole groups)
    for (int t0 = 0; t0 < cnt; t0 += CH_T) {
        const int nt = cnt - t0 < CH_T ? cnt - t0 : CH_T;
        __syncthreads();                                            // the group before has been read
        float zero = 0.f;                                           // not a number with a value that is not finite
        auto stage = [&](auto silu) {                               // silu(0) = 0
            auto put = [&](bf16_t *to, uint2 v, bool in) {
                if (!in) v = make_uint2(0, 0);
                if (decltype(silu)::value) v = ch_silu4(v);
                *(uint2 *)to = v;
                return v;
            };
            if (DP == 4 * UD || kd < DP)
#pragma unroll
                for (int it = 0; it < KIT; ++it) {
                    const int t = kt + it * KSTEP;
                    put(Ks + t * QROW + kd, rk[it], k_in && t < nt);
                    if (OUT) put(Qs + t * QROW + kd, rq[OUT ? it : 0], k_in && t < nt);
                }
#pragma unroll
            for (int it = 0; it < VIT; ++it) {
                const uint2 v = put(Vs + (vt + it * VSTEP) * VROW + vc, rv[it], v_in && vt + it * VSTEP < nt);
                if (!OUT) continue;
                zero = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(jl_bf16x2, v.x), jl_bf16x2{0, 0}, zero, false);
                zero = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(jl_bf16x2, v.y), jl_bf16x2{0, 0}, zero, false);
            }
            if (OUT && zero != 0.f) flawS[t0 / CH_T & 1] = 1;
        };
        if (act) stage(std::true_type());
        else stage(std::false_type());
        if (busy && (!fixed || t0 == 0 || nt < CH_T)) {             // a token per lane: step size, running log2 decay
            const bool in = lane < nt;
            const float u = !in ? 0.f : fixed ? 1.0f : softplus_f(rd + bias);
            double l = !in ? 0. : fixed ? (double)glog : (double)rate * u;      // far into a group with strong decays a sum in float would be off by more than the tokens' own decays
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const double y = __shfl_up(l, off, 64);
                if (lane >= off) l += y;
            }
            const double whole = __shfl(l, 63, 64);
            end = (float)whole;
            es[lane] = exp2f((float)(whole - l)) * u;
            if (OUT) {
                Ls[lane] = (float)l;
                us[lane] = u;
                el[lane] = exp2f((float)l);
            }
            g = exp2f(end);
        }
        l_all += end;
        __syncthreads();
        // Weights of zero must not meet a value that is not finite, in front of whose token they stand: it is left out of the products, and its column's outputs from its token on
        // and the column of the state are set behind them
        bool flawed = false;
        if (OUT) {
            flawed = __builtin_amdgcn_readfirstlane(flawS[t0 / CH_T & 1]);
            if (tid == 0) flawS[~(t0 / CH_T) & 1] = 0;
            if (flawed) {
                int broken = CH_T, here = l32;
                asm volatile("" : "+v"(here));                      // its addresses made here, not kept over the loop
#pragma unroll 1
                for (int s = 0; s < CH_T / 16; ++s) {
                    const jl_bf16x8 v = turned(Vs, VROW, 32 * wave, s);
#pragma unroll
                    for (int i = 7; i >= 0; --i)
                        if (!__builtin_isfinite((float)v[i])) {
                            const int t = 16 * s + 4 * hi + i + 4 * (i >> 2);
                            broken = min(broken, t);
                            Vs[t * VROW + 32 * wave + here] = (bf16_t)0;
                        }
                }
                broken = min(broken, __shfl_xor(broken, 32, 64));
                brokenS[here] = broken;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (t0 + CH_T < cnt) fetch(t0 + CH_T);                      // in flight while this group is multiplied
        if (OUT && t0 > 0) outputs(t0 - CH_T, CH_T);
        jl_bf16x8 vf[CH_T / 16];
        const bool more = !OUT || last || t0 + CH_T < cnt;          // else nobody reads this piece's final state: the next piece has its own
        if (busy) {
            if (OUT) {
                // A step's operands (rows from LDS, splits) are made while the step before is multiplied, and no sooner (sched_barrier): all at once they do not fit the registers.
                constexpr int KS = DP / 16;
#pragma unroll
                for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = 0.f;
                {
                    jl_bf16x8 q[2][2], part[2][CH_TERMS];
                    auto operands = [&](int s) {
                        q[s & 1][0] = row_of(Qs, l32, s);
                        q[s & 1][1] = row_of(Qs, 32 + l32, s);
                        jl_split8(acc8(S[s >> 1], s & 1), part[s & 1]);
                    };
                    operands(0);
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        if (s + 1 < KS) operands(s + 1);
#pragma unroll
                        for (int x = 0; x < CH_TERMS; ++x)
#pragma unroll
                            for (int y = 0; y < 2; ++y) o[y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(q[s & 1][y], part[s & 1][x], o[y], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                ch_f32x16 p[3];                                     // turned weights: keys 0 .. of queries 0 .., keys 0 .. of queries 32 .., keys 32 .. of queries 32 ..
#pragma unroll
                for (int r = 0; r < 16; ++r) p[0][r] = p[1][r] = p[2][r] = 0.f;
                {
                    jl_bf16x8 f[2][4];
                    auto operands = [&](int s) {
                        f[s & 1][0] = row_of(Qs, l32, s); f[s & 1][1] = row_of(Qs, 32 + l32, s); f[s & 1][2] = row_of(Ks, l32, s); f[s & 1][3] = row_of(Ks, 32 + l32, s);
                    };
                    operands(0);
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        if (s + 1 < KS) operands(s + 1);
                        p[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s & 1][2], f[s & 1][0], p[0], 0, 0, 0);
                        p[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s & 1][2], f[s & 1][1], p[1], 0, 0, 0);
                        p[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s & 1][3], f[s & 1][1], p[2], 0, 0, 0);
                        if (s < 2) {                                // beside the products: what S^T q is worth now
#pragma unroll
                            for (int x = 0; x < 4; ++x) {
                                const ch_f32x4 e4 = *(const ch_f32x4 *)(el + 32 * s + 8 * x + 4 * hi);
#pragma unroll
                                for (int i = 0; i < 4; ++i) o[s][4 * x + i] *= e4[i];
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (int s = 0; s < CH_T / 16; ++s) vf[s] = turned(Vs, VROW, 32 * wave, s);
                {
                    jl_bf16x8 part[2][CH_TERMS];
                    const float li[2] = {Ls[l32], Ls[32 + l32]};
                    int ahead = l32 - 4 * hi;                       // the query's place less the lane's first key's, in a block on the diagonal
                    asm volatile("" : "+v"(ahead));                 // compared where it is used: sixteen masks kept would not fit the scalar registers
                    auto weights = [&](int n) {                     // half n % 2 of block n / 2: keys 32 kb .., queries 32 qb ..
                        const int b = n >> 1, s = n & 1, kb = b == 2, qb = b != 0;
                        jl_f32x8 w = acc8(p[b], s);
#pragma unroll
                        for (int x = 0; x < 2; ++x) {
                            const int j0 = 32 * kb + 16 * s + 8 * x + 4 * hi;
                            const ch_f32x4 lj = *(const ch_f32x4 *)(Ls + j0), uj = *(const ch_f32x4 *)(us + j0);
#pragma unroll
                            for (int y = 0; y < 4; ++y) {
                                const float f = w[4 * x + y] * (__builtin_amdgcn_exp2f(li[qb] - lj[y]) * uj[y]);
                                w[4 * x + y] = b == 1 || 16 * s + 8 * x + y <= ahead ? f : 0.f;
                            }
                        }
                        jl_split8(w, part[n & 1]);
                    };
                    weights(0);
#pragma unroll
                    for (int n = 0; n < 6; ++n) {
                        if (n < 5) weights(n + 1);
#pragma unroll
                        for (int x = 0; x < CH_TERMS; ++x) o[n >= 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part[n & 1][x], vf[2 * (n >= 4) + (n & 1)], o[n >= 2], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if (a.skip)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[y][r] += skip * (float)vf[2 * y + (r >> 3)][r & 7];
                if (flawed) {
                    int here = l32;
                    asm volatile("" : "+v"(here));
                    const int broken = brokenS[here] - 4 * hi;
#pragma unroll
                    for (int y = 0; y < 2; ++y)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[y][r] = 32 * y + 8 * (r >> 2) + (r & 3) < broken ? o[y][r] : NAN;
                }
            } else {
#pragma unroll
                for (int s = 0; s < CH_T / 16; ++s) vf[s] = turned(Vs, VROW, 32 * wave, s);
            }
        }
        if (busy && more) {
#pragma unroll
            for (int x = 0; x < NT; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) S[x][r] *= g;
            jl_bf16x8 part[2][CH_TERMS], kf[2][NT];
            auto operands = [&](int s) {
                jl_f32x8 w = __builtin_convertvector(vf[s], jl_f32x8);
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const ch_f32x4 e4 = *(const ch_f32x4 *)(es + 16 * s + 8 * x + 4 * hi);
#pragma unroll
                    for (int y = 0; y < 4; ++y) w[4 * x + y] *= e4[y];
                }
                jl_split8(w, part[s & 1]);
#pragma unroll
                for (int x = 0; x < NT; ++x) kf[s & 1][x] = turned(Ks, QROW, 32 * x, s);
            };
            operands(0);
#pragma unroll
            for (int s = 0; s < CH_T / 16; ++s) {
                if (s + 1 < CH_T / 16) operands(s + 1);
#pragma unroll
                for (int y = 0; y < CH_TERMS; ++y)
#pragma unroll
                    for (int x = 0; x < NT; ++x) S[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s & 1][x], part[s & 1][y], S[x], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (flawed) {
                int here = l32;
                asm volatile("" : "+v"(here));
                if (brokenS[here] < CH_T)
#pragma unroll
                    for (int x = 0; x < NT; ++x)
#pragma unroll
                        for (int r = 0; r < 16; ++r) S[x][r] = NAN;
            }
        }
    }
    if (OUT) outputs((cnt - 1) / CH_T * CH_T, cnt - (cnt - 1) / CH_T * CH_T);
    if (!busy || (OUT && !last)) return;
    char *dst = (char *)(OUT ? a.state + ((int64_t)slot * H + h) * D * Dv : a.scratch + ((int64_t)piece * H + h) * D * Dv);
    if (sc < Dv) each_state([&](int d, uint32_t off, float v) { if (d < D) *(float *)(dst + off) = v; return v; });
    if (!OUT && lane == 0 && c_base == 0) a.scratch[(int64_t)a.chunks * H * D * Dv + (int64_t)piece * H + h] = l_all;
}

// The state every piece starts from, in place of its own contribution: S = the request's state (zero at position 0); for each piece in order
// its contribution is replaced by S, then S = exp(its log decay) S + contribution (a request's last piece has none: nobody reads on).
__global__ __launch_bounds__(256) void scan_join_kernel(jl_scan_args a) {
    const int b = blockIdx.x / a.H, h = blockIdx.x - b * a.H;
    const int p0 = a.req[4 * b], np = a.req[4 * b + 1], pos0 = a.req[4 * b + 2], slot = a.req[4 * b + 3];
    const int64_t ddv = (int64_t)a.D * a.Dv;
    const float *sp = a.state + ((int64_t)slot * a.H + h) * ddv, *ll = a.scratch + (int64_t)a.chunks * a.H * ddv;
    for (int64_t e = (int64_t)blockIdx.y * 256 + threadIdx.x; e < ddv; e += (int64_t)gridDim.y * 256) {
        float S = pos0 > 0 ? sp[e] : 0.f;
        float *lp = a.scratch + ((int64_t)p0 * a.H + h) * ddv + e;
        if (np == 1) {                                              // (its own way: single tokens beside a prompt are many)
            *lp = S;
            continue;
        }
        const float *l = ll + (int64_t)p0 * a.H + h;
        float local = *lp, fade = *l;
        for (int p = 0; p < np; ++p, lp += a.H * ddv) {
            l += a.H;
            const float next = p + 2 < np ? lp[a.H * ddv] : 0.f, next_fade = p + 2 < np ? *l : 0.f;      // on their way while this piece is joined
            *lp = S;
            if (p + 1 < np) S = exp2f(fade) * S + local;
            local = next;
            fade = next_fade;
        }
    }
}

template <int DP, int NW> static int scan_chunk_launch(const jl_scan_args &a, int heads, int blocks, hipStream_t st) {
    const int per_head = (a.Dv + 31) / 32;
    const dim3 grid((unsigned)a.chunks, (unsigned)(a.G * ((a.H / a.G + heads - 1) / heads)), (unsigned)((per_head + NW - 1) / NW));
    static_assert(ch_lds_bytes(DP, NW, true) <= 64 * 1024, "static limit of a launch");
    const bool alone = a.chunks == a.B;
    if (!alone) {
        scan_chunk_kernel<DP, NW, CH_LOCAL><<<grid, 64 * NW, ch_lds_bytes(DP, NW, false), st>>>(a, heads, blocks, 0);
        const int64_t ddv = (int64_t)a.D * a.Dv;
        scan_join_kernel<<<dim3((unsigned)(a.B * a.H), (unsigned)((ddv + 255) / 256 < 64 ? (ddv + 255) / 256 : 64)), 256, 0, st>>>(a);
    }
    scan_chunk_kernel<DP, NW, CH_OUT><<<grid, 64 * NW, ch_lds_bytes(DP, NW, true), st>>>(a, heads, blocks, alone);
    return jl_check_launch("scan_chunk_kernel");
}
// Four wavefronts per workgroup where a head's columns or the heads that read the same q and k fill more than two of them; else two.
template <int DP> static int scan_chunk_launch(const jl_scan_args &a, hipStream_t st) {
    const int per_head = (a.Dv + 31) / 32, sharing = a.H / a.G;
    const int heads = per_head >= 3 || sharing == 1 ? 1 : per_head == 1 && sharing >= 3 ? 4 : 2;
    if (heads * per_head > 2) return scan_chunk_launch<DP, 4>(a, heads, per_head < 4 ? per_head : 4, st);
    return scan_chunk_launch<DP, 2>(a, heads, per_head, st);
}

extern "C" int jl_linear_scan_chunked_ok(int dtype, int32_t D, int32_t Dv) { return dtype == JL_BF16 && D > 0 && D <= 128 && D % 4 == 0 && Dv > 0 && Dv % 4 == 0; }

// The pieces' kernel forms offsets of 64 rows of outputs and of src, and of a head's state, in 32 bits; wider calls take the scan.
static bool ch_in_reach(const jl_scan_args &a) { return (int64_t)a.H * a.Dv <= 1 << 24 && a.Dv <= 1 << 22 && a.ld <= 1 << 26; }

extern "C" int jl_linear_scan(const jl_scan_args *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_linear_scan: null arguments");
    const jl_scan_args &a = *ap;
    if (a.B <= 0) return JL_OK;
    if (!a.src || !a.seq || !a.state || !a.out || (!a.decay && (!a.dt || !a.A_log || !a.dt_bias))) return jl_fail(JL_E_INVALID, "jl_linear_scan: null pointer");
    if (a.H <= 0 || a.G <= 0 || a.H % a.G || a.D <= 0 || a.D > 256 || a.Dv <= 0) return jl_fail(JL_E_INVALID, "jl_linear_scan: heads must be a multiple of the key heads, D <= 256");
    if (a.q_col < 0 || a.k_col < 0 || a.v_col < 0 || a.q_col + (int64_t)a.G * a.D > a.ld || a.k_col + (int64_t)a.G * a.D > a.ld || a.v_col + (int64_t)a.H * a.Dv > a.ld ||
        (!a.decay && (a.dt_col < 0 || a.dt_col + (int64_t)a.H > a.dt_ld)))
        return jl_fail(JL_E_INVALID, "jl_linear_scan: columns do not fit the rows");
    if (a.act != JL_ACT_SILU && a.act != JL_ACT_NONE) return jl_fail(JL_E_INVALID, "jl_linear_scan: unknown activation %d", a.act);
    hipStream_t st = (hipStream_t)stream;
    if (a.chunks > 0) {
        if (!a.chunk_rec || !a.req || !a.scratch) return jl_fail(JL_E_INVALID, "jl_linear_scan: pieces need their records and a scratch");
        if (!jl_linear_scan_chunked_ok(a.dtype, a.D, a.Dv) || a.ld % 4 || a.q_col % 4 || a.k_col % 4 || a.v_col % 4 || (uintptr_t)a.src % 8)
            return jl_fail(JL_E_INVALID, "jl_linear_scan: pieces take bfloat16, D a multiple of four up to 128, Dv, columns and rows in multiples of four");
        if (ch_in_reach(a)) {
            if (a.D <= 32) return scan_chunk_launch<32>(a, st);
            if (a.D <= 64) return scan_chunk_launch<64>(a, st);
            if (a.D <= 96) return scan_chunk_launch<96>(a, st);
            return scan_chunk_launch<128>(a, st);
        }
    }
    JL_DISPATCH(a.dtype, return scan_launch<T>(a, st));
    return JL_OK;
}
