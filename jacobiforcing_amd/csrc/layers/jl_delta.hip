// jl_delta.hip — the gated delta rule: a recurrent mixer whose float state S [D, Dv] per (request slot, head) is decayed, corrected towards
// the current value along the current key, and read with the current query, token by token:
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// with q, k unit vectors per head (q also times q_scale), beta = sigmoid(b) and g = exp(-exp(A_log_h) softplus(a + dt_bias_h)) per head and
// token, and the output brought to unit RMS per head, times a weight over Dv, times silu(gate).  Everything but the inputs is float.
#include "jl_common.h"
#include <type_traits>

// One workgroup per (request, head).  The columns of S are independent of each other, so column j is owned by LPC adjacent lanes, each
// with DMAX / LPC consecutive rows in registers; the two dot products of a token (k . S_j and q . S_j) are partial sums per lane joined by
// LPC - 1 exchanges.  Tokens are taken DL_TT at a time: raw queries and keys go to LDS, a wavefront per token makes them unit vectors, one
// thread per token evaluates the decay and the step size; the per-head sums of squares of the outputs are reduced once per group.
constexpr int DL_TT = 8;

template <typename T, typename TQ, int DMAX, int LPC>
__global__ __launch_bounds__(1024) void delta_rule_kernel(const TQ *__restrict__ qkv, int64_t qkv_ld, int q_col, int k_col, int v_col,
                                                           const T *__restrict__ proj, int64_t ld, int a_col, int b_col, int g_col,
                                                           const float *__restrict__ A_log, const float *__restrict__ dt_bias,
                                                           const float *__restrict__ norm_w, const int32_t *__restrict__ seq, int H, int G, int D, int Dv,
                                                           float unit_eps, float q_scale, float eps, float *__restrict__ state, T *__restrict__ out) {
    constexpr int DPER = DMAX / LPC;
    extern __shared__ float lds[];
    float *qs = lds;                                   // [TT][DMAX]
    float *ks = qs + DL_TT * DMAX;                     // [TT][DMAX]
    float *gs = ks + DL_TT * DMAX;                     // [TT] decay
    float *bs = gs + DL_TT;                            // [TT] step size
    float *red = bs + DL_TT;                           // [TT][16]
    const int b = blockIdx.x / H, h = blockIdx.x - b * H, kh = h / (H / G);
    const int row0 = seq[4 * b], cnt = seq[4 * b + 1], pos0 = seq[4 * b + 2], slot = seq[4 * b + 3];
    if (cnt <= 0) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, nw = (blockDim.x + 63) >> 6;
    const int j = tid / LPC, sub = tid - j * LPC, d0 = sub * DPER;
    const bool live = j < Dv;
    const float neg_rate = -expf(A_log[h]), bias = dt_bias[h];
    float *sp = state + ((int64_t)slot * H + h) * D * Dv;
    float S[DPER];
#pragma unroll
    for (int i = 0; i < DPER; ++i) S[i] = (live && d0 + i < D && pos0 > 0) ? sp[(int64_t)(d0 + i) * Dv + j] : 0.f;

    for (int t0 = 0; t0 < cnt; t0 += DL_TT) {
        const int nt = cnt - t0 < DL_TT ? cnt - t0 : DL_TT;
        __syncthreads();
        for (int e = tid; e < nt * DMAX; e += blockDim.x) {
            const int tt = e / DMAX, d = e - tt * DMAX;
            const TQ *row = qkv + (int64_t)(row0 + t0 + tt) * qkv_ld + kh * D;
            qs[e] = d < D ? ld_f(row + q_col + d) : 0.f;
            ks[e] = d < D ? ld_f(row + k_col + d) : 0.f;
        }
        if (tid < nt) {
            const T *row = proj + (int64_t)(row0 + t0 + tid) * ld;
            gs[tid] = expf(neg_rate * softplus_f(ld_f(row + a_col + h) + bias));
            bs[tid] = 1.0f / (1.0f + expf(-ld_f(row + b_col + h)));
        }
        __syncthreads();
        for (int tt = wave; tt < nt; tt += nw) {               // unit vectors: a wavefront per token
            float sq = 0.f, sk = 0.f;
            for (int d = lane; d < D; d += 64) { const float a = qs[tt * DMAX + d], c = ks[tt * DMAX + d]; sq += a * a; sk += c * c; }
            sq = wave_sum_f32(sq);
            sk = wave_sum_f32(sk);
            const float rq = q_scale / sqrtf(sq + unit_eps), rk = 1.0f / sqrtf(sk + unit_eps);
            for (int d = lane; d < D; d += 64) { qs[tt * DMAX + d] *= rq; ks[tt * DMAX + d] *= rk; }
        }
        __syncthreads();
        float o[DL_TT];
#pragma unroll
        for (int tt = 0; tt < DL_TT; ++tt) {
            o[tt] = 0.f;
            if (tt < nt) {
                const float v = live ? ld_f(qkv + (int64_t)(row0 + t0 + tt) * qkv_ld + v_col + h * Dv + j) : 0.f;
                const float *qp = qs + tt * DMAX + d0, *kp = ks + tt * DMAX + d0;
                const float g = gs[tt], beta = bs[tt];
                float dot = 0.f;
#pragma unroll
                for (int i = 0; i < DPER; ++i) dot += kp[i] * S[i];
#pragma unroll
                for (int off = 1; off < LPC; off <<= 1) dot += __shfl_xor(dot, off, 64);
                const float u = beta * (v - g * dot);
                float acc = 0.f;
#pragma unroll
                for (int i = 0; i < DPER; ++i) {
                    S[i] = g * S[i] + kp[i] * u;
                    acc += S[i] * qp[i];
                }
#pragma unroll
                for (int off = 1; off < LPC; off <<= 1) acc += __shfl_xor(acc, off, 64);
                o[tt] = acc;
                const float ss = wave_sum_f32((live && sub == 0) ? acc * acc : 0.f);
                if (lane == 0) red[tt * 16 + wave] = ss;
            }
        }
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < DL_TT; ++tt)
            if (tt < nt && live && sub == 0) {
                float ss = 0.f;
                for (int w = 0; w < nw; ++w) ss += red[tt * 16 + w];
                const float r = 1.0f / sqrtf(ss / (float)Dv + eps);
                const int64_t n = row0 + t0 + tt;
                const float gt = ld_f(proj + n * ld + g_col + h * Dv + j);
                st_f(out + n * ((int64_t)H * Dv) + h * Dv + j, o[tt] * r * norm_w[j] * silu_f(gt));
            }
    }
    if (live)
#pragma unroll
        for (int i = 0; i < DPER; ++i)
            if (d0 + i < D) sp[(int64_t)(d0 + i) * Dv + j] = S[i];
}


// ---- long portions: the columns of S shared out over single-wavefront workgroups -------------------------------------------------------------
// A prompt's portion is a chain of cnt dependent steps per (request, head); what shortens it is less work per step and nothing to wait for
// inside it.  Here a workgroup is ONE wavefront that owns 64 / LPC columns of one head's state (grid.y walks the head's columns), so a step is
// DMAX / LPC * 3 multiply-adds per lane, and the chip runs B * H * Dv * LPC / 64 such chains side by side.  Every wavefront stages the group's
// queries and keys itself (eight lanes per token make them unit vectors) and fetches the next group's inputs into registers before it starts
// on the current one.  The outputs leave unnormalised (float): the norm over a head's Dv values spans workgroups and is delta_out_kernel's.
constexpr int DC_TT = 8;        // tokens per group = 64 lanes / 8 lanes per token in the unit-vector stage

// sum over the LPC adjacent lanes that share a column; four lanes are a quad, whose exchanges are register moves (DPP), not LDS traffic
template <int LPC>
__device__ __forceinline__ float column_sum(float v) {
    if constexpr (LPC == 4 || LPC == 8) {
        v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));      // quad_perm [1, 0, 3, 2]
        v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));      // quad_perm [2, 3, 0, 1]
        if constexpr (LPC == 8)                                                                           // lane i <-> 7 - i of each eight: the other quad's sum
            v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
    } else {
#pragma unroll
        for (int off = 1; off < LPC; off <<= 1) v += __shfl_xor(v, off, 64);
    }
    return v;
}

template <typename T, int DMAX, int LPC>
__global__ __launch_bounds__(64) void delta_cols_kernel(const float *__restrict__ qkv, int64_t qkv_ld, int q_col, int k_col, int v_col,
                                                         const T *__restrict__ proj, int64_t ld, int a_col, int b_col, const float *__restrict__ A_log,
                                                         const float *__restrict__ dt_bias, const int32_t *__restrict__ seq, int H, int G, int D, int Dv,
                                                         float unit_eps, float q_scale, float *__restrict__ state, float *__restrict__ raw) {
    // a token's row in LDS: the LPC lanes of a column read DPER consecutive values each, DPER apart — four floats between the parts keep
    // their 16-byte reads on different banks
    constexpr int DPER = DMAX / LPC, CPW = 64 / LPC, PRE = DC_TT * DMAX / 64, ROW = DMAX + 4 * LPC;
    __shared__ float qs[DC_TT * ROW], ks[DC_TT * ROW], gs[DC_TT], bs[DC_TT];
    auto at = [](int tt, int d) { return tt * ROW + d + (d / DPER) * 4; };
    const int b = blockIdx.x / H, h = blockIdx.x - b * H, kh = h / (H / G);
    const int row0 = seq[4 * b], cnt = seq[4 * b + 1], pos0 = seq[4 * b + 2], slot = seq[4 * b + 3];
    if (cnt <= 0) return;
    const int lane = threadIdx.x, j = blockIdx.y * CPW + lane / LPC, sub = lane % LPC, d0 = sub * DPER;
    const bool live = j < Dv;
    const float neg_rate = -expf(A_log[h]), bias = dt_bias[h];
    float *sp = state + ((int64_t)slot * H + h) * D * Dv;
    float S[DPER];
#pragma unroll
    for (int i = 0; i < DPER; ++i) S[i] = (live && d0 + i < D && pos0 > 0) ? sp[(int64_t)(d0 + i) * Dv + j] : 0.f;
    float pq[PRE], pk[PRE], pv[DC_TT], pa = 0.f, pb = 0.f;
    auto fetch = [&](int t0) {
        const int nt = cnt - t0 < DC_TT ? cnt - t0 : DC_TT;
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int e = i * 64 + lane, tt = e / DMAX, d = e - tt * DMAX;
            const bool ok = tt < nt && d < D;
            const float *row = qkv + (int64_t)(row0 + t0 + tt) * qkv_ld + kh * D + d;
            pq[i] = ok ? row[q_col] : 0.f;
            pk[i] = ok ? row[k_col] : 0.f;
        }
#pragma unroll
        for (int tt = 0; tt < DC_TT; ++tt) pv[tt] = (tt < nt && live) ? qkv[(int64_t)(row0 + t0 + tt) * qkv_ld + v_col + h * Dv + j] : 0.f;
        if (lane < nt) {
            const T *row = proj + (int64_t)(row0 + t0 + lane) * ld;
            pa = ld_f(row + a_col + h);
            pb = ld_f(row + b_col + h);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < cnt; t0 += DC_TT) {
        const int nt = cnt - t0 < DC_TT ? cnt - t0 : DC_TT;
        __syncthreads();                                        // the group before has been read
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int e = i * 64 + lane, tt = e / DMAX, d = e - tt * DMAX;
            qs[at(tt, d)] = pq[i];
            ks[at(tt, d)] = pk[i];
        }
        if (lane < nt) {
            gs[lane] = expf(neg_rate * softplus_f(pa + bias));
            bs[lane] = 1.0f / (1.0f + expf(-pb));
        }
        float v[DC_TT];
#pragma unroll
        for (int tt = 0; tt < DC_TT; ++tt) v[tt] = pv[tt];
        __syncthreads();
        {                                                       // unit vectors: eight lanes per token, its values in registers between the two passes
            const int tt = lane >> 3, s8 = lane & 7;
            float qv[DMAX / 8], kv[DMAX / 8];
            float sq = 0.f, sk = 0.f;
#pragma unroll
            for (int i = 0; i < DMAX / 8; ++i) {
                const int d = s8 + 8 * i;
                qv[i] = qs[at(tt, d)];
                kv[i] = ks[at(tt, d)];
                sq += qv[i] * qv[i];
                sk += kv[i] * kv[i];
            }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) { sq += __shfl_xor(sq, off, 64); sk += __shfl_xor(sk, off, 64); }
            const float rq = q_scale / sqrtf(sq + unit_eps), rk = 1.0f / sqrtf(sk + unit_eps);
#pragma unroll
            for (int i = 0; i < DMAX / 8; ++i) {
                const int d = s8 + 8 * i;
                qs[at(tt, d)] = qv[i] * rq;
                ks[at(tt, d)] = kv[i] * rk;
            }
        }
        __syncthreads();
        if (t0 + DC_TT < cnt) fetch(t0 + DC_TT);                // in flight while this group's steps run
#pragma unroll
        for (int tt = 0; tt < DC_TT; ++tt) {
            if (tt < nt) {
                const float *qp = qs + tt * ROW + d0 + sub * 4, *kp = ks + tt * ROW + d0 + sub * 4;
                const float g = gs[tt], beta = bs[tt];
                float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < DPER; ++i) dot[i & 3] += kp[i] * S[i];
                const float dsum = column_sum<LPC>((dot[0] + dot[1]) + (dot[2] + dot[3]));
                const float u = beta * (v[tt] - g * dsum);
                float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < DPER; ++i) {
                    S[i] = g * S[i] + kp[i] * u;
                    acc[i & 3] += S[i] * qp[i];
                }
                const float o = column_sum<LPC>((acc[0] + acc[1]) + (acc[2] + acc[3]));
                if (live && sub == 0) raw[(int64_t)(row0 + t0 + tt) * ((int64_t)H * Dv) + h * Dv + j] = o;
            }
        }
    }
    if (live)
#pragma unroll
        for (int i = 0; i < DPER; ++i)
            if (d0 + i < D) sp[(int64_t)(d0 + i) * Dv + j] = S[i];
}

// out_h(t) = o / sqrt(mean(o^2) + eps) * norm_w * silu(gate_h(t)): 32 lanes per (token, head), four values at a time where rows lie at their borders (bytes bound it:
// 134 MB at 8192 tokens x 16 heads of 128, a wavefront per row and a value per lane 59 us)
template <typename T, int VW>
__global__ __launch_bounds__(256) void delta_out_kernel(const float *__restrict__ raw, const T *__restrict__ proj, int64_t ld, int g_col,
                                                         const float *__restrict__ norm_w, int64_t NH, int H, int Dv, float eps, T *__restrict__ out) {
    const int64_t r = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    if (r >= NH) return;
    const int lane = threadIdx.x & 31;
    const int64_t n = r / H;
    const int h = (int)(r - n * H);
    const float *o = raw + r * Dv;
    const T *gate = proj + n * ld + g_col + (int64_t)h * Dv;
    float ss = 0.f, v[VW], g[VW];
    auto load = [&](int c) {
        if constexpr (VW == 4) ld4_f(o + c, v);
        else v[0] = o[c];
    };
    for (int c = VW * lane; c < Dv; c += 32 * VW) {
        load(c);
#pragma unroll
        for (int i = 0; i < VW; ++i) ss += v[i] * v[i];
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float rr = 1.0f / sqrtf(ss / (float)Dv + eps);
    for (int c = VW * lane; c < Dv; c += 32 * VW) {
        if (Dv > 32 * VW) load(c);                                  // otherwise it is still there
        if constexpr (VW == 4) ld4_f(gate + c, g);
        else g[0] = ld_f(gate + c);
#pragma unroll
        for (int i = 0; i < VW; ++i) g[i] = v[i] * rr * (norm_w ? norm_w[c + i] : 1.0f) * silu_f(g[i]);
        if constexpr (VW == 4) st4_f(out + r * Dv + c, g);
        else st_f(out + r * Dv + c, g[0]);
    }
}
template <typename T>
static int delta_out_launch(const float *raw, const void *proj, int64_t ld, int g_col, const float *norm_w, int64_t NH, int H, int Dv, float eps, void *out, hipStream_t st) {
    const dim3 grid((unsigned)((NH + 7) / 8));
    if ((ld | g_col | Dv) % 4 == 0 && !(((uintptr_t)raw & 15) | (((uintptr_t)proj | (uintptr_t)out) & (4 * sizeof(T) - 1))))
        delta_out_kernel<T, 4><<<grid, 256, 0, st>>>(raw, (const T *)proj, ld, g_col, norm_w, NH, H, Dv, eps, (T *)out);
    else delta_out_kernel<T, 1><<<grid, 256, 0, st>>>(raw, (const T *)proj, ld, g_col, norm_w, NH, H, Dv, eps, (T *)out);
    return jl_check_launch("delta_out_kernel");
}

int jl_heads_out(const float *raw, const void *proj, int dtype, int64_t ld, int g_col, const float *norm_w, int64_t NH, int H, int Dv, float eps, void *out, hipStream_t st) {
    JL_DISPATCH(dtype, return delta_out_launch<T>(raw, proj, ld, g_col, norm_w, NH, H, Dv, eps, out, st));
    return JL_OK;
}

// ---- long portions on the matrix instructions, of floats and (the chain) of bfloat16 terms: 64 tokens at a time ------------------------------------------------------------------------
// With c_t = the running sum of ln g within a chunk of 64 tokens, S the state the chunk starts from, and u_t the corrections, the recurrence is
//   (I + A) U = diag(beta) V - diag(beta e^c) K S,   A_tj = beta_t e^(c_t - c_j) (k_t . k_j) for j < t        (unit lower triangular)
//   o_t = e^(c_t) S^T q_t + sum_{j <= t} e^(c_t - c_j) (q_t . k_j) u_j,        S <- e^(c_63) S + sum_j e^(c_63 - c_j) k_j u_j^T
// so with T = (I + A)^-1, W1 = T diag(beta) V and W2 = T diag(beta e^c) K a chunk costs the chain four products: U = W1 - W2 S, then o and S.
// delta_chunk_kernel makes unit vectors, T, W1, -W2 and P_tj = e^(c_t - c_j) (q_t . k_j) for all chunks and heads side by side; delta_chain_kernel walks a request's
// chunks with 32 columns of one head's state in accumulators.  Everything is a 32-bit number, as in the scan; the sums c are 64-bit (differences of long sums).  A token
// that does not exist has k = q = v = 0, beta = 0, g = 1.  ln g below -1e4 counts as -1e4: e^ of it is zero all the same, and differences stay numbers.
//
// What is not finite in a token's key, value, decay or beta reaches its own and later tokens' outputs and the state, as in the scan, though products run over whole chunks: it is left
// out of them and set afterwards (in rare branches: W1's rows from that token on, the outputs' rows from a correction's token on, the state's columns).
//
// v_mfma_f32_32x32x2_f32: lane l supplies row (A) or column (B) l % 32 at depth l / 32; accumulator r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.  Four
// instructions take a unit of 16 bytes per lane, depths 8 u + 4 (l / 32) + i of unit u — which is also how four accumulators of a lane lie, so results are the next
// product's operand as they are: between the kernels (every operand as units [unit][lane], read as 1 KB per wavefront straight into registers, a chunk ahead) and in LDS
// between the wavefronts of a chain.  T comes from 16 x 16 blocks by substitution, joined by products, on one wavefront while the others make P.
// The chain's operands are split into three bfloat16 terms each, on the wavefronts that hold them, while the other wavefront of a SIMD multiplies: a product with S takes 48
// instructions of 32 cycles instead of 64 of 64, one with U 24 instead of 32.  Errors against 64 bits, heads of 128, 1021 tokens: outputs 1.20e-7 and state 1.02e-7, with
// products of floats 1.24e-7 and 1.17e-7; with long memories 1.55e-7 and 1.40e-7, 1.82e-7 and 1.76e-7.
// What bounds it: the chain's two waits per chunk, with the product with S (about 3900 cycles), then the correction's own split and the keys' product between them; in the chunks'
// kernel the phases of a workgroup that wait for memory and for each other (two workgroups per CU at 79 104 bytes of LDS).  Its loads set out together and V's in front of
// the stores: a load waits for the stores in front of it, here 57 000 of a workgroup's 145 000 cycles.
// Measured, norm and gate included, bfloat16, heads of 128: 16 heads, 4 x 2048 tokens 446 -> 328 us (chunks 210 -> 150, chain 200 -> 137, norm 40; columns walking token by token
// took 1446); float, 8 heads, 1021 + 851 + 681 tokens 147 -> 106, heads of 64 101 -> 80.
constexpr int DK_T = 64;
typedef float dk_f32x16 __attribute__((ext_vector_type(16)));
typedef float dk_f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ dk_f32x16 dk_mma(float4 a, float4 b, dk_f32x16 c) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, c, 0, 0, 0);
}
__device__ __forceinline__ dk_f32x4 dk_mma16(float4 a, float4 b, dk_f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}
// a product 16 deep of 32-bit operands: each the sum of three bfloat16 numbers, the pairs of terms whose product is above 2 ** -26 of the whole, the greatest apart from the others
struct dk_terms { jl_bf16x8 t[JL_SPLIT_TERMS]; };
__device__ __forceinline__ dk_terms dk_split(float4 a, float4 b) {
    dk_terms r;
    jl_split8(jl_f32x8{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, r.t);
    return r;
}
struct dk_sums { dk_f32x16 great, small; };
__device__ __forceinline__ void dk_clear(dk_sums &c) {
#pragma unroll
    for (int r = 0; r < 16; ++r) c.great[r] = c.small[r] = 0.f;
}
__device__ __forceinline__ dk_f32x16 dk_total(const dk_sums &c) { return c.great + c.small; }
__device__ __forceinline__ void dk_mma_split(const dk_terms &a, const dk_terms &b, dk_sums &c) {
    c.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[0], b.t[2], c.small, 0, 0, 0);
    c.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[1], b.t[1], c.small, 0, 0, 0);
    c.great = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[0], b.t[0], c.great, 0, 0, 0);
    c.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[2], b.t[0], c.small, 0, 0, 0);
    c.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[0], b.t[1], c.small, 0, 0, 0);
    c.small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.t[1], b.t[0], c.small, 0, 0, 0);
}
__device__ __forceinline__ void dk_wave_sync() {        // LDS written by some lanes is read by others of the same wavefront
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// e ** x of a 64-bit sum: the float next to x, and what is left of x to first order (rounding x itself would cost |x| 2 ** -25)
__device__ __forceinline__ float dk_exp(double x) {
    const float hi = (float)x, e = expf(hi);
    return fmaf(e, (float)(x - (double)hi), e);
}

// floats of scratch: per chunk and head W2, W1, P, e^c and e^(c_63 - c); per chunk and key head the unit vectors
struct dk_sizes { int64_t w2, w1, p, head, group; };
static __host__ __device__ inline dk_sizes dk_layout(int DP, int Dv) {
    dk_sizes z;
    z.w2 = 0;
    z.w1 = (int64_t)DK_T * DP;
    z.p = z.w1 + (int64_t)DK_T * ((Dv + 31) / 32 * 32);
    z.head = z.p + 3 * 1024 + 2 * DK_T;
    z.group = (int64_t)2 * DK_T * DP;
    return z;
}

// FAR: rows of qkv of which 64 are not within 32 bits of each other (where they are, offsets of 64 bits cost registers and 5 to 20 % of a launch)
template <typename T, int DP, bool FAR>
__global__ __launch_bounds__(256, 2) void delta_chunk_kernel(jl_delta_chunks a, int h0, int nh) {
    typedef typename std::conditional<FAR, int64_t, uint32_t>::type row_t;
    constexpr int U = DP / 4, DT = DP / 32;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float4 *Ks = (float4 *)smem, *Qs = Ks + DK_T * U, *Am = Qs + DK_T * U;          // rows of units, permuted by the row
    double *cs = (double *)(Am + 3 * 256);                                         // [64] sums of ln g
    float *bs = (float *)(cs + DK_T), *bg = bs + DK_T;                             // [64] beta; -beta e^c
    int *flawS = (int *)(bg + DK_T);                                               // [64] a key that is not a number
    const int hl = blockIdx.x % nh, h = h0 + hl, chunk = blockIdx.x / nh, per = a.H / a.G, kh = h / per, D = a.D, Dv = a.Dv;
    const int row0 = a.chunk_rec[4 * chunk], cnt = a.chunk_rec[4 * chunk + 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    const dk_sizes z = dk_layout(DP, Dv);
    float *head = a.scratch + ((int64_t)chunk * nh + hl) * z.head;
    float *group = a.scratch + (int64_t)a.chunks * nh * z.head + ((int64_t)chunk * (nh / per) + hl / per) * z.group;
    const bool leader = hl % per == 0;                                             // writes its key head's unit vectors
    auto at = [](int row, int u) { return u ^ (row & 15); };                        // rows have a multiple of 16 units
    auto am_at = [](int t, int u) { return t < 32 ? t * 8 + (u ^ (t & 7)) : 256 + (t - 32) * 16 + (u ^ (t & 15)); };    // A, then T: the first 32 rows have 32 columns
    const float *src = a.qkv + (int64_t)row0 * a.qkv_ld + kh * D;
    constexpr int IT = DK_T * U / 256;
    float ga = 0.f, gb = 0.f;
    if (wave == 0) {                                                               // everything that is read sets out here, V a phase later: nothing waits for memory twice
        const T *row = (const T *)a.proj + (int64_t)(row0 + min(lane, cnt - 1)) * a.ld;
        ga = ld_f(row + a.a_col + h);
        gb = ld_f(row + a.b_col + h);
    }
    float4 qv[IT], kv[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {                                              // a row that does not exist: the last one's, not used
        const int e = tid + it * 256, tt = min(e / U, cnt - 1), d = 4 * (e % U) < D ? 4 * (e % U) : 0;
        const row_t at = (row_t)tt * (row_t)a.qkv_ld + d;
        qv[it] = *(const float4 *)(src + a.q_col + at);
        kv[it] = *(const float4 *)(src + a.k_col + at);
    }
    if (wave == 0) {
        float lg = 0.f, beta = 0.f;
        if (lane < cnt) {
            lg = -expf(a.A_log[h]) * softplus_f(ga + a.dt_bias[h]);
            lg = lg < -1e4f ? -1e4f : lg;
            beta = 1.0f / (1.0f + expf(-gb));
        }
        double c = lg;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double y = __shfl_up(c, off, 64);
            if (lane >= off) c += y;
        }
        const double end = __shfl(c, 63, 64);
        const float gam = dk_exp(c);
        cs[lane] = c;
        bs[lane] = beta;
        bg[lane] = -beta * gam;
        head[z.p + 3 * 1024 + lane] = gam;
        head[z.p + 3 * 1024 + DK_T + lane] = dk_exp(end - c);
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {                                              // unit vectors: U adjacent lanes hold a row
        const int e = tid + it * 256, tt = e / U, u = e % U;
        const bool there = tt < cnt && 4 * u < D;
        float4 q = there ? qv[it] : make_float4(0.f, 0.f, 0.f, 0.f), k = there ? kv[it] : make_float4(0.f, 0.f, 0.f, 0.f);
        float sq = (q.x * q.x + q.y * q.y) + (q.z * q.z + q.w * q.w), sk = (k.x * k.x + k.y * k.y) + (k.z * k.z + k.w * k.w);
#pragma unroll
        for (int off = 1; off < U; off <<= 1) { sq += __shfl_xor(sq, off, 64); sk += __shfl_xor(sk, off, 64); }
        const float rq = tt < cnt ? a.q_scale / sqrtf(sq + a.unit_eps) : 0.f, rk = tt < cnt ? 1.0f / sqrtf(sk + a.unit_eps) : 0.f;
        Qs[tt * U + at(tt, u)] = make_float4(q.x * rq, q.y * rq, q.z * rq, q.w * rq);
        k = make_float4(k.x * rk, k.y * rk, k.z * rk, k.w * rk);
        const uint64_t none = __ballot(__builtin_isnan((k.x + k.y) + (k.z + k.w)));   // elements of a unit vector: what is not finite before is not a number now
        bool flaw = false;                                                          // the row's
        if (none) {
            flaw = none >> (lane & ~(U - 1)) & ((1ull << U) - 1);
            if (flaw) k = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        Ks[tt * U + at(tt, u)] = k;
        if (u == 0) flawS[tt] = flaw;
    }
    const int nv = (Dv + 31) / 32;
    const float *vp = a.qkv + (int64_t)row0 * a.qkv_ld + a.v_col + (int64_t)h * Dv;
    float vv[32];                                                                  // a wavefront's 32 columns of V, all tokens
    auto fetch_v = [&](int vt) {
        const int col = min(32 * vt + l32, Dv - 1);
#pragma unroll
        for (int i = 0; i < 32; ++i) vv[i] = vp[(row_t)min(8 * (i >> 2) + 4 * hi + (i & 3), cnt - 1) * (row_t)a.qkv_ld + col];
    };
    __syncthreads();
    // from the first token with a key, decay or beta that is not a number on: nothing here that zeros would spread to the tokens in front of it; W1 says so instead
    const uint64_t flaws = __ballot(flawS[lane] || !__builtin_isfinite((float)cs[lane]) || !__builtin_isfinite(bs[lane]));
    const int broken = flaws ? __builtin_ctzll(flaws) : DK_T;                       // the same in all wavefronts
    if (broken < DK_T) {
        __syncthreads();
        if (wave == 0 && lane >= broken) { bs[lane] = bg[lane] = 0.f; cs[lane] = broken > 0 ? cs[broken - 1] : 0.0; }
        __syncthreads();
    }
    // a quarter [32 t, 32 j] of K K^T or Q K^T: lane l ends with t = 32 ti + l % 32, unit y the four j at 32 tj + 8 y + 4 (l / 32)
    auto pairs = [&](const float4 *rows, int ti, int tj, bool diagonal, float row_factor, auto &&store) {
        const int t = 32 * ti + l32, j = 32 * tj + l32;
        dk_f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll 1
        for (int x0 = 0; x0 < U / 2; x0 += U / 4) {               // sums of 8 products in a row, met in pairs: what 64 in a row lose shows in the outputs
            dk_f32x16 half;
#pragma unroll
            for (int r = 0; r < 16; ++r) half[r] = 0.f;
#pragma unroll 1
            for (int x = x0; x < x0 + U / 4; x += 2) {
                dk_f32x16 s1, s2;
#pragma unroll
                for (int r = 0; r < 16; ++r) s1[r] = s2[r] = 0.f;
                s1 = dk_mma(Ks[j * U + at(j, 2 * x + hi)], rows[t * U + at(t, 2 * x + hi)], s1);
                s2 = dk_mma(Ks[j * U + at(j, 2 * x + 2 + hi)], rows[t * U + at(t, 2 * x + 2 + hi)], s2);
                half += s1 + s2;
            }
            s += half;
        }
        const double ct = cs[t];
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int jj = 32 * tj + 8 * y + 4 * hi + i;
                v[i] = jj < t || (diagonal && jj == t) ? s[4 * y + i] * row_factor * dk_exp(ct - cs[jj]) : 0.f;
            }
            store(t, y, make_float4(v[0], v[1], v[2], v[3]));
        }
    };
    if (wave < 3) {
        const int ti = wave > 0, tj = wave > 1;
        pairs(Ks, ti, tj, false, bs[32 * ti + l32], [&](int t, int y, float4 v) { Am[am_at(t, 8 * tj + 2 * y + hi)] = v; });
    } else if (leader) {
#pragma unroll 4
        for (int e = 0; e < 2 * (DP / 8); ++e) {
            const int t = 32 * (e / (DP / 8)) + l32, x = e % (DP / 8);
            ((float4 *)group)[e * 64 + lane] = Qs[t * U + at(t, 2 * x + hi)];
        }
    }
    if (wave < nv) fetch_v(wave);
    __syncthreads();
    if (wave == 0) {
        // (I + A)^-1 in place.  The four 16 x 16 blocks of the diagonal by substitution, a lane per column
        float *am = (float *)Am;
        auto el = [&](int t, int j) -> float & { return am[4 * am_at(t, j >> 2) + (j & 3)]; };
        {
            const int b0 = 16 * (lane >> 4), c = lane & 15;
            float x[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float s = r == c ? 1.0f : 0.f;
#pragma unroll
                for (int y = 0; y < (r + 3) / 4; ++y) {
                    const float4 v = Am[am_at(b0 + r, b0 / 4 + y)];
                    if (4 * y < r) s -= v.x * x[4 * y];
                    if (4 * y + 1 < r) s -= v.y * x[4 * y + 1];
                    if (4 * y + 2 < r) s -= v.z * x[4 * y + 2];
                    if (4 * y + 3 < r) s -= v.w * x[4 * y + 3];
                }
                x[r] = s;
            }
            dk_wave_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) el(b0 + r, b0 + c) = x[r];
            dk_wave_sync();
        }
        // below the diagonal: T_10 = -T_11 (A_10 T_00), of 16 x 16 blocks, then of 32 x 32 blocks
#pragma unroll
        for (int b0 = 0; b0 < 64; b0 += 32) {
            const int r16 = lane & 15, g = lane >> 4;
            const int t = b0 + 16 + r16;
            dk_f32x4 x = {0.f, 0.f, 0.f, 0.f};
            x = dk_mma16(Am[am_at(t, b0 / 4 + g)], make_float4(el(b0 + 4 * g, b0 + r16), el(b0 + 4 * g + 1, b0 + r16), el(b0 + 4 * g + 2, b0 + r16), el(b0 + 4 * g + 3, b0 + r16)), x);
            dk_f32x4 w = {0.f, 0.f, 0.f, 0.f};
            w = dk_mma16(Am[am_at(t, b0 / 4 + 4 + g)], make_float4(x[0], x[1], x[2], x[3]), w);
            dk_wave_sync();
#pragma unroll
            for (int i = 0; i < 4; ++i) el(b0 + 16 + 4 * g + i, b0 + r16) = -w[i];
            dk_wave_sync();
        }
        {
            const int t = 32 + l32;
            dk_f32x16 x, w;
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = w[r] = 0.f;
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const int j = 8 * y + 4 * hi;
                x = dk_mma(Am[am_at(t, 2 * y + hi)], make_float4(el(j, l32), el(j + 1, l32), el(j + 2, l32), el(j + 3, l32)), x);
            }
#pragma unroll
            for (int y = 0; y < 4; ++y) w = dk_mma(Am[am_at(t, 8 + 2 * y + hi)], make_float4(x[4 * y], x[4 * y + 1], x[4 * y + 2], x[4 * y + 3]), w);
            dk_wave_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) el(32 + 8 * (r >> 2) + 4 * hi + (r & 3), l32) = -w[r];
        }
    } else {
        const int ti = wave > 1, tj = wave > 2, tile = wave - 1;
        pairs(Qs, ti, tj, true, 1.0f, [&](int, int y, float4 v) { ((float4 *)(head + z.p))[(4 * tile + y) * 64 + lane] = v; });
    }
    __syncthreads();
    auto trow = [&](int ti, int y) { const int t = 32 * ti + l32; return Am[am_at(t, 2 * y + hi)]; };
    for (int task = wave; task < nv + DT; task += 4) {                             // V first: its loads would wait for the stores of the others
        float4 f[8];                                                               // 32 columns of K or V at all 64 depths
        dk_f32x16 acc[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;
        if (task < nv) {                                                           // W1: rows t, 32 columns of beta V
            const int vt = task, col = 32 * vt + l32;
#pragma unroll
            for (int y = 0; y < 8; ++y) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) { const int t = 8 * y + 4 * hi + i; v[i] = t < cnt && col < Dv ? vv[4 * y + i] * bs[t] : 0.f; }
                f[y] = make_float4(v[0], v[1], v[2], v[3]);
            }
#pragma unroll
            for (int y = 0; y < 8; ++y) {
                if (y < 4) acc[0] = dk_mma(trow(0, y), f[y], acc[0]);
                acc[1] = dk_mma(trow(1, y), f[y], acc[1]);
            }
            if (vt + 4 < nv) fetch_v(vt + 4);
            // all values of a column enter a row of the second half, one that is not finite as not a number: the same without it
            if (broken < DK_T || __any(!__builtin_isfinite(acc[1][0]))) {
                int none = broken;                                                 // this lane's column is not a number from here on
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;
#pragma unroll 1
                for (int y = 0; y < 8; ++y) {
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int t = 8 * y + 4 * hi + i;
                        v[i] = t < cnt && col < Dv ? vp[(row_t)t * (row_t)a.qkv_ld + col] * bs[t] : 0.f;
                        if (!__builtin_isfinite(v[i])) { v[i] = 0.f; none = min(none, t); }
                    }
                    if (y < 4) acc[0] = dk_mma(trow(0, y), make_float4(v[0], v[1], v[2], v[3]), acc[0]);
                    acc[1] = dk_mma(trow(1, y), make_float4(v[0], v[1], v[2], v[3]), acc[1]);
                }
                none = min(none, __shfl_xor(none, 32, 64));
#pragma unroll
                for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[ti][r] = 32 * ti + 8 * (r >> 2) + 4 * hi + (r & 3) < none ? acc[ti][r] : NAN;
            }
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int y = 0; y < 4; ++y)
                    ((float4 *)(head + z.w1))[((vt * 2 + ti) * 4 + y) * 64 + lane] = make_float4(acc[ti][4 * y], acc[ti][4 * y + 1], acc[ti][4 * y + 2], acc[ti][4 * y + 3]);
        } else {                                                                   // -W2 transposed: rows of K^T, columns t
            const float *kf = (const float *)Ks;
            const int x = task - nv, d = 32 * x + l32;
#pragma unroll
            for (int y = 0; y < 8; ++y) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) { const int t = 8 * y + 4 * hi + i; v[i] = kf[4 * (t * U + at(t, d >> 2)) + (d & 3)]; }
                f[y] = make_float4(v[0], v[1], v[2], v[3]);
                if (leader) ((float4 *)group)[(DP / 4 + 8 * x + y) * 64 + lane] = f[y];
            }
#pragma unroll
            for (int y = 0; y < 8; ++y) {
                const float4 s = *(const float4 *)(bg + 8 * y + 4 * hi), v = make_float4(f[y].x * s.x, f[y].y * s.y, f[y].z * s.z, f[y].w * s.w);
                if (y < 4) acc[0] = dk_mma(v, trow(0, y), acc[0]);
                acc[1] = dk_mma(v, trow(1, y), acc[1]);
            }
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int y = 0; y < 4; ++y)
                    ((float4 *)(head + z.w2))[(ti * (DP / 8) + 4 * x + y) * 64 + lane] = make_float4(acc[ti][4 * y], acc[ti][4 * y + 1], acc[ti][4 * y + 2], acc[ti][4 * y + 3]);
        }
    }
}

// Workgroup (request, head, 32 columns); the column blocks of a head lie eight apart, on one XCD, since they read the same operands.  Wavefronts 0 and 1 make U, 2 and 3 the
// outputs of 32 tokens each; the D / 32 that follow own 32 rows of S each.  What a wavefront takes from memory is split while another's matrix instructions run: two to a SIMD.
// WIDE: rows of outputs of which 64 lie further apart than a buffer reaches.
template <int DP, bool WIDE>
__global__ __launch_bounds__(256 + 2 * DP, 1) void delta_chain_kernel(jl_delta_chunks a, int h0, int nh, float *__restrict__ raw) {
    constexpr int NU = DP / 8;
    __shared__ jl_bf16x8 Sf[NU / 2 * 3 * 64], Uf[4 * 3 * 64];       // [16 depths][term][lane]
    __shared__ float4 Pf[2 * 4 * 64];                               // what the pairs take of U, as accumulators lie
    __shared__ int noneS[2][32];                                    // the first token of a half chunk whose correction is not finite, per column
    const int nv = (a.Dv + 31) / 32, lin = blockIdx.x >> 3, vt = lin % nv, bh = (lin / nv) * 8 + (blockIdx.x & 7);
    if (bh >= a.B * nh) return;
    const int b = bh / nh, hl = bh - b * nh, h = h0 + hl, per = a.H / a.G, D = a.D, Dv = a.Dv;
    const int first = a.req[4 * b], n = a.req[4 * b + 1], pos0 = a.req[4 * b + 2], slot = a.req[4 * b + 3];
    if (n <= 0) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5, col = 32 * vt + l32, ti = wave & 1;
    const dk_sizes z = dk_layout(DP, Dv);
    const float *heads = a.scratch + (int64_t)hl * z.head, *groups = a.scratch + (int64_t)a.chunks * nh * z.head + (int64_t)(hl / per) * z.group;
    const int64_t head_step = nh * z.head, group_step = (nh / per) * z.group;
    auto head_of = [&](int c) { return heads + (int64_t)c * head_step; };
    auto group_of = [&](int c) { return groups + (int64_t)c * group_step; };
    auto after = [&](int c) { return c + 1 < first + n ? c + 1 : c; };      // every operand's successor sets out when it has been used: a whole chunk ahead, in its registers
    auto unit_of = [&](const float *p, int u) { return ((const float4 *)p + u * 64)[(uint32_t)lane]; };
    auto four = [](const dk_f32x16 &v, int y) { return make_float4(v[4 * y], v[4 * y + 1], v[4 * y + 2], v[4 * y + 3]); };
    auto put = [&](jl_bf16x8 *to, int s, const dk_terms &v) {
#pragma unroll
        for (int x = 0; x < 3; ++x) to[(3 * s + x) * 64 + lane] = v.t[x];
    };
    auto get = [&](const jl_bf16x8 *from, int s) {
        dk_terms v;
#pragma unroll
        for (int x = 0; x < 3; ++x) v.t[x] = from[(3 * s + x) * 64 + lane];
        return v;
    };
    if (wave >= 4) {                                                // rows 32 (wave - 4) .. of S
        const int w = wave - 4;
        float *sp = a.state + ((int64_t)slot * a.H + h) * D * Dv;
        dk_f32x16 S;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int d = 32 * w + 8 * (r >> 2) + 4 * hi + (r & 3);
            S[r] = d < D && col < Dv && pos0 > 0 ? sp[(int64_t)d * Dv + col] : 0.f;
        }
        auto share = [&]() {
#pragma unroll
            for (int y = 0; y < 2; ++y) put(Sf, 2 * w + y, dk_split(four(S, 2 * y), four(S, 2 * y + 1)));
        };
        share();
        float4 fk[8], sc[8];                                        // keys, and what is left of a token's correction at the chunk's end
        float gend;
        auto fetch = [&](int c) {
            const float *k = group_of(c);
            const float *e = head_of(c) + z.p + 3 * 1024;
#pragma unroll
            for (int y = 0; y < 8; ++y) { fk[y] = unit_of(k, DP / 4 + 8 * w + y); sc[y] = ((const float4 *)(e + DK_T) + 2 * y)[(uint32_t)hi]; }
            gend = e[DK_T - 1];
        };
        fetch(first);
        for (int c = first; c < first + n; ++c) {
            __syncthreads();                                        // S is there, U has been read
            dk_terms k[4];
#pragma unroll
            for (int y = 0; y < 8; ++y) fk[y] = make_float4(fk[y].x * sc[y].x, fk[y].y * sc[y].y, fk[y].z * sc[y].z, fk[y].w * sc[y].w);
#pragma unroll
            for (int y = 0; y < 4; ++y) k[y] = dk_split(fk[2 * y], fk[2 * y + 1]);
            const float end = gend;
            fetch(after(c));
            dk_sums sum;
            dk_clear(sum);
            __syncthreads();                                        // U is there, S has been read
#pragma unroll
            for (int y = 0; y < 4; ++y) dk_mma_split(k[y], get(Uf, y), sum);
            const dk_f32x16 more = dk_total(sum);
#pragma unroll
            for (int r = 0; r < 16; ++r) S[r] = fmaf(S[r], end, more[r]);
            const int none = min(noneS[0][l32], noneS[1][l32]);
            if (__any(none < DK_T))                                 // U has zeros instead
#pragma unroll
                for (int r = 0; r < 16; ++r) S[r] = none < DK_T ? NAN : S[r];
            share();
        }
        __syncthreads();                                            // the last outputs' pairs are there
        if (col < Dv)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int d = 32 * w + 8 * (r >> 2) + 4 * hi + (r & 3);
                if (d < D) sp[(int64_t)d * Dv + col] = S[r];
            }
        return;
    }
    const bool maker = wave < 2;
    float4 fa[NU];                                                  // what U, or the outputs, take of S
    auto taken = [&](int c) { return (maker ? head_of(c) + z.w2 : group_of(c)) + ti * NU * 256; };
    {
        const float *q = taken(first);
#pragma unroll
        for (int u = 0; u < NU; ++u) fa[u] = unit_of(q, u);
    }
    dk_terms f[2];
    // Short sums that start from nothing, then met: what 128 products in a row lose, or as many onto a W1 larger than they are, is more than the lanes of the other forms do
    auto product = [&](const float *next) {                        // f[0] is there already
        dk_sums sum;
        dk_clear(sum);
        dk_terms s1 = get(Sf, 0);
#pragma unroll
        for (int s = 0; s < NU / 2; ++s) {
            const dk_terms s0 = s1;
            if (s + 1 < NU / 2) {
                s1 = get(Sf, s + 1);
                f[(s + 1) & 1] = dk_split(fa[2 * s + 2], fa[2 * s + 3]);
            }
            fa[2 * s] = unit_of(next, 2 * s);
            fa[2 * s + 1] = unit_of(next, 2 * s + 1);
            dk_mma_split(f[s & 1], s0, sum);
#pragma unroll
            for (int i = 0; i < 6; ++i) {                           // a matrix instruction, and what the next step needs meanwhile
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return dk_total(sum);
    };
    if (maker) {
        float4 w1[4], fp[8];                                        // fp: the pairs
        auto fetch = [&](int c) {
#pragma unroll
            for (int y = 0; y < 4; ++y) w1[y] = unit_of(head_of(c) + z.w1, (vt * 2 + ti) * 4 + y);
        };
        auto fetch_pairs = [&](int c) {
#pragma unroll
            for (int y = 0; y < 8; ++y) fp[y] = unit_of(head_of(c) + z.p, 4 * ti + y);      // the first half's upper four are not used
        };
        fetch(first);
        fetch_pairs(first);
        for (int c = first; c < first + n; ++c) {
            f[0] = dk_split(fa[0], fa[1]);
            __syncthreads();                                        // S is there, U has been read
            dk_f32x16 u = product(taken(after(c)));
#pragma unroll
            for (int r = 0; r < 16; ++r) u[r] += ((const float *)&w1[r >> 2])[r & 3];
            fetch(after(c));
            float zero[4] = {0.f, 0.f, 0.f, 0.f};                   // not a number if a correction is not finite
#pragma unroll
            for (int r = 0; r < 16; ++r) zero[r & 3] = fmaf(u[r], 0.f, zero[r & 3]);
            int none = DK_T;
            if (__any((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.f)) {      // the outputs of the tokens in front of it must not meet it
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (!__builtin_isfinite(u[r])) { u[r] = 0.f; none = min(none, 32 * ti + 8 * (r >> 2) + 4 * hi + (r & 3)); }
                none = min(none, __shfl_xor(none, 32, 64));
            }
            if (hi == 0) noneS[ti][l32] = none;
#pragma unroll
            for (int y = 0; y < 2; ++y) put(Uf, 2 * ti + y, dk_split(four(u, 2 * y), four(u, 2 * y + 1)));
            __syncthreads();                                        // U is there, S has been read
            dk_sums sum;
            dk_clear(sum);
#pragma unroll
            for (int y = 0; y < 4; ++y)
                if (y < 2 || ti) dk_mma_split(dk_split(fp[2 * y], fp[2 * y + 1]), get(Uf, y), sum);
            fetch_pairs(after(c));
            const dk_f32x16 o = dk_total(sum);
#pragma unroll
            for (int y = 0; y < 4; ++y) Pf[(4 * ti + y) * 64 + lane] = four(o, y);
        }
        __syncthreads();                                            // the last outputs' pairs are there
        return;
    }
    float4 sc[4];                                                   // what is left of S at a token
    auto fetch = [&](int c) {
#pragma unroll
        for (int y = 0; y < 4; ++y) sc[y] = ((const float4 *)(head_of(c) + z.p + 3 * 1024 + 32 * ti) + 2 * y)[(uint32_t)hi];
    };
    fetch(first);
    // A chunk's outputs are stored while the next one's state is made.  Always 16 stores, those of tokens and columns that do not exist beyond the buffer's end: were their number
    // not known, the next operand's loads, which came before them, could only be waited for together with them
    dk_f32x16 o, done;
#pragma unroll
    for (int r = 0; r < 16; ++r) o[r] = 0.f;
    int none = DK_T, none_done, row0 = 0, cnt = 0;
    const int ld = a.H * Dv;
    auto add_pairs = [&]() {
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const float4 p = Pf[(4 * ti + y) * 64 + lane];
            done[4 * y] = o[4 * y] + p.x;
            done[4 * y + 1] = o[4 * y + 1] + p.y;
            done[4 * y + 2] = o[4 * y + 2] + p.z;
            done[4 * y + 3] = o[4 * y + 3] + p.w;
        }
        none_done = none;
    };
    auto store = [&]() {
        if constexpr (WIDE) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int t = 32 * ti + 8 * (r >> 2) + 4 * hi + (r & 3);
                if (t < cnt && col < Dv) raw[((int64_t)(row0 + t) * a.H + h) * Dv + col] = t < none_done ? done[r] : NAN;
            }
            return;
        }
        const auto to = __builtin_amdgcn_make_buffer_rsrc(raw + ((int64_t)row0 * a.H + h) * Dv, 0, cnt * ld * 4, 0x00020000);
        const int t0 = 32 * ti + 4 * hi;
        uint32_t at = col < Dv ? (uint32_t)(t0 * ld + col) * 4 : 0x80000000u;
        asm("" : "+v"(at));                                         // not sixteen offsets kept over the loop
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int x = 8 * (r >> 2) + (r & 3);
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, t0 + x < none_done ? done[r] : NAN), to, at + x * ld * 4, 0, 0);
        }
    };
    for (int c = first; c < first + n; ++c) {
        f[0] = dk_split(fa[0], fa[1]);
        __syncthreads();                                            // S is there, U has been read, the pairs' part of the last outputs is there
        add_pairs();
        __builtin_amdgcn_sched_barrier(0);
        o = product(taken(after(c)));
#pragma unroll
        for (int r = 0; r < 16; ++r) o[r] *= ((const float *)&sc[r >> 2])[r & 3];
        fetch(after(c));
        __syncthreads();                                            // U is there, S has been read
        store();                                                    // at first of no tokens
        none = min(noneS[0][l32], noneS[1][l32]);
        row0 = __builtin_amdgcn_readfirstlane(a.chunk_rec[4 * c]);
        cnt = __builtin_amdgcn_readfirstlane(a.chunk_rec[4 * c + 1]);
    }
    __syncthreads();                                                // the last outputs' pairs are there
    add_pairs();
    store();
}

template <typename T, int DMAX>
static int delta_cols_launch(const void *qkv, int64_t qkv_ld, int q_col, int k_col, int v_col, const void *proj, int64_t ld, int a_col, int b_col, int g_col,
                             const float *A_log, const float *dt_bias, const float *norm_w, const int32_t *seq, int B, int64_t N, int H, int G, int D, int Dv,
                             float unit_eps, float q_scale, float eps, float *state, float *raw, void *out, hipStream_t st) {
    constexpr int LPC = DMAX >= 128 ? 8 : 4;            // 16 or 32 rows of a column per lane
    const dim3 grid((unsigned)(B * H), (unsigned)((Dv + 64 / LPC - 1) / (64 / LPC)));
    delta_cols_kernel<T, DMAX, LPC><<<grid, 64, 0, st>>>((const float *)qkv, qkv_ld, q_col, k_col, v_col, (const T *)proj, ld, a_col, b_col, A_log, dt_bias, seq, H, G,
                                                         D, Dv, unit_eps, q_scale, state, raw);
    int rc = jl_check_launch("delta_cols_kernel");
    if (rc != JL_OK) return rc;
    return delta_out_launch<T>(raw, proj, ld, g_col, norm_w, N * H, H, Dv, eps, out, st);
}

template <typename T, typename TQ, int DMAX, int LPC>
static int delta_launch(const void *qkv, int64_t qkv_ld, int q_col, int k_col, int v_col, const void *proj, int64_t ld, int a_col, int b_col, int g_col,
                        const float *A_log, const float *dt_bias, const float *norm_w, const int32_t *seq, int B, int H, int G, int D, int Dv, float unit_eps,
                        float q_scale, float eps, float *state, void *out, hipStream_t st) {
    const int threads = (Dv * LPC + 63) / 64 * 64;
    const size_t lds = (size_t)(2 * DL_TT * DMAX + 2 * DL_TT + DL_TT * 16) * 4;
    delta_rule_kernel<T, TQ, DMAX, LPC><<<dim3((unsigned)(B * H)), threads, lds, st>>>((const TQ *)qkv, qkv_ld, q_col, k_col, v_col, (const T *)proj, ld, a_col,
                                                                                      b_col, g_col, A_log, dt_bias, norm_w, seq, H, G, D, Dv, unit_eps,
                                                                                      q_scale, eps, state, (T *)out);
    return jl_check_launch("delta_rule_kernel");
}

extern "C" int jl_delta_rule(const void *qkv, int qkv_dtype, int64_t qkv_ld, int32_t q_col, int32_t k_col, int32_t v_col, const void *proj, int dtype,
                             int64_t ld, int32_t a_col, int32_t b_col, int32_t g_col, const float *A_log, const float *dt_bias, const float *norm_w,
                             const int32_t *seq, int32_t B, int64_t N, int32_t H, int32_t G, int32_t D, int32_t Dv, float unit_eps, float q_scale, float eps,
                             float *state, float *raw, void *out, void *stream) {
    if (B <= 0) return JL_OK;
    if (!qkv || !proj || !A_log || !dt_bias || !norm_w || !seq || !state || !out) return jl_fail(JL_E_INVALID, "jl_delta_rule: null pointer");
    if (H <= 0 || G <= 0 || H % G || D <= 0 || D > 256 || Dv <= 0 || Dv > 1024)
        return jl_fail(JL_E_INVALID, "jl_delta_rule: heads must be a multiple of the key heads, D <= 256, Dv <= 1024");
    if (q_col < 0 || k_col < 0 || v_col < 0 || a_col < 0 || b_col < 0 || g_col < 0 || q_col + (int64_t)G * D > qkv_ld || k_col + (int64_t)G * D > qkv_ld ||
        v_col + (int64_t)H * Dv > qkv_ld || a_col + (int64_t)H > ld || b_col + (int64_t)H > ld || g_col + (int64_t)H * Dv > ld)
        return jl_fail(JL_E_INVALID, "jl_delta_rule: columns do not fit the rows");
    hipStream_t st = (hipStream_t)stream;
    if (raw) {                                          // long portions: the state's columns shared out over single-wavefront workgroups
        if (qkv_dtype != JL_F32 || N <= 0) return jl_fail(JL_E_INVALID, "jl_delta_rule: q, k, v after their convolution are float; N rows of scratch");
#define DC_CASE(DM) JL_DISPATCH(dtype, return (delta_cols_launch<T, DM>(qkv, qkv_ld, q_col, k_col, v_col, proj, ld, a_col, b_col, g_col, A_log, dt_bias, norm_w, \
                                                                         seq, B, N, H, G, D, Dv, unit_eps, q_scale, eps, state, raw, out, st)))
        if (D <= 64) DC_CASE(64);
        else if (D <= 128) DC_CASE(128);
        else DC_CASE(256);
#undef DC_CASE
    }
    const int lpc = Dv * 4 <= 1024 ? 4 : 1;             // four lanes per column while the workgroup holds them
#define DL_ARGS qkv, qkv_ld, q_col, k_col, v_col, proj, ld, a_col, b_col, g_col, A_log, dt_bias, norm_w, seq, B, H, G, D, Dv, unit_eps, q_scale, eps, state, out, st
#define DL_CASE(N)                                                                                                        \
    do {                                                                                                                  \
        if (dtype == JL_BF16 && qkv_dtype == JL_F32) return lpc == 4 ? delta_launch<bf16_t, float, N, 4>(DL_ARGS) : delta_launch<bf16_t, float, N, 1>(DL_ARGS); \
        if (dtype == JL_F32 && qkv_dtype == JL_F32) return lpc == 4 ? delta_launch<float, float, N, 4>(DL_ARGS) : delta_launch<float, float, N, 1>(DL_ARGS);   \
        return jl_fail(JL_E_INVALID, "jl_delta_rule: q, k, v after their convolution are float");                          \
    } while (0)
    if (D <= 64) DL_CASE(64);
    else if (D <= 128) DL_CASE(128);
    else DL_CASE(256);
#undef DL_CASE
#undef DL_ARGS
    return JL_OK;
}

extern "C" int jl_delta_chunks_ok(int32_t D, int32_t Dv) { return D > 0 && D <= 128 && D % 4 == 0 && Dv > 0 && Dv <= 1024; }

// heads come in whole key groups
extern "C" int64_t jl_delta_chunks_floats(int32_t chunks, int32_t heads, int32_t H, int32_t G, int32_t D, int32_t Dv) {
    if (chunks <= 0 || heads <= 0 || G <= 0 || H <= 0 || H % G || !jl_delta_chunks_ok(D, Dv)) return 0;
    const dk_sizes z = dk_layout(D <= 64 ? 64 : 128, Dv);
    return (int64_t)chunks * (heads * z.head + heads / (H / G) * z.group);
}

template <typename T, int DP> static int delta_chunks_launch(const jl_delta_chunks &a, hipStream_t st) {
    const size_t lds = (size_t)(2 * DK_T * DP + 3 * 1024 + 3 * DK_T) * 4 + DK_T * 8;
    auto chunk = a.qkv_ld > 1 << 26 ? delta_chunk_kernel<T, DP, true> : delta_chunk_kernel<T, DP, false>;
    hipError_t e = hipFuncSetAttribute((const void *)chunk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return jl_fail(JL_E_LAUNCH, "jl_delta_chunks_run: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    const int nv = (a.Dv + 31) / 32;
    const bool wide = (int64_t)a.H * a.Dv > 1 << 22;                 // 2 GiB of 64 rows and what lies behind them
    for (int h0 = 0; h0 < a.H; h0 += a.pass_heads) {                 // as many heads at a time as the scratch holds
        const int nh = a.H - h0 < a.pass_heads ? a.H - h0 : a.pass_heads;
        chunk<<<dim3((unsigned)nh * (unsigned)a.chunks), 256, lds, st>>>(a, h0, nh);
        (wide ? delta_chain_kernel<DP, true> : delta_chain_kernel<DP, false>)<<<dim3((unsigned)((a.B * nh + 7) / 8 * nv * 8)), 256 + 2 * DP, 0, st>>>(a, h0, nh, a.raw);
    }
    int rc = jl_check_launch("delta_chunk_kernel");
    if (rc != JL_OK) return rc;
    return a.out ? delta_out_launch<T>(a.raw, a.proj, a.ld, a.g_col, a.norm_w, a.N * a.H, a.H, a.Dv, a.eps, a.out, st) : JL_OK;
}

extern "C" int jl_delta_chunks_run(const jl_delta_chunks *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_delta_chunks_run: null arguments");
    const jl_delta_chunks &a = *ap;
    if (a.B <= 0 || a.chunks <= 0) return JL_OK;
    if (!a.qkv || !a.proj || !a.A_log || !a.dt_bias || !a.norm_w || !a.chunk_rec || !a.req || !a.state || !a.scratch || !a.raw)
        return jl_fail(JL_E_INVALID, "jl_delta_chunks_run: null pointer");
    if (!jl_delta_chunks_ok(a.D, a.Dv) || a.H <= 0 || a.G <= 0 || a.H % a.G || a.N <= 0 || (int64_t)a.chunks * a.H > INT32_MAX / 256 || a.pass_heads <= 0 || a.pass_heads % (a.H / a.G) || a.qkv_ld % 4 ||
        (a.q_col | a.k_col) % 4 || (((uintptr_t)a.qkv | (uintptr_t)a.scratch) & 15) || (a.dtype != JL_BF16 && a.dtype != JL_F32))
        return jl_fail(JL_E_INVALID, "jl_delta_chunks_run: sizes, columns or alignment (ask jl_delta_chunks_ok)");
    if (a.q_col < 0 || a.k_col < 0 || a.v_col < 0 || a.a_col < 0 || a.b_col < 0 || a.g_col < 0 || a.q_col + (int64_t)a.G * a.D > a.qkv_ld || a.k_col + (int64_t)a.G * a.D > a.qkv_ld ||
        a.v_col + (int64_t)a.H * a.Dv > a.qkv_ld || a.a_col + (int64_t)a.H > a.ld || a.b_col + (int64_t)a.H > a.ld || a.g_col + (int64_t)a.H * a.Dv > a.ld)
        return jl_fail(JL_E_INVALID, "jl_delta_chunks_run: columns do not fit the rows");
    if (a.scratch_floats < jl_delta_chunks_floats(a.chunks, a.pass_heads < a.H ? a.pass_heads : a.H, a.H, a.G, a.D, a.Dv))
        return jl_fail(JL_E_INVALID, "jl_delta_chunks_run: scratch is too small");
    JL_DISPATCH(a.dtype, return a.D <= 64 ? delta_chunks_launch<T, 64>(a, (hipStream_t)stream) : delta_chunks_launch<T, 128>(a, (hipStream_t)stream));
    return JL_OK;
}
