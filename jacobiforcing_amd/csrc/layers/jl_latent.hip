// jl_latent.hip — attention through a low-rank latent: the pool holds, per token, the normalised key/value latent and one rotary
// key part shared by all heads; queries are brought into the pool's coordinates (the key up-projection is applied to the query),
// attention runs over the pool with one key/value "head", and the value up-projection follows.  This file: the norms, rotations and
// packing around the library products, and for steps of few tokens the products themselves.
#include "jl_common.h"

__device__ __forceinline__ float rot_half(const float *v, int d, int rot_dims, const float *cs, const float *sn, int pairing) {
    // value of dimension d of the rotated vector; v the unrotated vector (float, in LDS or registers)
    const int half = rot_dims >> 1;
    if (d >= rot_dims) return v[d];
    if (pairing == JL_ROT_NEIGHBOURS) {                         // dimension 2i pairs with 2i + 1
        const int i = d >> 1;
        return (d & 1) ? v[d] * cs[i] + v[d - 1] * sn[i] : v[d] * cs[i] - v[d + 1] * sn[i];
    }
    if (d < half) return v[d] * cs[d] - v[d + half] * sn[d];
    return v[d] * cs[d - half] + v[d - half] * sn[d - half];
}

template <typename T>
__global__ __launch_bounds__(256) void latent_prep_kernel(const T *__restrict__ proj, int64_t ld, int q_col, int Rq, int kv_col, int R, int rd,
                                                           int rot_dims, const T *__restrict__ wq, const T *__restrict__ wkv, float eps,
                                                           const int32_t *__restrict__ pos, const float *__restrict__ cos_t,
                                                           const float *__restrict__ sin_t, T *__restrict__ cq_out, T *__restrict__ pool,
                                                           const int64_t *__restrict__ slot, int pairing) {
    __shared__ float red[16];
    extern __shared__ float kr[];                               // [rd] the unrotated rotary key
    const int64_t n = blockIdx.x;
    const T *row = proj + n * ld;
    float sq = 0.f, sk = 0.f;
    for (int c = threadIdx.x; c < Rq; c += blockDim.x) { const float v = ld_f(row + q_col + c); sq += v * v; }
    if (pool) for (int c = threadIdx.x; c < R; c += blockDim.x) { const float v = ld_f(row + kv_col + c); sk += v * v; }
    if (pool) for (int c = threadIdx.x; c < rd; c += blockDim.x) kr[c] = ld_f(row + kv_col + R + c);
    sq = block_sum_f32(sq, red);
    sk = block_sum_f32(sk, red);                                // its barriers also publish kr
    const float rq = Rq > 0 ? 1.0f / sqrtf(sq / (float)Rq + eps) : 0.f, rk = pool ? 1.0f / sqrtf(sk / (float)R + eps) : 0.f;
    for (int c = threadIdx.x; c < Rq; c += blockDim.x) st_f(cq_out + n * Rq + c, ld_f(row + q_col + c) * rq * ld_f(wq + c));
    if (!pool) return;
    const int64_t sl = slot[n];
    if (sl < 0) return;
    T *dst = pool + sl * (int64_t)(R + rd);
    for (int c = threadIdx.x; c < R; c += blockDim.x) st_f(dst + c, ld_f(row + kv_col + c) * rk * ld_f(wkv + c));
    const float *cs = cos_t + (int64_t)pos[n] * (rot_dims >> 1), *sn = sin_t + (int64_t)pos[n] * (rot_dims >> 1);
    for (int c = threadIdx.x; c < rd; c += blockDim.x) st_f(dst + R + c, rot_half(kr, c, rot_dims, cs, sn, pairing));
}

// The same with four values per load and thread, kept in registers between the two passes, and one pass of sums for both latents.  us, one value at a time / four: 8192 rows of 768 + 512 + 64
// 28.2 / 18.5 (their bytes 8.5); of 384 + 256 + 64 18.7 / 10.7; 32 rows 5.0 / 3.8.
constexpr int LP_UNITS = 2;                                          // of four values per thread and latent
template <typename T>
__global__ __launch_bounds__(256) void latent_prep_vec_kernel(const T *__restrict__ proj, int64_t ld, int q_col, int Rq, int kv_col, int R, int rd, int rot_dims, const T *__restrict__ wq,
                                                              const T *__restrict__ wkv, float eps, const int32_t *__restrict__ pos, const float *__restrict__ cos_t,
                                                              const float *__restrict__ sin_t, T *__restrict__ cq_out, T *__restrict__ pool, const int64_t *__restrict__ slot, int pairing) {
    __shared__ float red[2][4];
    extern __shared__ float kr[];                                    // [rd] the unrotated rotary key
    const int64_t n = blockIdx.x;
    const int tid = threadIdx.x, step = blockDim.x * 4, waves = blockDim.x >> 6;
    const T *row = proj + n * ld;
    float q[LP_UNITS][4], k[LP_UNITS][4], sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < LP_UNITS; ++i) {
        const int c = i * step + tid * 4;
        if (c < Rq) ld4_f(row + q_col + c, q[i]);
        if (pool && c < R) ld4_f(row + kv_col + c, k[i]);
    }
    if (pool) for (int c = tid; c < rd; c += blockDim.x) kr[c] = ld_f(row + kv_col + R + c);
    const int64_t sl = pool ? slot[n] : -1;
#pragma unroll
    for (int i = 0; i < LP_UNITS; ++i) {
        const int c = i * step + tid * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (c < Rq) sq += q[i][e] * q[i][e];
            if (pool && c < R) sk += k[i][e] * k[i][e];
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) { sq += __shfl_xor(sq, off, 64); sk += __shfl_xor(sk, off, 64); }
    if ((tid & 63) == 0) { red[0][tid >> 6] = sq; red[1][tid >> 6] = sk; }
    __syncthreads();
    sq = red[0][0]; sk = red[1][0];
    for (int i = 1; i < waves; ++i) { sq += red[0][i]; sk += red[1][i]; }
    const float rq = Rq > 0 ? 1.0f / sqrtf(sq / (float)Rq + eps) : 0.f, rk = pool ? 1.0f / sqrtf(sk / (float)R + eps) : 0.f;
    T *dst = pool + (sl < 0 ? 0 : sl) * (int64_t)(R + rd);
#pragma unroll
    for (int i = 0; i < LP_UNITS; ++i) {
        const int c = i * step + tid * 4;
        float w[4];
        if (c < Rq) {
            ld4_f(wq + c, w);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] *= q[i][e] * rq;
            st4_f(cq_out + n * Rq + c, w);
        }
        if (sl >= 0 && c < R) {
            ld4_f(wkv + c, w);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] *= k[i][e] * rk;
            st4_f(dst + c, w);
        }
    }
    if (sl < 0) return;
    const float *cs = cos_t + (int64_t)pos[n] * (rot_dims >> 1), *sn = sin_t + (int64_t)pos[n] * (rot_dims >> 1);
    for (int c = tid; c < rd; c += blockDim.x) st_f(dst + R + c, rot_half(kr, c, rot_dims, cs, sn, pairing));
}

extern "C" int jl_latent_prep(const void *proj, int dtype, int64_t N, int64_t ld, int32_t q_col, int32_t Rq, int32_t kv_col, int32_t R,
                              int32_t rd, int32_t rot_dims, const void *wq, const void *wkv, float eps, const int32_t *pos,
                              const float *cos_t, const float *sin_t, int64_t table_len, void *cq_out, void *pool, const int64_t *slot,
                              int32_t pairing, void *stream) {
    if (N <= 0) return JL_OK;
    if (!proj || !pos || (pool && (!wkv || !slot)) || (Rq > 0 && (!wq || !cq_out)) || (!pool && Rq <= 0)) return jl_fail(JL_E_INVALID, "jl_latent_prep: null pointer");
    if (!pool) { R = rd = rot_dims = 0; kv_col = 0; }
    if (pairing != JL_ROT_HALVES && pairing != JL_ROT_NEIGHBOURS) return jl_fail(JL_E_INVALID, "jl_latent_prep: unknown pairing %d", pairing);
    if (Rq < 0 || (pool && R <= 0) || rd < 0 || q_col + (int64_t)Rq > ld || kv_col + (int64_t)R + rd > ld)
        return jl_fail(JL_E_INVALID, "jl_latent_prep: columns do not fit the row stride");
    if (rot_dims < 0 || rot_dims > rd || (rot_dims & 1) || (rot_dims && (!cos_t || !sin_t || table_len <= 0)))
        return jl_fail(JL_E_INVALID, "jl_latent_prep: rot_dims must be even, at most rd, with angle tables");
    // narrow rows (a few hundred values per token): one wavefront per token instead of four, of which three would idle
    const int threads = (int64_t)Rq + R + rd <= 512 ? 64 : 256;
    auto al = [&](const void *q) { return ((uintptr_t)q % (dtype == JL_BF16 ? 8 : 16)) == 0; };
    const int units = ((Rq > R ? Rq : R) + 3) / 4, wide = units <= 64 ? 64 : units <= 128 ? 128 : 256;
    if ((ld | q_col | kv_col | Rq | R | rd) % 4 == 0 && units <= LP_UNITS * wide && al(proj) && al(wq) && al(wkv) && al(cq_out) && al(pool)) {
        JL_DISPATCH(dtype, latent_prep_vec_kernel<T><<<dim3((unsigned)N), wide, (size_t)(rd > 0 ? rd : 1) * 4, (hipStream_t)stream>>>(
                               (const T *)proj, ld, q_col, Rq, kv_col, R, rd, rot_dims, (const T *)wq, (const T *)wkv, eps, pos, cos_t, sin_t, (T *)cq_out, (T *)pool, slot, pairing));
        return jl_check_launch("latent_prep_vec_kernel");
    }
    JL_DISPATCH(dtype, latent_prep_kernel<T><<<dim3((unsigned)N), threads, (size_t)(rd > 0 ? rd : 1) * 4, (hipStream_t)stream>>>(
                           (const T *)proj, ld, q_col, Rq, kv_col, R, rd, rot_dims, (const T *)wq, (const T *)wkv, eps, pos, cos_t, sin_t,
                           (T *)cq_out, (T *)pool, slot, pairing));
    return jl_check_launch("latent_prep_kernel");
}

// one workgroup per token: q_out[n, h] = [qa[h, n, :R] | rotate(q[n, h, D:])]
template <typename T>
__global__ __launch_bounds__(256) void latent_q_pack_kernel(const T *__restrict__ qa, const T *__restrict__ q, int64_t q_ld, int64_t N, int H, int D, int R, int rd,
                                                             int rot_dims, const int32_t *__restrict__ pos, const float *__restrict__ cos_t,
                                                             const float *__restrict__ sin_t, T *__restrict__ q_out, int pairing) {
    extern __shared__ float qr[];                               // [H][rd]
    const int64_t n = blockIdx.x;
    const int Dq = D + rd, Do = R + rd;
    for (int e = threadIdx.x; e < H * rd; e += 256) { const int h = e / rd, c = e - h * rd; qr[e] = ld_f(q + n * q_ld + (int64_t)h * Dq + D + c); }
    for (int e = threadIdx.x; e < H * R; e += 256) {
        const int h = e / R, c = e - h * R;
        q_out[(n * H + h) * Do + c] = qa[((int64_t)h * N + n) * R + c];
    }
    __syncthreads();
    const float *cs = cos_t + (int64_t)pos[n] * (rot_dims >> 1), *sn = sin_t + (int64_t)pos[n] * (rot_dims >> 1);
    for (int e = threadIdx.x; e < H * rd; e += 256) {
        const int h = e / rd, c = e - h * rd;
        st_f(q_out + (n * H + h) * Do + R + c, rot_half(qr + h * rd, c, rot_dims, cs, sn, pairing));
    }
}

extern "C" int jl_latent_q_pack(const void *qa, const void *q, int64_t q_ld, int dtype, int64_t N, int32_t H, int32_t D, int32_t R, int32_t rd,
                                int32_t rot_dims, const int32_t *pos, const float *cos_t, const float *sin_t, int64_t table_len, void *q_out,
                                int32_t pairing, void *stream) {
    if (N <= 0) return JL_OK;
    if (!qa || !q || !pos || !q_out || H <= 0 || D < 0 || R <= 0 || rd < 0 || q_ld < (int64_t)H * (D + rd))
        return jl_fail(JL_E_INVALID, "jl_latent_q_pack: null pointer or bad sizes");
    if (pairing != JL_ROT_HALVES && pairing != JL_ROT_NEIGHBOURS) return jl_fail(JL_E_INVALID, "jl_latent_q_pack: unknown pairing %d", pairing);
    if (rot_dims < 0 || rot_dims > rd || (rot_dims & 1) || (rot_dims && (!cos_t || !sin_t || table_len <= 0)))
        return jl_fail(JL_E_INVALID, "jl_latent_q_pack: rot_dims must be even, at most rd, with angle tables");
    const size_t lds = (size_t)(H * rd > 0 ? H * rd : 1) * 4;
    if (lds > 48 * 1024) return jl_fail(JL_E_INVALID, "jl_latent_q_pack: %d heads x %d rotary dimensions exceed the kernel's LDS", H, rd);
    JL_DISPATCH(dtype, latent_q_pack_kernel<T><<<dim3((unsigned)N), 256, lds, (hipStream_t)stream>>>((const T *)qa, (const T *)q, q_ld, N, H, D, R, rd, rot_dims,
                                                                                                   pos, cos_t, sin_t, (T *)q_out, pairing));
    return jl_check_launch("latent_q_pack_kernel");
}

// q[n, h, D + d] for d < rot_dims <- rotated, in place: a thread owns a pair.  A workgroup of 256 walks 256 / half heads of consecutive rows at a time; what
// it moves is the rotary columns only (8 192 rows x 16 heads x 64 of 192 columns: 9 us).
template <typename T>
__global__ __launch_bounds__(256) void rotate_heads_kernel(T *__restrict__ q, int64_t N, int64_t ld, int H, int D, int rd, int rot_dims, const int32_t *__restrict__ pos,
                                                            const float *__restrict__ cos_t, const float *__restrict__ sin_t, int pairing) {
    const int half = rot_dims >> 1, per_row = H * half;
    for (int64_t n = blockIdx.x; n < N; n += gridDim.x) {
        const float *cs = cos_t + (int64_t)pos[n] * half, *sn = sin_t + (int64_t)pos[n] * half;
        T *row = q + n * ld + D;
        for (int e = threadIdx.x; e < per_row; e += 256) {
            const int h = e / half, i = e - h * half;
            T *v = row + (int64_t)h * (D + rd);
            const int x = pairing == JL_ROT_NEIGHBOURS ? 2 * i : i, y = pairing == JL_ROT_NEIGHBOURS ? 2 * i + 1 : i + half;
            const float a = ld_f(v + x), b = ld_f(v + y);
            st_f(v + x, a * cs[i] - b * sn[i]);
            st_f(v + y, b * cs[i] + a * sn[i]);
        }
    }
}

// four neighbouring pairs per thread, where halves and heads start at borders of four values (8192 rows x 16 heads x 64 of 192 columns, a pair / four per thread: 11.3 / 8.5 us; 1207 rows 3.5 / 3.2)
template <typename T>
__global__ __launch_bounds__(256) void rotate_heads_vec_kernel(T *__restrict__ q, int64_t N, int64_t ld, int H, int D, int rd, int rot_dims, const int32_t *__restrict__ pos,
                                                                const float *__restrict__ cos_t, const float *__restrict__ sin_t, int pairing) {
    const int half = rot_dims >> 1, per_head = half >> 2, per_row = H * per_head;
    const int64_t total = N * per_row;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int64_t n = e / per_row;
        const int r = (int)(e - n * per_row), h = r / per_head, i = 4 * (r - h * per_head);
        T *v = q + n * ld + (int64_t)h * (D + rd) + D;
        const bool near = pairing == JL_ROT_NEIGHBOURS;
        T *const pa = v + (near ? 2 * i : i), *const pb = v + (near ? 2 * i + 4 : i + half);
        float a[4], b[4], c[4], s[4];
        ld4_f(pa, a);
        ld4_f(pb, b);
        const int64_t at = (int64_t)pos[n] * half + i;
        ld4_f(cos_t + at, c);
        ld4_f(sin_t + at, s);
        float x[4], y[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {                                // near: values 2k and 2k + 1 of the eight
            const float u = !near ? a[k] : k < 2 ? a[(2 * k) & 3] : b[(2 * k) & 3], w = !near ? b[k] : k < 2 ? a[(2 * k + 1) & 3] : b[(2 * k + 1) & 3];
            x[k] = u * c[k] - w * s[k];
            y[k] = w * c[k] + u * s[k];
        }
        if (near) {
            const float lo[4] = {x[0], y[0], x[1], y[1]}, up[4] = {x[2], y[2], x[3], y[3]};
            st4_f(pa, lo);
            st4_f(pb, up);
        } else {
            st4_f(pa, x);
            st4_f(pb, y);
        }
    }
}

extern "C" int jl_rotate_heads(void *q, int dtype, int64_t N, int64_t ld, int32_t H, int32_t D, int32_t rd, int32_t rot_dims, const int32_t *pos, const float *cos_t,
                               const float *sin_t, int64_t table_len, int32_t pairing, void *stream) {
    if (N <= 0 || rot_dims == 0) return JL_OK;
    if (!q || !pos || !cos_t || !sin_t || table_len <= 0 || H <= 0 || D < 0 || rd <= 0 || ld < (int64_t)H * (D + rd)) return jl_fail(JL_E_INVALID, "jl_rotate_heads: null pointer or bad sizes");
    if (rot_dims < 0 || rot_dims > rd || (rot_dims & 1)) return jl_fail(JL_E_INVALID, "jl_rotate_heads: rot_dims must be even and at most rd");
    if (pairing != JL_ROT_HALVES && pairing != JL_ROT_NEIGHBOURS) return jl_fail(JL_E_INVALID, "jl_rotate_heads: unknown pairing %d", pairing);
    if ((rot_dims % 8 | ld % 4 | D % 4 | rd % 4) == 0 && ((uintptr_t)q % (dtype == JL_BF16 ? 8 : 16) | (uintptr_t)cos_t % 16 | (uintptr_t)sin_t % 16) == 0) {
        const int64_t groups = (N * H * (rot_dims / 8) + 255) / 256;
        JL_DISPATCH(dtype, rotate_heads_vec_kernel<T><<<dim3((unsigned)(groups < 1 << 20 ? groups : 1 << 20)), 256, 0, (hipStream_t)stream>>>((T *)q, N, ld, H, D, rd, rot_dims, pos, cos_t, sin_t, pairing));
        return jl_check_launch("rotate_heads_vec_kernel");
    }
    JL_DISPATCH(dtype, rotate_heads_kernel<T><<<dim3((unsigned)(N < 65535 * 16 ? N : 65535 * 16)), 256, 0, (hipStream_t)stream>>>((T *)q, N, ld, H, D, rd, rot_dims, pos, cos_t,
                                                                                                                                sin_t, pairing));
    return jl_check_launch("rotate_heads_kernel");
}

template <typename T>
__global__ __launch_bounds__(256) void heads_gate_kernel(const T *__restrict__ ov, const T *__restrict__ gate, int64_t gate_ld, int64_t N, int H, int Dv,
                                                          T *__restrict__ out) {
    const int64_t n = blockIdx.x;
    for (int e = threadIdx.x; e < H * Dv; e += 256) {
        const int h = e / Dv, d = e - h * Dv;
        float v = ld_f(ov + ((int64_t)h * N + n) * Dv + d);
        if (gate) v *= 1.0f / (1.0f + expf(-ld_f(gate + n * gate_ld + e)));
        st_f(out + n * (int64_t)(H * Dv) + e, v);
    }
}

extern "C" int jl_heads_gate(const void *ov, const void *gate, int64_t gate_ld, int dtype, int64_t N, int32_t H, int32_t Dv, void *out,
                             void *stream) {
    if (N <= 0) return JL_OK;
    if (!ov || !out || H <= 0 || Dv <= 0 || (gate && gate_ld < (int64_t)H * Dv)) return jl_fail(JL_E_INVALID, "jl_heads_gate: null pointer or bad sizes");
    JL_DISPATCH(dtype, heads_gate_kernel<T><<<dim3((unsigned)N), 256, 0, (hipStream_t)stream>>>((const T *)ov, (const T *)gate, gate_ld, N, H, Dv, (T *)out));
    return jl_check_launch("heads_gate_kernel");
}

// ---- the per-head products on both sides of attention over the latent, few tokens (bfloat16): out[n, h] = x[n, h] W[h], with what follows it ---------------------------------------
// In front: queries by the key up-projection, straight into rows [latent | rotary part rotated] of the attention's queries.  Behind: latent outputs by the value up-projection, gated, the heads side by
// side.  Before, either was a batched library product, whose operands lie [H, N, ..], and a launch that put its rows in order: 24 and 5 us of the host; GPU time, 32 tokens of 16 heads
// of 128, latent 512: in front 14.7 / 7.7, behind 13.9 / 5.7; 1390 tokens of 8 heads of 64, latent 128: 13.5 / 6.7, 10.1 / 7.1.
// What bounds it is the way through one workgroup: W of a head comes in tiles of DEPTH x COLS (32 KB, every load on its way at once), x straight into the operands.  W is depth-major: it is turned by
// ds_read_b64_tr_b16 on its way out of LDS, whose rows are permuted so that a lane's eight depths are neighbours in x.  Four wavefronts share the columns where the depth is short (queries), the depth
// where the columns are few (outputs); W's columns are the rows of the result, so that a lane stores four neighbouring columns.
typedef float lh_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t lh_u32x4 __attribute__((ext_vector_type(4)));
typedef short lh_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) lh_s16x4 lh_lds_s16x4;

template <int WC>                                                    // wavefronts side by side over the columns; the others share the depth
__global__ __launch_bounds__(256, 2) void latent_heads_kernel(jl_latent_heads a) {
    constexpr int WK = 4 / WC, COLS = 32 * WC, DEPTH = 128 * WK, ROW = COLS + 16, PASS = 256 / (COLS / 8), LOADS = DEPTH / PASS;
    __shared__ __attribute__((aligned(16))) bf16_t tile[DEPTH * ROW];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5, wc = wave % WC, wk = wave / WC;
    const int col_blocks = (a.O + COLS - 1) / COLS, h = blockIdx.x / col_blocks, o0 = (blockIdx.x - h * col_blocks) * COLS, K = a.K, O = a.O;
    const int64_t n0 = (int64_t)blockIdx.y * 32, n = n0 + l32 < a.N ? n0 + l32 : a.N - 1;      // a row that does not exist repeats the last one and is not stored
    const bf16_t *x = (const bf16_t *)a.x + n * a.x_ld + (int64_t)h * a.x_head, *w = (const bf16_t *)a.w + (int64_t)h * K * O;
    const int row = tid / (COLS / 8), col = tid % (COLS / 8) * 8;
    const int tr_row = 4 * hi + ((lane & 15) >> 2), tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3) + 32 * wc;
    lh_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const lh_u32x4 zero = {0, 0, 0, 0};
    for (int k0 = 0; k0 < K; k0 += DEPTH) {
        lh_u32x4 v[LOADS], xv[8];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int d = k0 + row + i * PASS;
            v[i] = d < K && o0 + col < O ? *(const lh_u32x4 *)(w + (int64_t)d * O + o0 + col) : zero;
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int d = k0 + 128 * wk + 16 * s + 8 * hi;
            xv[s] = d < K ? *(const lh_u32x4 *)(x + d) : zero;
        }
        if (k0 > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int d = row + i * PASS, at = (d & ~15) | (d & 4) << 1 | (d & 8) >> 1 | (d & 3);      // depth 8 h + 4 y + i of sixteen in row 8 y + 4 h + i
            *(lh_u32x4 *)(tile + at * ROW + col) = v[i];
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            lh_s16x4 half[2];
#pragma unroll
            for (int y = 0; y < 2; ++y) half[y] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lh_lds_s16x4 *)(tile + (128 * wk + 16 * s + 8 * y + tr_row) * ROW + tr_col));
            const jl_bf16x8 wf = __builtin_bit_cast(jl_bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, __builtin_bit_cast(jl_bf16x8, xv[s]), acc, 0, 0, 0);
        }
    }
    if (WK > 1) {                                                    // the shares of the depth meet
        float *part = (float *)tile;
        __syncthreads();
        if (wk > 0)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[(((wk - 1) * WC + wc) * 16 + r) * 64 + lane] = acc[r];
        __syncthreads();
        if (wk == 0)
#pragma unroll
            for (int i = 0; i < WK - 1; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] += part[((i * WC + wc) * 16 + r) * 64 + lane];
    }
    if (wk == 0 && n0 + l32 < a.N) {
        bf16_t *out = (bf16_t *)a.out + n * a.out_ld + (int64_t)h * a.out_head;
        const bf16_t *gate = a.gate ? (const bf16_t *)a.gate + n * a.gate_ld + (int64_t)h * O : nullptr;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int o = o0 + 32 * wc + 8 * g + 4 * hi;
            if (o >= O) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = acc[4 * g + i];
            if (gate)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] *= 1.0f / (1.0f + expf(-ld_f(gate + o + i)));
            st4_f(out + o, v);
        }
    }
    if (a.rd > 0 && o0 == 0) {                                       // the rotary part behind the latent
        const int half = a.rot_dims >> 1;
        for (int e = tid; e < 32 * a.rd; e += 256) {
            const int m = e / a.rd, d = e - m * a.rd;
            if (n0 + m >= a.N) break;
            const bf16_t *from = (const bf16_t *)a.x + (n0 + m) * a.x_ld + (int64_t)h * a.x_head + K;
            float v = ld_f(from + d);
            if (d < a.rot_dims) {                                    // (without a rotation there are no positions and no tables)
                const float *cs = a.cos_t + (int64_t)a.pos[n0 + m] * half, *sn = a.sin_t + (int64_t)a.pos[n0 + m] * half;
                const bool near = a.pairing == JL_ROT_NEIGHBOURS, second = near ? d & 1 : d >= half;
                const int i = near ? d >> 1 : second ? d - half : d;
                const float other = ld_f(from + (near ? d ^ 1 : second ? d - half : d + half));
                v = second ? v * cs[i] + other * sn[i] : v * cs[i] - other * sn[i];
            }
            st_f((bf16_t *)a.out + (n0 + m) * a.out_ld + (int64_t)h * a.out_head + O + d, v);
        }
    }
}

extern "C" int jl_latent_heads_run(const jl_latent_heads *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_latent_heads_run: null arguments");
    const jl_latent_heads &a = *ap;
    if (a.N <= 0) return JL_OK;
    if (!a.x || !a.w || !a.out || a.H <= 0 || a.K <= 0 || a.O <= 0 || a.rd < 0 || (a.rd > 0 && a.gate)) return jl_fail(JL_E_INVALID, "jl_latent_heads_run: null pointer or bad sizes");
    if (a.K % 8 || a.O % 8 || a.x_ld % 8 || a.x_head % 8 || a.out_ld % 4 || a.out_head % 4 || (((uintptr_t)a.x | (uintptr_t)a.w) & 15) || ((uintptr_t)a.out & 7))
        return jl_fail(JL_E_INVALID, "jl_latent_heads_run: rows and heads of x and W at 16-byte borders, the result's at 8");
    if (a.x_head < a.K + a.rd || a.x_ld < (int64_t)a.H * a.x_head || a.out_head < a.O + a.rd || a.out_ld < (int64_t)a.H * a.out_head || (a.gate && a.gate_ld < (int64_t)a.H * a.O))
        return jl_fail(JL_E_INVALID, "jl_latent_heads_run: heads do not fit the rows");
    if (a.rot_dims < 0 || a.rot_dims > a.rd || a.rot_dims % 2 || (a.rot_dims && (!a.pos || !a.cos_t || !a.sin_t))) return jl_fail(JL_E_INVALID, "jl_latent_heads_run: rot_dims must be even and at most rd, with angle tables");
    if (a.pairing != JL_ROT_HALVES && a.pairing != JL_ROT_NEIGHBOURS) return jl_fail(JL_E_INVALID, "jl_latent_heads_run: unknown pairing %d", a.pairing);
    const int wc = a.K <= 128 ? 4 : a.K <= 256 ? 2 : 1;
    const int64_t groups = (int64_t)a.H * ((a.O + 32 * wc - 1) / (32 * wc));
    if (groups > 0x7fffffff || (a.N + 31) / 32 > 65535) return jl_fail(JL_E_INVALID, "jl_latent_heads_run: too many tiles");
    (wc == 4 ? latent_heads_kernel<4> : wc == 2 ? latent_heads_kernel<2> : latent_heads_kernel<1>)<<<dim3((unsigned)groups, (unsigned)((a.N + 31) / 32)), 256, 0, (hipStream_t)stream>>>(a);
    return jl_check_launch("latent_heads_kernel");
}
