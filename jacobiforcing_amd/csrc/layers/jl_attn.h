// jl_attn.h — what the attention sources share.
#ifndef JL_ATTN_H
#define JL_ATTN_H

#include "jl_common.h"

// floats -> bfloat16 (round to nearest even) through the compiler's own conversion: one packed instruction per pair
typedef __bf16 ar_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ar_f32x4 __attribute__((ext_vector_type(4)));
typedef float ar_f32x8 __attribute__((ext_vector_type(8)));
typedef float ar_f32x16 __attribute__((ext_vector_type(16)));
typedef short ar_s16x4 __attribute__((ext_vector_type(4)));
typedef short ar_s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) ar_s16x4 ar_lds_s16x4;

// where 16-byte unit u of row r sits in a row of U units
template <int U> __device__ __forceinline__ int ar_key_unit(int r, int u) { return U % 16 == 0 ? u ^ (r & 15) : u ^ ((r >> 1) & 7); }
template <int U> __device__ __forceinline__ int ar_value_unit(int r, int u) { return U == 16 ? u ^ ((r & 3) << 2) : u ^ ((r & 2) << 1); }

// Scores are scaled behind their maximum, in the exponent's own instruction (queries take a negative scale's sign), which takes a factor above zero: one so small that its products could vanish (zero
// too) is multiplied with the scores one by one
constexpr float AR_LOG2E = 1.44269504088896341f;
__host__ __device__ __forceinline__ bool ar_one_by_one(float scale) { return scale > -1e-30f && scale < 1e-30f; }

// A weight is 2 ** fma(score, c2, -m): its exponent keeps what the rounding of m = score * c2 left over, 2^-24 of m, the same for all of a row.  That is no more than one up to 2^24; rows beyond, whose
// weights it would carry out of range, have their products rounded as m was.  Such rows enter the branch that scales the sums for every tile (`entry`: the maximum beyond which a row enters it).
__device__ __forceinline__ bool ar_far(float m) { return fabsf(m) >= 16777216.f && m > -INFINITY; }
__device__ __forceinline__ float ar_entry(float m) { return ar_far(m) ? -INFINITY : m; }
template <int N> __device__ __forceinline__ float ar_factor(ar_f32x16 (&sc)[N], float c2, float m) {
    const bool far = ar_far(m);
    if (!__any(far)) return c2;
#pragma unroll
    for (int h = 0; h < N; ++h)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[h][i] *= far ? c2 : 1.0f;
    return far ? 1.0f : c2;
}

constexpr int AR_ROWS = 128;          // (query, head) rows of a tile of the wide form

// tiles and groups (``hb`` per key head) lie along one axis of the grid: up to 2 ** 32 threads of workgroups of 256
static inline bool jl_attn_grid_fits(const jl_attn_args &a, int hb) { return (int64_t)a.n_tiles * a.G * hb < (1 << 24); }

// the wide form's launch (jl_attn_rows.hip); sizes as jl_attn_sweep has checked them, ``hf`` heads of a.TQ queries per tile, ``hb`` tiles per group
int jl_attn_rows_launch(const jl_attn_args &a, int hf, int hb, bool v_in_k, hipStream_t st);

// Portions of a few tokens (jl_attn_token.hip), at most a.longest per tile: a.Gv, strides, checks and tiles as in the forms they are called from (jl_attn_talk, jl_attn_narrow, jl_attn_sweep)
bool jl_attn_token_fits(const jl_attn_args &a, bool v_in_k);
int jl_attn_token_launch(const jl_attn_args &a, bool v_in_k, hipStream_t st);

// where keys and values come from: pages of pools, pages whose key rows hold the values in their first columns, or contiguous rows per request whose heads
// share their last columns (keys and values built for this step)
enum { AR_PAGED, AR_V_IN_K, AR_BUILT };

// float activations (jl_attn_f32.hip): tiles of 128 rows (``wide``) or of 32, whose keys may be shared out
bool jl_attn_f32_fits(int H, int G, int Gv, int D, int Dv, int64_t k_ld, int64_t v_ld, bool v_in_k);
int jl_attn_f32_launch(const jl_attn_args &a, int hf, int hb, int src, bool wide, hipStream_t st);

#endif
