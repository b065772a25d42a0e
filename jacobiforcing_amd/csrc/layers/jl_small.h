// jl_small.h — products of a few rows straight from memory into the matrix cores, shared by the dense products (jl_linear.hip) and the experts' router (jl_moe.hip).
#ifndef JL_SMALL_H
#define JL_SMALL_H

#include "jl_common.h"

constexpr int LS_AHEAD = 4;

typedef float ls_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 ls_bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ ls_f32x4 ls_mma(const bf16_t *, uint4 a, uint4 b, ls_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ls_bf16x8, a), __builtin_bit_cast(ls_bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ ls_f32x4 ls_mma(const float *, uint4 a, uint4 b, ls_f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
}

__device__ __forceinline__ uint4 ls_unit(const bf16_t *p, const bf16_t *) { return *(const uint4 *)p; }
__device__ __forceinline__ uint4 ls_unit(const float *p, const float *) { return *(const uint4 *)p; }
__device__ __forceinline__ uint4 ls_unit(const bf16_t *p, const float *) {        // four 16-bit values for a float product
    const uint2 v = *(const uint2 *)p;
    return make_uint4(v.x << 16, v.x & 0xffff0000u, v.y << 16, v.y & 0xffff0000u);
}

// acc[o][t]: rows o0 + 16 o .. of W (first operand) by rows 16 t .. of x, summed over this wavefront's share of the depth (NW wavefronts share it); rows that do not exist repeat the last
// (w_ld: how far W's rows lie apart, if not K).  AHEAD steps' units are on their way at once; TURNS: and as many more while those are multiplied
template <typename TX, typename T, int NT, int OT, int NW, int AHEAD = LS_AHEAD, bool TURNS = false>
__device__ __forceinline__ void ls_products(ls_f32x4 (&acc)[OT][NT], const TX *__restrict__ x, int64_t x_ld, const T *__restrict__ w, int N, int K, int o0, int O, int wave, int lane, int w_ld = 0) {
    constexpr int UNIT = 16 / sizeof(T), LINE = 8 * UNIT;           // elements of a unit, of the 128 bytes that a step takes from every row
    const int r16 = lane & 15, g = lane >> 4;
    const int k_lane = UNIT * g;
    const T *wp[OT];
    const TX *xp[NT];
#pragma unroll
    for (int o = 0; o < OT; ++o) {
        const int r = o0 + 16 * o + r16;
        wp[o] = w + (int64_t)(r < O ? r : O - 1) * (w_ld ? w_ld : K) + k_lane;      // rows and columns that do not exist repeat the last one and are not stored
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[o][t] = (ls_f32x4){0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int n = 16 * t + r16;
        xp[t] = x + (int64_t)(n < N ? n : N - 1) * x_ld + k_lane;
    }
    const int steps = (K + LINE - 1) / LINE, s0 = steps * wave / NW, s1 = steps * (wave + 1) / NW;
    auto load = [&](int s, uint4 (&wr)[AHEAD][2][OT], uint4 (&xr)[AHEAD][2][NT]) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int k = (s + i) * LINE + 4 * UNIT * y;
                const bool in = s + i < s1 && k + k_lane < K;
#pragma unroll
                for (int o = 0; o < OT; ++o) wr[i][y][o] = in ? *(const uint4 *)(wp[o] + k) : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; ++t) xr[i][y][t] = in ? ls_unit(xp[t] + k, (const T *)nullptr) : make_uint4(0, 0, 0, 0);
            }
    };
    auto multiply = [&](const uint4 (&wr)[AHEAD][2][OT], const uint4 (&xr)[AHEAD][2][NT]) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int o = 0; o < OT; ++o)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[o][t] = ls_mma((const T *)nullptr, wr[i][y][o], xr[i][y][t], acc[o][t]);
    };
    if constexpr (!TURNS) {
        uint4 wr[AHEAD][2][OT], xr[AHEAD][2][NT];
        for (int s = s0; s < s1; s += AHEAD) {
            load(s, wr, xr);
            multiply(wr, xr);
        }
    } else {
        uint4 wr[2][AHEAD][2][OT], xr[2][AHEAD][2][NT];
        load(s0, wr[0], xr[0]);
        for (int s = s0; s < s1; s += 2 * AHEAD) {
            load(s + AHEAD, wr[1], xr[1]);
            multiply(wr[0], xr[0]);
            load(s + 2 * AHEAD, wr[0], xr[0]);
            multiply(wr[1], xr[1]);
        }
    }
}

#endif
