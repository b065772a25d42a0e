// jl_split.h — products of 32-bit operands on the bfloat16 matrix instructions, shared by the dense products (jl_linear.hip) and the routed experts (jl_moe.hip).
#ifndef JL_SPLIT_H
#define JL_SPLIT_H

#include "jl_common.h"

typedef float sp_f32x16 __attribute__((ext_vector_type(16)));
typedef float sp_f32x4 __attribute__((ext_vector_type(4)));

// A float is the sum of three bfloat16 numbers (jl_split8: 3 x 8 bits; what lies below bfloat16's last place, 2^-133, is lost, which shows in operands below 2^-118), and a product of two is nine products
// of such terms, of which the six down to 2^-16 of it are formed here: what is left out is at most 2^-23 of a product and mostly far less, where a float's own rounding is 2^-24.  They are formed smallest first, exactly, and added in 32 bits like products of
// floats; fewer of them are rounded one by one, so that the sums are closer to 64 bits than those of the float instructions (2-norm of 1024 rows of normal numbers by 2048, own / library's: depth 4 3.2e-8 / 4.0e-8, 16 3.4e-8 / 7.4e-8, 64
// 1.1e-7 / 1.4e-7, 1024 4.9e-7 / 5.7e-7; largest against the sum of absolute products 1.0 to 3.1e-7 / 1.8 to 3.6e-7).  The bfloat16 instructions are sixteen
// times as fast as the float ones, so six of them take 0.38 of the time.
// What bounds a tile of 128 x 128: per 32 depths 1536 cycles of products, 1150 of LDS (terms written once and read by two wavefronts) and 500 of vector instructions that make the terms, which
// overlap where two or three workgroups share a CU.  Terms are made once, on the way from memory to LDS, not by every wavefront that multiplies them.
//
// What a term loses of values that are not finite (inf - inf) would reach results as NaN where the sum is an infinity: a wavefront whose sums are not all finite forms them again from memory with
// the float instructions, in the order in which products of floats are summed elsewhere (units of four depths of two halves).
//
// Tiles of TM rows of X by WR of W, both K-major and of K % 4 == 0 depths, rows at 16-byte borders; NW wavefronts, WM of them over the rows; LDS: split_units(TM, WR, TKU) units of 16 bytes.
// Stages of 8 * TKU depths: registers hold the next two while this one is multiplied.
// x_at(m) / w_at(j): where row m < TM / j < WR of the tile starts (a row that does not exist repeats another).  x_row(x) / w_row(t): first row of this wavefront's 32-row tiles.
constexpr int split_units(int TM, int WR, int TKU) { return (TM + WR) * TKU * JL_SPLIT_TERMS; }

template <int TM, int WR, int NW, int WM, int TKU, int XT, int NT, typename XAt, typename WAt, typename XRow, typename WRow>
__device__ __forceinline__ void split_products(sp_f32x16 (&acc)[XT][NT], uint4 *smem, int K, XAt x_at, WAt w_at, XRow x_row, WRow w_row) {
    constexpr int PASS = 64 * NW / TKU, XP = TM / PASS, WP = WR / PASS, ROWS = TM + WR, KS = 8 * TKU;
    static_assert(XT == TM / WM / 32 && NT == WR * WM / NW / 32 && XP * PASS == TM && WP * PASS == WR, "tile");
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hi = lane >> 5, lr = tid / TKU, lu = tid % TKU;
    // units of a row (8 depths of a term) permuted so that 16 neighbouring rows meet different banks
    auto at = [](int term, int row, int u) { return (term * ROWS + row) * TKU + (u ^ (TKU == 4 ? (row >> 2) & 3 : (row >> 1) & 7)); };
    const float *xp[XP], *wp[WP];
#pragma unroll
    for (int x = 0; x < XP; ++x) xp[x] = x_at(lr + PASS * x) + 8 * lu;
#pragma unroll
    for (int x = 0; x < WP; ++x) wp[x] = w_at(lr + PASS * x) + 8 * lu;
    const int full = K / KS, stages = (K + KS - 1) / KS;
    sp_f32x4 ahead[2][XP + WP][2];
    auto fetch = [&](sp_f32x4 (&reg)[XP + WP][2], int i) {
        if (i >= stages) return;
        const int k = i * KS;
        if (i < full) {
#pragma unroll
            for (int x = 0; x < XP + WP; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) reg[x][y] = *(const sp_f32x4 *)((x < XP ? xp[x < XP ? x : 0] : wp[x < XP ? 0 : x - XP]) + k + 4 * y);
        } else {                                                    // depths beyond K are zero: the lane reads its row's last four
            const sp_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < XP + WP; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const int d = k + 8 * lu + 4 * y;
                    const sp_f32x4 v = *(const sp_f32x4 *)((x < XP ? xp[x < XP ? x : 0] : wp[x < XP ? 0 : x - XP]) - 8 * lu + (d < K ? d : K - 4));
                    reg[x][y] = d < K ? v : zero;
                }
        }
    };
#pragma unroll
    for (int x = 0; x < XT; ++x)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[x][t][i] = 0.f;
    // The instructions cut what they add to a sum towards minus infinity, so that all sums would lean one way: by 0.5e-7 of their root mean square at a depth of 1024, 2.1e-7 at 4096, which means over
    // rows (attention's, a state's) do not take out as they do roundings.  So the sums are held with a minus sign for half of the depths, 16 at a time by + - - +, whose operands of X have one too:
    // less than 0.02e-7 is left from depths of 256 on (0.04e-7 at 64).  us, without / with: 4096 of 4096 by 4096 731 / 748, 2553 of 1024 by 1024 48.8 / 50.0, 128 of 1024 by 16384 32.3 / 32.7.
    auto turn = [&](uint32_t sign) {
#pragma unroll
        for (int x = 0; x < XT; ++x)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[x][t][i] = __uint_as_float(__float_as_uint(acc[x][t][i]) ^ sign);
    };
    constexpr int SWAPS = KS / 32;                                  // of the sums' sign in a stage
    auto stage = [&](sp_f32x4 (&reg)[XP + WP][2], int i) {
        const uint32_t sign = (uint32_t)(i * SWAPS + ((lu >> 1) + 1) / 2) << 31;
        __syncthreads();                                            // everybody has read the stage in front of this one
#pragma unroll
        for (int x = 0; x < XP + WP; ++x) {
            jl_f32x8 v;
#pragma unroll
            for (int y = 0; y < 4; ++y) { v[y] = reg[x][0][y]; v[4 + y] = reg[x][1][y]; }
            if (x < XP)
#pragma unroll
                for (int y = 0; y < 8; ++y) v[y] = __uint_as_float(__float_as_uint(v[y]) ^ sign);
            jl_bf16x8 part[JL_SPLIT_TERMS];
            jl_split8(v, part);
#pragma unroll
            for (int p = 0; p < JL_SPLIT_TERMS; ++p) smem[at(p, lr + PASS * x, lu)] = __builtin_bit_cast(uint4, part[p]);
        }
        fetch(reg, i + 2);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS / 16; ++s) {
            if (s & 1) turn(0x80000000u);
            jl_bf16x8 xf[JL_SPLIT_TERMS][XT], wf[JL_SPLIT_TERMS][NT];
#pragma unroll
            for (int p = JL_SPLIT_TERMS - 1; p >= 0; --p) {
#pragma unroll
                for (int x = 0; x < XT; ++x) xf[p][x] = __builtin_bit_cast(jl_bf16x8, smem[at(p, x_row(x) + l32, 2 * s + hi)]);
#pragma unroll
                for (int t = 0; t < NT; ++t) wf[p][t] = __builtin_bit_cast(jl_bf16x8, smem[at(p, TM + w_row(t) + l32, 2 * s + hi)]);
            }
#pragma unroll
            for (int d = JL_SPLIT_TERMS - 1; d >= 0; --d)           // the terms whose numbers add up to d
#pragma unroll
                for (int p = 0; p <= d; ++p)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int x = 0; x < XT; ++x) acc[x][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[p][x], wf[d - p][t], acc[x][t], 0, 0, 0);
        }
    };
    fetch(ahead[0], 0);
    fetch(ahead[1], 1);
    for (int i = 0; i < stages; i += 2) {
        stage(ahead[0], i);
        if (i + 1 < stages) stage(ahead[1], i + 1);
    }
    turn((uint32_t)(stages * SWAPS) << 31);
    float odd = 0.f;                                                // not a number if any sum is not finite
#pragma unroll
    for (int x = 0; x < XT; ++x)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) odd = __builtin_fmaf(acc[x][t][i], 0.f, odd);
    if (__ballot(odd != 0.f) == 0) return;
#pragma unroll 1
    for (int x = 0; x < XT; ++x)
#pragma unroll 1
        for (int t = 0; t < NT; ++t) {
            const float *xs = x_at(x_row(x) + l32), *ws = w_at(w_row(t) + l32);
            sp_f32x16 sum;
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[i] = 0.f;
            for (int k = 4 * hi; k < K + 4 * hi; k += 8) {          // the same number of turns for both halves
                const bool in = k < K;
                const sp_f32x4 zero = {0.f, 0.f, 0.f, 0.f}, a = in ? *(const sp_f32x4 *)(xs + k) : zero, b = in ? *(const sp_f32x4 *)(ws + k) : zero;
#pragma unroll
                for (int y = 0; y < 4; ++y) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(a[y], b[y], sum, 0, 0, 0);
            }
#pragma unroll
            for (int xx = 0; xx < XT; ++xx)
#pragma unroll
                for (int tt = 0; tt < NT; ++tt)
                    if (xx == x && tt == t) acc[xx][tt] = sum;
        }
}

#endif
