// jl_moe.hip — routed experts: the router's choice (sigmoid scores with a correction, a softmax renormalised over the chosen with or without
// a correction, or a softmax over the chosen logits alone), the rows grouped by expert (a choice of an expert without weights has none), and
// the grouped products: up with relu^2, plain, or with the gated unit in its epilogue, down with the routing weights.
#include "jl_small.h"
#include "jl_split.h"
#include <stdlib.h>
#include <type_traits>
constexpr int MOE_MAX_E = 4096;   // experts (router outputs) at most
struct MoeAct { int kind; float limit, alpha, shift; };       // the gated unit of JL_MOE_UP_GATED (jl_gated_act's kinds)

// ---- router: one wavefront per token, NJ router outputs per lane (lane + 64 j) -------------------------------------------------------
// Every lane keeps its outputs' comparison values and scores in registers; `top` rounds find the largest comparison value (ties: the lowest
// index) by a butterfly over (value, index, score).  An output that was chosen leaves the race through a bit per lane and j.
//   kind                      comparison value                       score
//   JL_ROUTE_SIGMOID          sigmoid(z) + correction                sigmoid(z)
//   JL_ROUTE_SOFTMAX_RENORM   softmax(z) + correction (none: z)      softmax(z), divided by the chosen scores' sum + renorm_eps
//   JL_ROUTE_TOP_SOFTMAX      z                                      exp(z - the largest z), divided by the chosen ones' sum
template <int NJ>
__global__ __launch_bounds__(256) void moe_route_kernel(const float *__restrict__ logits, const float *__restrict__ correction, int64_t N, int E, int top,
                                                         float scale, int32_t *__restrict__ ids, float *__restrict__ weights, int kind, float renorm_eps) {
    const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (n >= N) return;
    const float *z = logits + n * E;
    float cmp[NJ], sc[NJ], zmax = -INFINITY;
    uint64_t open = 0;                                              // bit j: this lane's output j exists and is not chosen yet
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int e = lane + 64 * j;
        cmp[j] = sc[j] = -INFINITY;
        if (e < E) { cmp[j] = z[e]; open |= 1ull << j; zmax = fmaxf(zmax, cmp[j]); }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) zmax = fmaxf(zmax, __shfl_xor(zmax, off, 64));
    float den = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int e = lane + 64 * j;
        if (e >= E) continue;
        sc[j] = kind == JL_ROUTE_SIGMOID ? 1.0f / (1.0f + expf(-cmp[j])) : expf(cmp[j] - zmax);
        den += sc[j];
    }
    if (kind == JL_ROUTE_SOFTMAX_RENORM) den = wave_sum_f32(den);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int e = lane + 64 * j;
        if (e >= E) continue;
        if (kind == JL_ROUTE_SOFTMAX_RENORM) sc[j] /= den;
        if (kind == JL_ROUTE_SIGMOID) cmp[j] = sc[j];
        if (kind == JL_ROUTE_SOFTMAX_RENORM && correction) cmp[j] = sc[j];
        if (correction && kind != JL_ROUTE_TOP_SOFTMAX) cmp[j] += correction[e];
        if (cmp[j] != cmp[j]) cmp[j] = INFINITY;                    // not a number: as the largest, here as in moe_route_rows
    }
    float chosen = 0.f;
    for (int s = 0; s < top; ++s) {
        float bv = -INFINITY, bs = 0.f;
        int be = 0x7fffffff;                                        // none
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if ((open >> j & 1) && (be == 0x7fffffff || cmp[j] > bv)) { bv = cmp[j]; bs = sc[j]; be = lane + 64 * j; }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 64), os = __shfl_xor(bs, off, 64);
            const int oe = __shfl_xor(be, off, 64);
            if (oe != 0x7fffffff && (be == 0x7fffffff || ov > bv || (!(bv > ov) && oe < be))) { bv = ov; bs = os; be = oe; }
        }
        be = __shfl(be, 0, 64);                                     // one winner for all lanes
        bs = __shfl(bs, 0, 64);
        if ((be & 63) == lane) open &= ~(1ull << (be >> 6));
        if ((s & 63) == lane) { ids[n * top + s] = be; weights[n * top + s] = bs; }
        chosen += bs;
    }
    const float by = kind == JL_ROUTE_SIGMOID ? 1.0f : kind == JL_ROUTE_SOFTMAX_RENORM ? chosen + renorm_eps : chosen;
    for (int s = lane; s < top; s += 64) weights[n * top + s] = weights[n * top + s] / by * scale;      // what this lane wrote above
}

extern "C" int jl_moe_route(const float *logits, const float *correction, int64_t N, int32_t E, int32_t top, float scale, int32_t *ids,
                            float *weights, int32_t kind, float renorm_eps, void *stream) {
    if (N <= 0) return JL_OK;
    if (!logits || !ids || !weights || E <= 0 || top <= 0 || top > E) return jl_fail(JL_E_INVALID, "jl_moe_route: null pointer or top > experts");
    if (kind < JL_ROUTE_SIGMOID || kind > JL_ROUTE_TOP_SOFTMAX) return jl_fail(JL_E_INVALID, "jl_moe_route: unknown kind %d", kind);
    if (E > MOE_MAX_E) return jl_fail(JL_E_INVALID, "jl_moe_route: at most %d router outputs", MOE_MAX_E);
#define ROUTE_CASE(NJ) moe_route_kernel<NJ><<<dim3((unsigned)((N + 3) / 4)), 256, 0, (hipStream_t)stream>>>(logits, correction, N, E, top, scale, ids, weights, kind, renorm_eps)
    if (E <= 64) ROUTE_CASE(1);
    else if (E <= 256) ROUTE_CASE(4);
    else if (E <= 1024) ROUTE_CASE(16);
    else ROUTE_CASE(64);
#undef ROUTE_CASE
    return jl_check_launch("moe_route_kernel");
}

// ---- grouping: one workgroup counts, scans and places (a step holds at most a few 10^5 rows) ----------------------------------------
constexpr int MOE_TM = 64;        // rows and output columns of a tile of the product for any size
constexpr int MOE_TN = 64;
constexpr int MOE_TK = 32;        // depth of one LDS stage

// Its time is the latency of the trips to memory and of the counters, so a thread has MG_IN_FLIGHT ids on the way at once, and up to 16 wavefronts count in
// tables of their own (8 192 rows x 4 choices over 32 experts: 53 us with one id at a time on shared counters, 15 us so).
constexpr int MG_IN_FLIGHT = 16, MG_COUNTERS = 8192;
__global__ __launch_bounds__(1024) void moe_group_kernel(const int32_t *__restrict__ ids, int64_t rows, int E, int tile_rows,
                                                          int32_t *__restrict__ perm, int32_t *__restrict__ offsets,
                                                          int32_t *__restrict__ tile_expert, int32_t *__restrict__ tile_row0, int max_tiles) {
    __shared__ int cnt[MG_COUNTERS];                                  // [tables][E]: counts, then the next free place of a table's rows
    __shared__ int first_tile[MOE_MAX_E + 1];
    __shared__ int wave_sum[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tables = MG_COUNTERS / E < 16 ? MG_COUNTERS / E : 16;
    int *mine = cnt + (wave % tables) * E;
    for (int e = tid; e < tables * E; e += 1024) cnt[e] = 0;
    __syncthreads();
    auto each = [&](auto &&f) {
        for (int64_t r0 = 0; r0 < rows; r0 += 1024 * MG_IN_FLIGHT) {
            int e[MG_IN_FLIGHT];
#pragma unroll
            for (int i = 0; i < MG_IN_FLIGHT; ++i) {
                const int64_t r = r0 + i * 1024 + tid;
                e[i] = r < rows ? ids[r] : -1;
            }
#pragma unroll
            for (int i = 0; i < MG_IN_FLIGHT; ++i)
                if (e[i] >= 0 && e[i] < E) f((int32_t)(r0 + i * 1024 + tid), e[i]);      // an expert without weights has no rows
        }
    };
    each([&](int32_t, int e) { atomicAdd(&mine[e], 1); });
    __syncthreads();
    // a thread owns MOE_MAX_E / 1024 neighbouring experts: their rows and tiles, summed over the threads in front of it
    constexpr int PER = MOE_MAX_E / 1024;
    int n_rows[PER], sum_r = 0, sum_t = 0;
#pragma unroll
    for (int x = 0; x < PER; ++x) {
        const int e = tid * PER + x;
        n_rows[x] = 0;
        if (e < E)
            for (int t = 0; t < tables; ++t) n_rows[x] += cnt[t * E + e];
        sum_r += n_rows[x];
        sum_t += (n_rows[x] + tile_rows - 1) / tile_rows;
    }
    int inc_r = sum_r, inc_t = sum_t;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int a = __shfl_up(inc_r, off, 64), b = __shfl_up(inc_t, off, 64);
        if (lane >= off) { inc_r += a; inc_t += b; }
    }
    if (lane == 63) { wave_sum[0][wave] = inc_r; wave_sum[1][wave] = inc_t; }
    __syncthreads();
    int o = inc_r - sum_r, t0 = inc_t - sum_t;
    for (int w = 0; w < wave; ++w) { o += wave_sum[0][w]; t0 += wave_sum[1][w]; }
#pragma unroll
    for (int x = 0; x < PER; ++x) {
        const int e = tid * PER + x;
        if (e < E) {
            offsets[e] = o;
            first_tile[e] = t0;
            int at = o;
            for (int t = 0; t < tables; ++t) { const int c = cnt[t * E + e]; cnt[t * E + e] = at; at += c; }
        }
        o += n_rows[x];
        t0 += (n_rows[x] + tile_rows - 1) / tile_rows;
    }
    if (tid == 1023) { offsets[E] = o; offsets[E + 1] = t0 < max_tiles ? t0 : max_tiles; first_tile[E] = t0; }
    __syncthreads();
    const int tiles = first_tile[E];
    for (int t = tid; t < max_tiles; t += 1024) {
        int lo = 0, hi = E;                                           // the expert whose tiles t is among: the last with first_tile <= t that has rows
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (first_tile[mid] <= t) lo = mid; else hi = mid;
        }
        tile_expert[t] = t < tiles ? lo : -1;
        tile_row0[t] = t < tiles ? cnt[lo] + (t - first_tile[lo]) * tile_rows : 0;      // table 0's first place is the expert's first row
    }
    __syncthreads();
    // placement: a row's place within its expert is whatever the counter says when it arrives.  The order of an expert's rows
    // changes nothing in the results (every row is computed by itself); only which tile a row lands in differs from run to run.
    each([&](int32_t r, int e) { perm[atomicAdd(&mine[e], 1)] = r; });
}

// Rows of a tile.  High tiles read the weights less often and do more per byte of LDS, low ones pad less, give more workgroups and overlap their starts and ends.
// 128 rows need both products to fill the chip and about a tile of rows per expert; 64 need as many blocks as the chip takes at once.  Measured, experts alone, gated,
// bfloat16, us at 32 / 64 / 128 rows, choice and grouping included: 8192 tokens x 4 of 32 (2048 x 1024) 1046 / 716 / 539, 1024 tokens 195 / 168 / 159, 512 tokens 136 / 132 / 143, 256 tokens
// 111 / 117 / 140; 4096 x 4 of 16 (1024 x 512) 175 / 122 / 110, 1024 tokens 64 / 57 / 73, 512 tokens 47 / 51 / 69; 4096 x 4 of 12 (768 x 512) 147 / 105 / 91, 2048 tokens 85 / 66 / 70;
// float, 2048 x 4 of 16 (1024 x 512), 32 / 64 rows: 356 / 318 (64 on the float instructions).
// Sizes the matrix-core product does not take (rows that do not start at 16-byte borders) go in tiles of MOE_TM.
static bool moe_mm_sizes(int dtype, int64_t K) { return (dtype == JL_BF16 && K % 8 == 0) || (dtype == JL_F32 && K % 4 == 0); }
extern "C" int jl_moe_tile_rows(int dtype, int64_t rows, int32_t E, int32_t W, int32_t ff) {
    if (E <= 0 || !moe_mm_sizes(dtype, W) || !moe_mm_sizes(dtype, ff)) return MOE_TM;
    auto blocks = [&](int tm, int width, int tn) { return (rows / tm + E / 2) * ((width + tn - 1) / tn); };
    if (dtype == JL_BF16 && blocks(128, ff, 128) >= 256 && blocks(128, W, 256) >= 256 && rows >= (int64_t)96 * E) return 128;
    return rows >= (int64_t)48 * E && blocks(64, ff, 128) + blocks(64, W, 256) >= 512 ? 64 : 32;
}

// Tiles of 128 rows in pairs: the way up in tiles of 256 x 256 (moe_big_kernel), one workgroup per CU, so from two and a half rounds of the chip's CUs on; the way down walks the pairs' halves.
// us, experts alone, gated, tiles of 128 / 256: 8192 tokens x 4 of 32 (2048 x 1024; 1152 workgroups) 656 / 598, 6554 x 4 (944) 546 / 509, 4096 x 4 (640) 372 / 355, 8192 x 4 of 24 (1536 x 768; 840)
// 403 / 382; below: 8192 x 2 of 8 (1024 x 1024; 544) 188 / 190, 8192 x 3 of 9 (1088 x 704; 600) 216 / 221.
// moe_big_kernel takes depths in whole stages and rows within 32 bits (gathered ones are at most as many as sorted ones).
static bool moe_big_sizes(int64_t K, int64_t rows) { return K % 64 == 0 && rows * K * 2 <= UINT32_MAX; }
extern "C" int jl_moe_tile_pairs(int64_t rows, int32_t E, int32_t W, int32_t ff, int32_t gated) {
    const int cols = gated ? 128 : 256;
    return E > 0 && rows >= (int64_t)256 * E && (rows / 256 + E / 2) * ((ff + cols - 1) / cols) >= 640 && moe_big_sizes(W, rows + (int64_t)256 * E);
}

// Float tiles of 64 rows in fours, which the products walk in parts of 128 rows (moe_split_kernel), where experts fill them.  us, experts alone, gated, 64 / 128: 638 rows per expert (2553 x 4 of 16 of
// 1024 x 512) 276 / 248, 383 170 / 158, 340 (2042 x 4 of 24 of 768 x 320) 124 / 116; below the line 311 (700 x 4 of 9 of 1024 x 1024) 167 / 220, 263 (2042 x 4 of 31 of 960 x 704) 304 / 330, 255 167 / 147 and 137 / 156.
extern "C" int jl_moe_float_tiles(int64_t rows, int32_t E, int32_t W, int32_t ff) {
    return E > 0 && rows >= (int64_t)320 * E && moe_mm_sizes(JL_F32, W) && moe_mm_sizes(JL_F32, ff) ? 256 : 64;
}

extern "C" int jl_moe_group(const int32_t *ids, int64_t N, int32_t top, int32_t E, int32_t tile_rows, int32_t *perm, int32_t *offsets,
                            int32_t *tile_expert, int32_t *tile_row0, int32_t max_tiles, void *stream) {
    if (N <= 0) return JL_OK;
    if (!ids || !perm || !offsets || !tile_expert || !tile_row0) return jl_fail(JL_E_INVALID, "jl_moe_group: null pointer");
    if (E <= 0 || E > MOE_MAX_E || top <= 0 || tile_rows <= 0 || (int64_t)max_tiles < N * top / tile_rows + E)
        return jl_fail(JL_E_INVALID, "jl_moe_group: experts must be <= %d and max_tiles >= rows / tile_rows + experts", MOE_MAX_E);
    moe_group_kernel<<<1, 1024, 0, (hipStream_t)stream>>>(ids, N * top, E, tile_rows, perm, offsets, tile_expert, tile_row0, max_tiles);
    return jl_check_launch("moe_group_kernel");
}

// ---- a layer's whole choice in one or two launches: router product, choice, grouping (up to 64 router outputs) --------------------------------------
// Every workgroup takes 16 or 32 tokens: it forms their logits (the depth shared by eight wavefronts, rows of x and W straight from memory into the float matrix instructions: ls_products) or reads
// them (LOGITS), chooses per token from LDS and counts its choices per expert; with one workgroup it groups them too.  With more, a second launch of as many workgroups adds the counts up to where each
// one's rows go: no workgroup walks all rows.  What bounds them: what one CU takes in, 26 GB/s of x and W (more of them on the way, or the products on the bfloat16 instructions in three terms, change
// nothing), then the table of counts.  us, product + choice + grouping in launches of their own / in these (from logits): 8192 x 1024 bfloat16 by 16 outputs 57 / 17 (9), 8192 x 2048 float by 32
// 51 / 32 (13), by 40 56 / 45 (19), 32 x 1024 by 16 24 / 11 in one launch instead of three, 32 x 2048 float by 32 27 / 21 (in slices of the depth, jl_moe_router_slices: 13), 2246 x 1024 float by 16 28 / 13.
constexpr int MR_MAX_E = 64, MR_NW = 8;

// lane e of the first wavefront: where expert e's rows and tiles start; offsets and the list of tiles (the first workgroup's to write)
__device__ __forceinline__ void moe_group_list(const jl_moe_router &a, int rows_e, int lane, int &start, int *first_tile) {
    const int tiles_e = (rows_e + a.tile_rows - 1) / a.tile_rows;
    int inc_r = rows_e, inc_t = tiles_e;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(inc_r, off, 64), y = __shfl_up(inc_t, off, 64);
        if (lane >= off) { inc_r += x; inc_t += y; }
    }
    start = inc_r - rows_e;
    first_tile[lane] = inc_t - tiles_e;                             // an expert without rows has no tiles: the same number as the next
    if (lane == 63) first_tile[64] = inc_t;
    if (blockIdx.x == 0) {
        if (lane < a.experts) a.offsets[lane] = start;
        if (lane == 63) { a.offsets[a.experts] = inc_r; a.offsets[a.experts + 1] = inc_t < a.max_tiles ? inc_t : a.max_tiles; }
    }
}
__device__ __forceinline__ void moe_tile_list(const jl_moe_router &a, const int *starts, const int *first_tile, int tid, int threads) {
    for (int t = tid; t < a.max_tiles; t += threads) {
        int lo = 0, hi = a.experts;                                 // the last expert with first_tile <= t
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (first_tile[mid] <= t) lo = mid; else hi = mid;
        }
        const bool in = t < first_tile[64];
        a.tile_expert[t] = in ? lo : -1;
        a.tile_row0[t] = in ? starts[lo] + (t - first_tile[lo]) * a.tile_rows : 0;
    }
}

// the largest over groups of P lanes (16, 32 or 64); within rows of 16 by exchanges in the vector unit
template <int P> __device__ __forceinline__ float moe_group_max(float v) {
#define MR_STEP(ctrl) v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), ctrl, 0xF, 0xF, true)))
    MR_STEP(0xB1);                                                  // quad_perm [1, 0, 3, 2], [2, 3, 0, 1], half rows and rows mirrored
    MR_STEP(0x4E);
    MR_STEP(0x141);
    MR_STEP(0x140);
#undef MR_STEP
    if (P > 16) v = fmaxf(v, __shfl_xor(v, 16, 64));
    if (P > 32) v = fmaxf(v, __shfl_xor(v, 32, 64));
    return v;
}
// moe_route_kernel's choice for R tokens per P lanes at once (their chains of exchanges run side by side), 64 / P groups of lanes: this lane's output is e = lane % P, the logits of token r at z[r];
// each(r, s, e, weight) by the lane of the s-th choice.  A choice is the lowest index among the largest comparison values (one that is not a number counts as the largest): the wavefront's
// mask of them has it without passing indices on.  The sums are those of moe_route_kernel in the same order.
template <int P, int R, typename Each>
__device__ __forceinline__ void moe_route_rows(const float *const (&z)[R], const float *__restrict__ correction, int E, int top, int kind, float scale, float renorm_eps, int lane, Each each) {
    const int e = lane % P, base = lane - e;
    const uint64_t group = P == 64 ? ~0ull : (1ull << P) - 1;
    float cmp[R], sc[R], zmax[R], den[R], chosen[R];
    int turn[R];                                                    // which choice this lane's output is; -1: none yet, -2: there is no such output
#pragma unroll
    for (int r = 0; r < R; ++r) { turn[r] = e < E ? -1 : -2; cmp[r] = e < E ? z[r][e] : -INFINITY; zmax[r] = moe_group_max<P>(cmp[r]); }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        sc[r] = e >= E ? -INFINITY : kind == JL_ROUTE_SIGMOID ? 1.0f / (1.0f + expf(-cmp[r])) : expf(cmp[r] - zmax[r]);
        den[r] = e < E ? sc[r] : 0.f;
        chosen[r] = 0.f;
    }
    if (kind == JL_ROUTE_SOFTMAX_RENORM)
#pragma unroll
        for (int off = P / 2; off > 0; off >>= 1)
#pragma unroll
            for (int r = 0; r < R; ++r) den[r] += __shfl_xor(den[r], off, 64);
    const float add = e < E && correction && kind != JL_ROUTE_TOP_SOFTMAX ? correction[e] : 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (kind == JL_ROUTE_SOFTMAX_RENORM) sc[r] /= den[r];
        if (kind == JL_ROUTE_SIGMOID || (kind == JL_ROUTE_SOFTMAX_RENORM && correction)) cmp[r] = sc[r];
        if (correction && kind != JL_ROUTE_TOP_SOFTMAX) cmp[r] += add;
        if (cmp[r] != cmp[r]) cmp[r] = INFINITY;
    }
    for (int s = 0; s < top; ++s) {
        float most[R];
#pragma unroll
        for (int r = 0; r < R; ++r) most[r] = moe_group_max<P>(turn[r] == -1 ? cmp[r] : -INFINITY);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint64_t largest = __ballot(turn[r] == -1 && cmp[r] == most[r]) >> base & group;
            const int be = largest ? __ffsll((unsigned long long)largest) - 1 : 0;
            chosen[r] += __shfl(sc[r], base + be, 64);
            if (be == e) turn[r] = s;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (turn[r] >= 0) each(r, turn[r], e, sc[r] / (kind == JL_ROUTE_SIGMOID ? 1.0f : kind == JL_ROUTE_SOFTMAX_RENORM ? chosen[r] + renorm_eps : chosen[r]) * scale);
}

// a slice of the depth of a block's logits: [slices][N][E] in a.parts, for moe_router_kernel to add up
template <typename TX, int NT, int OT>
__global__ __launch_bounds__(64 * MR_NW) void moe_router_part_kernel(jl_moe_router a) {
    constexpr int ROWS = 16 * NT;
    __shared__ ls_f32x4 part[MR_NW][OT][NT][64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, k0 = (int)((int64_t)a.K * blockIdx.y / a.slices) & ~31, k1 = blockIdx.y + 1 == (unsigned)a.slices ? a.K : (int)((int64_t)a.K * (blockIdx.y + 1) / a.slices) & ~31;
    const int64_t n0 = (int64_t)blockIdx.x * ROWS;
    const int rows = a.N - n0 < ROWS ? (int)(a.N - n0) : ROWS;
    ls_f32x4 acc[OT][NT];
    ls_products<TX, float, NT, OT, MR_NW, 1>(acc, (const TX *)a.x + n0 * a.x_ld + k0, a.x_ld, a.w + k0, rows, k1 - k0, 0, a.E, wave, lane, a.K);
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
        for (int t = 0; t < NT; ++t) part[wave][o][t][lane] = acc[o][t];
    __syncthreads();
    float *to = a.parts + ((int64_t)blockIdx.y * a.N + n0) * a.E;
    for (int e = tid; e < OT * NT * 64; e += 64 * MR_NW) {
        const int l = e & 63, t = (e >> 6) % NT, ot = (e >> 6) / NT, o = 16 * ot + 4 * (l >> 4), n = 16 * t + (l & 15);
        ls_f32x4 s = part[0][ot][t][l];
#pragma unroll
        for (int i = 1; i < MR_NW; ++i) s += part[i][ot][t][l];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n < rows && o + i < a.E) to[n * a.E + o + i] = s[i];
    }
}

template <typename TX, int NT, int OT, bool LOGITS>
__global__ __launch_bounds__(64 * MR_NW) void moe_router_kernel(jl_moe_router a) {
    constexpr int ROWS = 16 * NT;
    __shared__ ls_f32x4 part[LOGITS ? 1 : MR_NW][OT][NT][64];
    __shared__ float z[ROWS][16 * OT];
    __shared__ int count[MR_MAX_E], starts[MR_MAX_E], first_tile[MR_MAX_E + 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t n0 = (int64_t)blockIdx.x * ROWS;
    const int rows = a.N - n0 < ROWS ? (int)(a.N - n0) : ROWS;
    if (tid < MR_MAX_E) count[tid] = 0;
    if constexpr (LOGITS) {
        const float *from = (a.slices > 1 ? a.parts : (const float *)a.x) + n0 * a.E;
        for (int i = tid; i < rows * a.E; i += 64 * MR_NW) {
            float sum = from[i];
#pragma unroll 8
            for (int p = 1; p < a.slices; ++p) sum += from[p * a.N * a.E + i];
            z[i / a.E][i % a.E] = a.bias ? sum + a.bias[i % a.E] : sum;
        }
    } else {
        ls_f32x4 acc[OT][NT];
        ls_products<TX, float, NT, OT, MR_NW, 1, true>(acc, (const TX *)a.x + n0 * a.x_ld, a.x_ld, a.w, rows, a.K, 0, a.E, wave, lane);
#pragma unroll
        for (int o = 0; o < OT; ++o)
#pragma unroll
            for (int t = 0; t < NT; ++t) part[wave][o][t][lane] = acc[o][t];
        __syncthreads();
        for (int e = tid; e < OT * NT * 64; e += 64 * MR_NW) {
            const int l = e & 63, t = (e >> 6) % NT, ot = (e >> 6) / NT, o = 16 * ot + 4 * (l >> 4);
            ls_f32x4 s = part[0][ot][t][l];
#pragma unroll
            for (int i = 1; i < MR_NW; ++i) s += part[i][ot][t][l];
#pragma unroll
            for (int i = 0; i < 4; ++i) z[16 * t + (l & 15)][o + i] = a.bias && o + i < a.E ? s[i] + a.bias[o + i] : s[i];
        }
    }
    __syncthreads();
    // a wavefront's tokens: its share of the rows, a few side by side
    constexpr int P = 16 * OT <= 16 ? 16 : 16 * OT <= 32 ? 32 : 64, SHARE = ROWS / MR_NW, GROUPS = 64 / P < SHARE ? 64 / P : SHARE, R = SHARE / GROUPS;
    const float *zr[R];
    int64_t first[R];                                               // where the row's choices lie
    bool real[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int g = lane / P < GROUPS ? lane / P : GROUPS - 1, row = wave * SHARE + r * GROUPS + g;
        real[r] = lane / P < GROUPS && row < rows;
        zr[r] = z[row];
        first[r] = (n0 + row) * a.top;
    }
    moe_route_rows<P, R>(zr, a.correction, a.E, a.top, a.kind, a.scale, a.renorm_eps, lane, [&](int r, int s, int e, float weight) {
        if (!real[r]) return;
        a.ids[first[r] + s] = e;
        a.weights[first[r] + s] = weight;
        if (e < a.experts) atomicAdd(&count[e], 1);                 // an expert without weights has no rows
    });
    __syncthreads();
    if (gridDim.x > 1) {
        if (tid < a.experts) a.counts[(int64_t)blockIdx.x * a.experts + tid] = count[tid];
        return;
    }
    if (wave == 0) {
        int start;
        moe_group_list(a, lane < a.experts ? count[lane] : 0, lane, start, first_tile);
        starts[lane] = start;
    }
    __syncthreads();
    moe_tile_list(a, starts, first_tile, tid, 64 * MR_NW);
    __syncthreads();
    for (int i = tid; i < rows * a.top; i += 64 * MR_NW) {
        const int e = a.ids[i];
        if (e >= 0 && e < a.experts) a.perm[atomicAdd(&starts[e], 1)] = i;
    }
}

// the workgroups of moe_router_kernel again: rows_per_block tokens each
__global__ __launch_bounds__(1024) void moe_place_kernel(jl_moe_router a, int rows_per_block) {
    __shared__ int total[16][MR_MAX_E], before[16][MR_MAX_E], starts[MR_MAX_E], place[MR_MAX_E], first_tile[MR_MAX_E + 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, blocks = gridDim.x, P = a.experts <= 16 ? 16 : a.experts <= 32 ? 32 : 64, e = lane % P, per = 64 / P;
    int tot = 0, bef = 0;
#pragma unroll 8
    for (int b = wave * per + lane / P; b < blocks; b += 16 * per) {
        const int c = e < a.experts ? a.counts[(int64_t)b * a.experts + e] : 0;
        tot += c;
        bef += b < (int)blockIdx.x ? c : 0;
    }
    for (int off = P; off < 64; off <<= 1) { tot += __shfl_xor(tot, off, 64); bef += __shfl_xor(bef, off, 64); }
    total[wave][lane] = lane < P ? tot : 0;
    before[wave][lane] = lane < P ? bef : 0;
    __syncthreads();
    if (wave == 0) {
        int rows_e = 0, in_front = 0, start;
#pragma unroll
        for (int i = 0; i < 16; ++i) { rows_e += total[i][lane]; in_front += before[i][lane]; }
        moe_group_list(a, rows_e, lane, start, first_tile);
        starts[lane] = start;
        place[lane] = start + in_front;
    }
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * rows_per_block * a.top, i1 = i0 + rows_per_block * a.top < a.N * a.top ? i0 + rows_per_block * a.top : a.N * a.top;
    for (int64_t i = i0 + tid; i < i1; i += 1024) {
        const int x = a.ids[i];
        if (x >= 0 && x < a.experts) a.perm[atomicAdd(&place[x], 1)] = (int32_t)i;
    }
    if (blockIdx.x == 0) moe_tile_list(a, starts, first_tile, tid, 1024);
}

// ---- the same choice for the few tokens of a decode, a workgroup each, which group nothing (moe_few_kernel finds an expert's rows among the choices) -------------------------------------
// What bounds it is what a CU takes in (all of W: 64 KB in 5 us of launch and choice included, 256 KB in 9) and the exchanges of the choice; the outputs are dealt out to sixteen wavefronts, each of
// which has 2048 (up to 32 outputs) or 1024 depths of its outputs' rows on the way at once.  us, one workgroup for 32 tokens / in four slices and another launch / so: 32 x 1024 bfloat16 by 16 13.5 / - / 4.9,
// 32 x 2048 float by 32 - / 17 / 8.7.
constexpr int RF_NW = 16;
template <typename TX, int RF_E>                                    // outputs of each of the wavefronts, at most
__global__ __launch_bounds__(64 * RF_NW) void moe_router_few_kernel(jl_moe_router a) {
    __shared__ float z[MR_MAX_E];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int64_t n = blockIdx.x;
    if (!a.w) {
        if (tid < a.E) z[tid] = ((const float *)a.x)[n * a.E + tid];
    } else {
        const TX *x = (const TX *)a.x + n * a.x_ld;
        float sum[RF_E] = {};
        auto of = [&](int i) { const int e = wave + RF_NW * i; return a.w + (int64_t)(e < a.E ? e : a.E - 1) * a.K; };
        const int outputs = (a.E - wave + RF_NW - 1) / RF_NW;       // of this wavefront; none and fewer are the same for all lanes
        constexpr int AHEAD = RF_E > 2 ? 4 : 8;
        for (int k0 = 0; k0 < a.K; k0 += 256 * AHEAD) {             // four values per lane, of AHEAD pieces of 256
            float xv[AHEAD][4];
            float4 wv[RF_E][AHEAD];
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) {
                const int k = k0 + 256 * s + 4 * lane, at = k < a.K ? k : 0;
                ld4_f(x + at, xv[s]);
#pragma unroll
                for (int i = 0; i < RF_E; ++i)
                    if (i < outputs) wv[i][s] = *(const float4 *)(of(i) + at);
            }
#pragma unroll
            for (int i = 0; i < RF_E; ++i)
                if (i < outputs)
#pragma unroll
                    for (int s = 0; s < AHEAD; ++s) {
                        const bool in = k0 + 256 * s + 4 * lane < a.K;      // a weight that is not finite counts where it is, not beyond the depth
                        sum[i] = in ? fmaf(xv[s][3], wv[i][s].w, fmaf(xv[s][2], wv[i][s].z, fmaf(xv[s][1], wv[i][s].y, fmaf(xv[s][0], wv[i][s].x, sum[i])))) : sum[i];
                    }
        }
#pragma unroll
        for (int i = 0; i < RF_E; ++i)
            if (i < outputs) {
                const float s = wave_sum_f32(sum[i]);
                const int e = wave + RF_NW * i;
                if (lane == 0) z[e] = a.bias ? s + a.bias[e] : s;
            }
    }
    __syncthreads();
    if (wave > 0) return;
    const float *const zr[1] = {z};
    moe_route_rows<64, 1>(zr, a.correction, a.E, a.top, a.kind, a.scale, a.renorm_eps, lane, [&](int, int s, int e, float weight) {
        a.ids[n * a.top + s] = e;
        a.weights[n * a.top + s] = weight;
    });
}

extern "C" int jl_moe_router_blocks(int64_t N) { return (int)(N <= 16 ? 1 : (N + 31) / 32 < 0x7fffffff ? (N + 31) / 32 : 0x7fffffff); }
// The product in four slices of the depth, in front of the choice, where a workgroup would take in half a MB of x and W by itself.  us of product, choice and grouping, one / four slices: 32 x 2048 float
// by 32 outputs 20.6 / 12.9 (two 15.9, eight 13.1), by 40 27.7 / 17.0, 128 by 32 23.1 / 15.1, 1 by 32 12.7 / 8.7, 48 x 2048 bfloat16 by 32 24.7 / 15.9, 1400 x 1024 float by 20 15.4 / 13.5; below the
// line it saves less than a launch costs: 32 x 1024 bfloat16 by 16 10.3 / 8.7, 1 token 6.6 / 6.8.
extern "C" int jl_moe_router_slices(int64_t N, int32_t E, int32_t K) { return jl_moe_router_blocks(N) <= 64 && (int64_t)K * ((E + 15) / 16) >= 2048 ? 4 : 1; }
extern "C" int jl_moe_router_run(const jl_moe_router *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_moe_router_run: null arguments");
    const jl_moe_router &a = *ap;
    if (a.N <= 0) return JL_OK;
    const int blocks = jl_moe_router_blocks(a.N);
    bool logits = !a.w;
    if (!a.x || !a.ids || !a.weights || !a.perm || !a.offsets || !a.tile_expert || !a.tile_row0 || (blocks > 1 && !a.counts)) return jl_fail(JL_E_INVALID, "jl_moe_router_run: null pointer");
    if (a.E <= 0 || a.E > MR_MAX_E || a.experts <= 0 || a.experts > a.E || a.top <= 0 || a.top > a.E || a.kind < JL_ROUTE_SIGMOID || a.kind > JL_ROUTE_TOP_SOFTMAX)
        return jl_fail(JL_E_INVALID, "jl_moe_router_run: up to %d router outputs, experts and choices among them", MR_MAX_E);
    if (a.N * a.top > INT32_MAX || blocks > JL_MOE_ROUTER_BLOCKS || a.tile_rows <= 0 || (int64_t)a.max_tiles < a.N * a.top / a.tile_rows + a.experts)
        return jl_fail(JL_E_INVALID, "jl_moe_router_run: up to %d tokens and max_tiles >= rows / tile_rows + experts", 32 * JL_MOE_ROUTER_BLOCKS);
    const int unit = a.x_dtype == JL_BF16 ? 8 : 4;
    if (logits && (a.x_dtype != JL_F32 || a.bias)) return jl_fail(JL_E_INVALID, "jl_moe_router_run: logits are float and whole");
    if (!logits && ((a.x_dtype != JL_BF16 && a.x_dtype != JL_F32) || a.K <= 0 || a.K % 4 || a.x_ld < a.K || a.x_ld % unit || (((uintptr_t)a.x | (uintptr_t)a.w) & 15)))
        return jl_fail(JL_E_INVALID, "jl_moe_router_run: rows of x and W at 16-byte borders");
    hipStream_t st = (hipStream_t)stream;
#define MR_CASE(NT, OT)                                                                                                          \
    do {                                                                                                                          \
        if (logits) moe_router_kernel<float, NT, OT, true><<<dim3((unsigned)blocks), 64 * MR_NW, 0, st>>>(a);                      \
        else JL_DISPATCH(a.x_dtype, moe_router_kernel<T, NT, OT, false><<<dim3((unsigned)blocks), 64 * MR_NW, 0, st>>>(a));        \
    } while (0)
    const int ot = (a.E + 15) / 16;
    if (a.slices > 1) {
        if (logits || !a.parts) return jl_fail(JL_E_INVALID, "jl_moe_router_run: slices of a product, and room for them");
#define MR_PART(NT, OT) JL_DISPATCH(a.x_dtype, moe_router_part_kernel<T, NT, OT><<<dim3((unsigned)blocks, (unsigned)a.slices), 64 * MR_NW, 0, st>>>(a))
        if (a.N <= 16) { if (ot == 1) MR_PART(1, 1); else if (ot == 2) MR_PART(1, 2); else if (ot == 3) MR_PART(1, 3); else MR_PART(1, 4); }
        else { if (ot == 1) MR_PART(2, 1); else if (ot == 2) MR_PART(2, 2); else if (ot == 3) MR_PART(2, 3); else MR_PART(2, 4); }
#undef MR_PART
        logits = true;
    }
    if (a.N <= 16) { if (ot == 1) MR_CASE(1, 1); else if (ot == 2) MR_CASE(1, 2); else if (ot == 3) MR_CASE(1, 3); else MR_CASE(1, 4); }
    else { if (ot == 1) MR_CASE(2, 1); else if (ot == 2) MR_CASE(2, 2); else if (ot == 3) MR_CASE(2, 3); else MR_CASE(2, 4); }
#undef MR_CASE
    if (blocks > 1) moe_place_kernel<<<dim3((unsigned)blocks), 1024, 0, st>>>(a, 32);
    return jl_check_launch("moe_router_kernel");
}

// ---- grouped product, any dtype and size: a 64 x 64 tile of one expert's rows per workgroup, float FMAs ------------------------------------

// GATED: W holds 2 * n_out rows per expert, gate rows on linear rows; a tile forms both products of its columns and stores the unit
template <typename T, bool GATED>
__global__ __launch_bounds__(256) void moe_gemm_kernel(const T *__restrict__ X, const T *__restrict__ Wt, int mode, int K, int n_out, int top,
                                                        const int32_t *__restrict__ perm, const int32_t *__restrict__ offsets,
                                                        const int32_t *__restrict__ tile_expert, const int32_t *__restrict__ tile_row0,
                                                        const float *__restrict__ weights, void *__restrict__ out, MoeAct act, int tile_rows) {
    __shared__ float Xs[MOE_TM][MOE_TK + 1];
    __shared__ float Ws[(GATED ? 2 : 1) * MOE_TN][MOE_TK + 1];
    __shared__ int rin[MOE_TM];
    const int e = tile_expert[blockIdx.x];
    if (e < 0) return;
    const int r0 = tile_row0[blockIdx.x] + blockIdx.z * MOE_TM, left = offsets[e + 1] - r0 < tile_rows - (int)blockIdx.z * MOE_TM ? offsets[e + 1] - r0 : tile_rows - (int)blockIdx.z * MOE_TM;
    const int nr = left < MOE_TM ? left : MOE_TM;
    if (nr <= 0) return;
    const int n0 = blockIdx.y * MOE_TN;
    const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
    if (tid < MOE_TM) rin[tid] = tid < nr ? (mode != 1 ? perm[r0 + tid] / top : r0 + tid) : -1;
    const T *We = Wt + (int64_t)e * (GATED ? 2 : 1) * n_out * K;
    float acc[4][4] = {};
    float acu[GATED ? 4 : 1][4] = {};
    for (int k0 = 0; k0 < K; k0 += MOE_TK) {
        __syncthreads();
        for (int i = tid; i < MOE_TM * MOE_TK; i += 256) {
            const int m = i / MOE_TK, kk = i - m * MOE_TK;
            Xs[m][kk] = (rin[m] >= 0 && k0 + kk < K) ? ld_f(X + (int64_t)rin[m] * K + k0 + kk) : 0.f;
        }
        for (int i = tid; i < MOE_TN * MOE_TK; i += 256) {
            const int n = i / MOE_TK, kk = i - n * MOE_TK;
            Ws[n][kk] = (n0 + n < n_out && k0 + kk < K) ? ld_f(We + (int64_t)(n0 + n) * K + k0 + kk) : 0.f;
            if (GATED) Ws[MOE_TN + n][kk] = (n0 + n < n_out && k0 + kk < K) ? ld_f(We + (int64_t)(n_out + n0 + n) * K + k0 + kk) : 0.f;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < MOE_TK; ++kk) {
            float av[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) av[a] = Xs[ty + 16 * a][kk];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float w = Ws[tx + 16 * c][kk];
#pragma unroll
                for (int a = 0; a < 4; ++a) acc[a][c] += av[a] * w;
                if (GATED) {
                    const float wu = Ws[MOE_TN + tx + 16 * c][kk];
#pragma unroll
                    for (int a = 0; a < 4; ++a) acu[GATED ? a : 0][c] += av[a] * wu;
                }
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int m = ty + 16 * a;
        if (m >= nr) continue;
        const int r = r0 + m;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int n = n0 + tx + 16 * c;
            if (n >= n_out) continue;
            if (GATED) {
                st_f((T *)out + (int64_t)r * n_out + n, gated_unit_f(acc[a][c], acu[GATED ? a : 0][c], act.kind, act.limit, act.alpha, act.shift));
            } else if (mode == JL_MOE_UP_PLAIN) {
                st_f((T *)out + (int64_t)r * n_out + n, acc[a][c]);
            } else if (mode == 0) {
                const float v = fmaxf(acc[a][c], 0.f);
                st_f((T *)out + (int64_t)r * n_out + n, v * v);
            } else {
                const int p = perm[r];
                ((float *)out)[(int64_t)p * n_out + n] = acc[a][c] * weights[p];
            }
        }
    }
}

// ---- grouped product on the matrix cores -------------------------------------------------------------------------------------------------
// A tile of TM rows of one expert by WR of its weight rows, both K-major, walked in stages of TKU 16-byte units per row (8 bfloat16 or 4 floats each)
// through two LDS buffers: the next stage's units travel from memory while this one is multiplied, one barrier per stage.  NW wavefronts (two over the
// rows when TM is 128) hold 32 x 32 accumulators; the rows are the A operand, the weights the B operand, so that a lane ends with sixteen rows of ONE output
// column and 32 lanes store neighbouring ones (moe_store).  A lane's operand is one 16-byte unit: in bfloat16 the eight depths 8 (lane / 32) .. of
// v_mfma_f32_32x32x16_bf16; in float four v_mfma_f32_32x32x2_f32, one for each of its floats (the depths meet in the order 0, 4, 1, 5, ..: a sum of
// products rounded one by one, as a chain of multiply-adds is).  Units of a row are permuted so that 16 neighbouring rows meet different banks.
// GATED: the WR weight rows are WR / 2 of the gate and the WR / 2 of the linear branch that belong to them (rows n_out further on); both products
// of a column end in the same lane, which stores the gated unit.
// TM = 128 (an expert has about a hundred rows or more) is bound by the matrix cores and LDS: 128 x 256 reads 48 KB of LDS per 64 products.  Rows go from memory straight into LDS
// (16 bytes per lane, every lane fetching the unit that the permutation puts into its place), one stage ahead: no registers and no LDS writes for them, so that three workgroups fit a
// CU and cover each other's barriers (through registers, two of them: gated product at 8192 x 4 of 32 experts of 2048 x 1024 406 -> 363 us, the way down 290 -> 252).  More stages ahead in fewer
// workgroups change nothing; without their loads the two products take 238 and 160 us, without their products 335 and 200, so where rows are many the gated one goes in larger tiles (below).
// Workgroups of an XCD (every eighth) take neighbouring tiles and all their columns, so that an expert's weights are read into one L2.  Tiles of 32 rows (decoding) have a kernel of
// their own.
// Loads carry no branch and no 64-bit address arithmetic of their own: offsets of 32 bits from a base (of the tile where its rows lie together; FAR: rows gathered from more than
// 4 GiB have 64-bit addresses), rows that do not exist repeat another, stages behind the last repeat the
// first, depths beyond the last whole stage come after the loop (a condition per load had cost six vector instructions per product: 431 us instead of 406 for the gated product
// above).
struct MoeMM {
    const void *X, *Wt;
    const int32_t *perm, *offsets, *tile_expert, *tile_row0;
    const float *weights;
    void *out;
    int mode, K, n_out, top, E, col_blocks, max_tiles, parts;       // parts: of TM rows, that a tile of the list is walked in
    MoeAct act;
    const int32_t *ids;                                             // moe_few_kernel without a grouping: the choices of all rows, which are then where they were
    int rows;
};
typedef __bf16 mm_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 mm_bf16x2 __attribute__((ext_vector_type(2)));
typedef float mm_f32x2 __attribute__((ext_vector_type(2)));
typedef float mm_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t mm_u32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct mm_type;
template <> struct mm_type<bf16_t> {
    static constexpr int UNIT = 8;
    static __device__ __forceinline__ mm_f32x16 mma(uint4 a, uint4 b, mm_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mm_bf16x8, a), __builtin_bit_cast(mm_bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct mm_type<float> {
    static constexpr int UNIT = 4;
    static __device__ __forceinline__ mm_f32x16 mma(uint4 a, uint4 b, mm_f32x16 c) {
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
    }
};

// What a wavefront's products leave: XT x NT tiles of 32 rows (from row_of(x) of the tile's) by 32 columns (from col_of(t)); a lane has sixteen rows of column lane % 32.  A store instruction writes
// 32 neighbouring columns of two rows (float), or of four rows once neighbouring lanes have exchanged a value (bfloat16): whole lines or their halves.  (Four neighbouring columns of one row
// per lane, 32 rows per instruction: the experts of 8192 x 4 of 32 of 2048 x 1024 took 687 us instead of 647, 8192 x 4 of 16 of 1024 x 512 174 instead of 163.)
template <typename T, int XT, int NT, bool GATED, bool DOWN, typename Down, typename Rows, typename Cols, typename To>
__device__ __forceinline__ void moe_store(const MoeMM &a, const mm_f32x16 (&acc)[XT][NT], int nr, int n0, Down down, Rows row_of, Cols col_of, int lane, To to) {
    constexpr int OT = GATED ? NT / 2 : NT;
    const int n_out = a.n_out, l32 = lane & 31, hi = lane >> 5;
    const bool pairs = n_out % 2 == 0, odd = lane & 1;
#pragma unroll
    for (int x = 0; x < XT; ++x)
#pragma unroll
        for (int t = 0; t < OT; ++t) {
            const int n = n0 + col_of(t) + l32;
            if (n - l32 >= n_out) continue;                         // the whole wavefront
            const bool in = n < n_out;                              // both lanes of a pair, or neither, where columns come in pairs; all lanes take part in what crosses them
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const int m = row_of(x) + 8 * (r >> 2) + 4 * hi + (r & 3);
                float v[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float c = acc[x][t][r + i];
                    if (GATED) v[i] = gated_unit_f<sizeof(T) == 2>(c, acc[x][t + (GATED ? OT : 0)][r + i], a.act.kind, a.act.limit, a.act.alpha, a.act.shift);
                    else if (a.mode == 0) { const float q = fmaxf(c, 0.f); v[i] = q * q; }
                    else v[i] = c;
                }
                if (DOWN && a.mode == 1) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        int p;
                        float w;
                        down(x, 8 * (r >> 2) + 4 * hi + (r & 3) + i, p, w);
                        if (in && m + i < nr) ((float *)a.out)[(int64_t)p * n_out + n] = v[i] * w;
                    }
                } else if (sizeof(T) == 2 && pairs) {
                    const float other = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(odd ? v[0] : v[1]), 0xB1, 0xF, 0xF, true));      // quad_perm [1, 0, 3, 2]
                    const mm_f32x2 both = {odd ? other : v[0], odd ? v[1] : other};
                    if (in && m + odd < nr) *(uint32_t *)((bf16_t *)a.out + (int64_t)to(m + odd) * n_out + n - odd) = __builtin_bit_cast(uint32_t, __builtin_convertvector(both, mm_bf16x2));
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        if (in && m + i < nr) st_f((T *)a.out + (int64_t)to(m + i) * n_out + n, v[i]);
                }
            }
        }
}

template <typename T, int TM, int NW, int WR, int TKU, bool GATED, bool FAR>
__global__ __launch_bounds__(64 * NW, 3) void moe_mm_kernel(MoeMM a) {
    constexpr int THREADS = 64 * NW, UNIT = mm_type<T>::UNIT, WM = TM == 128 ? 2 : 1, WN = NW / WM, XT = TM / WM / 32, NT = WR / WN / 32;
    constexpr int XPF = TM * TKU / THREADS, WPF = WR * TKU / THREADS, TN = GATED ? WR / 2 : WR, STAGE = TKU * UNIT;
    static_assert(XPF * THREADS == TM * TKU && WPF * THREADS == WR * TKU && (!GATED || NT % 2 == 0), "tile");
    __shared__ uint4 smem[2 * (TM + WR) * TKU];
    __shared__ int rows_out[TM];                                    // way down: the flat indices and weights of the tile's rows
    __shared__ float rows_weight[TM];
    // workgroups with the same remainder by 8 share an XCD
    const int per_xcd = (a.offsets[a.E + 1] + 7) / 8, xcd = blockIdx.x & 7, s = blockIdx.x >> 3;
    if (s >= per_xcd * a.col_blocks * a.parts) return;
    const int tile = xcd * per_xcd + s / (a.col_blocks * a.parts), part = s / a.col_blocks % a.parts, col = s % a.col_blocks;
    if (tile >= a.max_tiles) return;
    const int e = a.tile_expert[tile];
    if (e < 0) return;
    const int r0 = a.tile_row0[tile] + part * TM, K = a.K, n_out = a.n_out, n0 = col * TN;
    if (a.offsets[e + 1] <= r0) return;
    const int nr = a.offsets[e + 1] - r0 < TM ? a.offsets[e + 1] - r0 : TM;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5, wm = wave / WN, wn = wave % WN;
    auto at = [](int row, int u) { return row * TKU + (u ^ (TKU == 4 ? (row >> 2) & 3 : (row >> 1) & 7)); };
    if (!GATED && a.mode == 1)
        for (int m = tid; m < nr; m += THREADS) {
            const int p = a.perm[r0 + m];
            rows_out[m] = p;
            rows_weight[m] = a.weights[p];
        }
    // loaders: unit tid % TKU of rows tid / TKU + x * THREADS / TKU; a row that does not exist repeats another and is not stored
    const int lr = tid / TKU;
    auto unit_of = [&](int x) { return at(lr + x * (THREADS / TKU), tid % TKU) % TKU; };      // what belongs into this thread's place of LDS
    // byte offsets from a base that is the same for all lanes: a load is one instruction (the launch has checked that 32 bits hold them)
    uint32_t xo[XPF], wo[WPF];
    const char *xfar[FAR ? XPF : 1];
    const char *Xb = (const char *)((const T *)a.X + (a.mode != 1 ? 0 : (int64_t)r0 * K));
#pragma unroll
    for (int x = 0; x < XPF; ++x) {
        const int m = lr + x * (THREADS / TKU), row = m < nr ? m : 0;
        const int64_t at_x = (a.mode != 1 ? a.perm[r0 + row] / a.top : row) * (int64_t)K + unit_of(x) * UNIT;
        if constexpr (FAR) xfar[x] = Xb + at_x * sizeof(T);
        xo[x] = (uint32_t)at_x * sizeof(T);
    }
    // the first half of a gated tile's rows are the gate's, the others the linear branch's, n_out further on
    const char *Wb = (const char *)((const T *)a.Wt + ((int64_t)e * (GATED ? 2 : 1) * n_out + n0) * K), *Wl = Wb + (int64_t)(GATED ? n_out : 0) * K * sizeof(T);
#pragma unroll
    for (int x = 0; x < WPF; ++x) {
        const int j = lr + x * (THREADS / TKU), c = GATED ? j % TN : j;
        wo[x] = (uint32_t)((n0 + c < n_out ? c : n_out - 1 - n0) * (int64_t)K + unit_of(x) * UNIT) * sizeof(T);
    }
    auto w_base = [&](int x) { return GATED && x >= WPF / 2 ? Wl : Wb; };
    const int full = K / STAGE;                                     // whole stages; what is left of K comes last
    mm_f32x16 acc[XT][NT];
#pragma unroll
    for (int x = 0; x < XT; ++x)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[x][t][i] = 0.f;
    // weight row (within the tile) of this wavefront's tile t: gate tiles first, then the linear branch's
    auto w_row = [&](int t) { return GATED ? (t < NT / 2 ? 0 : TN) + wn * (TN / WN) + 32 * (t % (NT / 2 > 0 ? NT / 2 : 1)) : wn * (WR / WN) + 32 * t; };
    auto products = [&](int sel) {
        const uint4 *Xs = smem + sel * (TM + WR) * TKU, *Ws = Xs + TM * TKU;
#pragma unroll
        for (int s = 0; s < TKU / 2; ++s) {
            uint4 xf[XT], wf[NT];
#pragma unroll
            for (int x = 0; x < XT; ++x) xf[x] = Xs[at(wm * (TM / WM) + 32 * x + l32, 2 * s + hi)];
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t] = Ws[at(w_row(t) + l32, 2 * s + hi)];

#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int x = 0; x < XT; ++x) acc[x][t] = mm_type<T>::mma(xf[x], wf[t], acc[x][t]);

        }
    };
    if (full > 0) {
        // straight into LDS: a wavefront's 64 places of 16 bytes per load, one stage ahead
        const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)(smem + wave * 64));
        auto issue = [&](int i, int sel) {
            const int64_t k = i < full ? (int64_t)i * STAGE * sizeof(T) : 0;
            const uint32_t dst = lds + sel * (TM + WR) * TKU * 16;
#pragma unroll
            for (int x = 0; x < XPF; ++x) {
                if constexpr (FAR) jl_load_lds_far(xfar[x] + k, dst + x * THREADS * 16);
                else jl_load_lds(Xb + k, xo[x], dst + x * THREADS * 16);
            }
#pragma unroll
            for (int x = 0; x < WPF; ++x) jl_load_lds(w_base(x) + k, wo[x], dst + (XPF + x) * THREADS * 16);
        };
        issue(0, 0);
        for (int i = 0; i < full; ++i) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // stage i is in LDS; everybody has read stage i - 1, whose place is free
            __syncthreads();
            issue(i + 1, (i + 1) & 1);
            products(i & 1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    if (full * STAGE < K) {                                         // depths beyond K are zero
        const mm_u32x4 zero = {0, 0, 0, 0};
        auto last = [&](const char *from, int u) {                  // a lane beyond K reads its row's first unit: a row may be shorter than a stage
            const bool in = full * STAGE + u * UNIT < K;
            const mm_u32x4 v = *(const mm_u32x4 *)(from + (in ? (int64_t)full * STAGE * sizeof(T) : -(int64_t)(u * UNIT * sizeof(T))));
            return in ? v : zero;
        };
#pragma unroll
        for (int x = 0; x < XPF; ++x) smem[tid + x * THREADS] = __builtin_bit_cast(uint4, last(FAR ? xfar[FAR ? x : 0] : Xb + xo[x], unit_of(x)));
#pragma unroll
        for (int x = 0; x < WPF; ++x) smem[tid + (XPF + x) * THREADS] = __builtin_bit_cast(uint4, last(w_base(x) + wo[x], unit_of(x)));
        __syncthreads();
        products(0);
    }
    moe_store<T, XT, NT, GATED, !GATED>(a, acc, nr, n0, [&](int x, int k, int &p, float &w) { const int m = wm * (TM / WM) + 32 * x + k; p = rows_out[m]; w = rows_weight[m]; },
                                [&](int x) { return wm * (TM / WM) + 32 * x; }, w_row, lane, [&](int m) { return r0 + m; });
}

// ---- the same product for few rows per expert (decoding): 32 rows by 64 weight rows, the depth shared by two or four wavefronts ----------------------
// What bounds it is reading the weights, and with few tiles the way there: one wavefront has 24 KB of its share of the depth on the way in registers, passes it through LDS of its own (no barrier) into the
// products, and the shares meet in the end.  Rows of x come eight at a time, as many as there are.  (Three workgroups of four per CU do not fit the registers: spills, 106 us for the first line.)
// us of both products, gated, weights from memory, one wavefront with all of the depth / two / four: 32 rows x 4 of 32 of 2048 x 1024 92 / 79 / 80 (402 MB: 5.0 TB/s), 1 x 4 of the same 28 / 21 / 19, 32 x 4 of
// 16 of 1024 x 512 (plain) 22 / 18 / 16, 100 x 3 of 24 of 1536 x 704 37 / 37 / 41, 400 x 4 of 16 (plain) 27 / 25 / 28; float, 16 x 4 of 16 of 1024 x 512 62 / 38 / 27, 150 x 4 66 / 65 / 46.
template <typename T, int MF_NW, bool GATED, bool FAR, bool LIST = false, int WR = 64>
__global__ __launch_bounds__(64 * MF_NW, 2) void moe_few_kernel(MoeMM a) {
    constexpr int TM = 32, TKU = 8, NT = WR / 32, XPF = TM * TKU / 64, WPF = WR * TKU / 64, TN = GATED ? WR / 2 : WR, UNIT = mm_type<T>::UNIT, STAGE = TKU * UNIT, OWN = (TM + WR) * TKU;
    __shared__ uint4 smem[MF_NW * OWN];
    __shared__ int rows_out[TM];                                    // way down: the flat indices and weights of the tile's rows
    __shared__ float rows_weight[TM];
    const int tile = blockIdx.x / a.col_blocks, e = LIST ? tile % a.E : a.tile_expert[tile];
    if (!LIST && e < 0) return;
    const int K = a.K, n_out = a.n_out, n0 = (int)(blockIdx.x - tile * a.col_blocks) * TN, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5;
    auto at = [](int row, int u) { return row * TKU + (u ^ ((row >> 1) & 7)); };
    // loaders: unit lane % 8 of rows lane / 8 + 8 x; a row that does not exist repeats another and is not stored.  Byte offsets from a base that is the same for all lanes
    const int lr = lane / TKU, lu = lane % TKU, full = K / STAGE, s0 = full * wave / MF_NW, s1 = full * (wave + 1) / MF_NW;      // whole stages; what is left of K is the last wavefront's
    uint32_t xo[XPF], wo[WPF];
    mm_u32x4 reg[2][XPF + WPF];
    const char *Wb = (const char *)((const T *)a.Wt + ((int64_t)e * (GATED ? 2 : 1) * n_out + n0) * K), *Wl = Wb + (int64_t)(GATED ? n_out : 0) * K * sizeof(T);
#pragma unroll
    for (int x = 0; x < WPF; ++x) {
        const int j = lr + 8 * x, c = GATED ? j % TN : j;
        wo[x] = (uint32_t)((n0 + c < n_out ? c : n_out - 1 - n0) * (int64_t)K + lu * UNIT) * sizeof(T);
    }
    auto w_base = [&](int x) { return GATED && x >= WPF / 2 ? Wl : Wb; };
    int r0 = 0, nr;
    if constexpr (LIST) {
        // the rows from 32 * (tile / E) on of this expert's, in order: every wavefront looks through the choices by itself, and all write the same
        const int first = tile / a.E * TM;
        int found = 0;
        for (int i0 = 0; i0 < a.rows; i0 += 256) {
            int id[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) { const int r = i0 + 64 * i + lane; id[i] = a.ids[r < a.rows ? r : a.rows - 1]; }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = i0 + 64 * i + lane;
                const uint64_t mine = __ballot(r < a.rows && id[i] == e);
                const int m = found + __popcll(mine & ((1ull << lane) - 1)) - first;
                if ((mine >> lane & 1) && m >= 0 && m < TM) rows_out[m] = r;
                found += __popcll(mine);
            }
        }
        nr = found - first < TM ? found - first : TM;
        if (nr <= 0) return;                                        // the whole workgroup
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (!GATED && a.mode == 1 && (int)threadIdx.x < nr) rows_weight[threadIdx.x] = a.weights[rows_out[threadIdx.x]];
    } else {
        r0 = a.tile_row0[tile];
        const int left = a.offsets[e + 1] - r0;
        nr = left < TM ? left : TM;
        if (!GATED && a.mode == 1 && (int)threadIdx.x < nr) {
            const int p = a.perm[r0 + threadIdx.x];
            rows_out[threadIdx.x] = p;
            rows_weight[threadIdx.x] = a.weights[p];
        }
    }
    const char *xfar[FAR ? XPF : 1];
    const char *Xb = (const char *)((const T *)a.X + (a.mode != 1 || LIST ? 0 : (int64_t)r0 * K));
#pragma unroll
    for (int x = 0; x < XPF; ++x) {
        const int m = lr + 8 * x, row = m < nr ? m : 0;
        const int from = LIST ? rows_out[row] : a.mode != 1 ? a.perm[r0 + row] : row;
        const int64_t at_x = (a.mode != 1 ? from / a.top : from) * (int64_t)K + lu * UNIT;
        if constexpr (FAR) xfar[x] = Xb + at_x * sizeof(T);
        xo[x] = (uint32_t)at_x * sizeof(T);
    }
    auto fetch = [&](mm_u32x4 (&r)[XPF + WPF], int i) {             // behind the last stage, the first again (never used)
        const int64_t k = i < s1 ? (int64_t)i * STAGE * sizeof(T) : 0;
#pragma unroll
        for (int x = 0; x < XPF; ++x) {
            if (8 * x >= nr) continue;                              // the same for all lanes: LDS keeps whatever lies there, for rows that are not stored
            if constexpr (FAR) r[x] = *(const mm_u32x4 *)(xfar[x] + k);
            else r[x] = *(const mm_u32x4 *)(Xb + k + xo[x]);
        }
#pragma unroll
        for (int x = 0; x < WPF; ++x) r[XPF + x] = *(const mm_u32x4 *)(w_base(x) + k + wo[x]);
    };
    uint4 *Xs = smem + wave * OWN, *Ws = Xs + TM * TKU;
    auto sync = [] {                                                // LDS written by some lanes is read by others of the same wavefront
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto stash = [&](const mm_u32x4 (&r)[XPF + WPF]) {
        sync();
#pragma unroll
        for (int x = 0; x < XPF; ++x)
            if (8 * x < nr) Xs[at(lr + 8 * x, lu)] = __builtin_bit_cast(uint4, r[x]);
#pragma unroll
        for (int x = 0; x < WPF; ++x) Ws[at(lr + 8 * x, lu)] = __builtin_bit_cast(uint4, r[XPF + x]);
        sync();
    };
    mm_f32x16 acc[1][NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][t][i] = 0.f;
    auto products = [&]() {
#pragma unroll
        for (int s = 0; s < TKU / 2; ++s) {
            const uint4 xf = Xs[at(l32, 2 * s + hi)];
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[0][t] = mm_type<T>::mma(xf, Ws[at(32 * t + l32, 2 * s + hi)], acc[0][t]);
        }
    };
    if (s0 < s1) {
        fetch(reg[0], s0);
        fetch(reg[1], s0 + 1);
        for (int i = s0; i < s1; i += 2) {                          // two stages ahead: a trip to memory takes longer than one stage's products
            stash(reg[0]);
            fetch(reg[0], i + 2);
            products();
            if (i + 1 >= s1) break;
            stash(reg[1]);
            fetch(reg[1], i + 3);
            products();
        }
    }
    if (full * STAGE < K && wave == MF_NW - 1) {                    // depths beyond K are zero; a lane beyond K reads its row's first unit: a row may be shorter than a stage
        const mm_u32x4 zero = {0, 0, 0, 0};
        const bool in = full * STAGE + lu * UNIT < K;
        const int64_t k = in ? (int64_t)full * STAGE * sizeof(T) : -(int64_t)(lu * UNIT * sizeof(T));
#pragma unroll
        for (int x = 0; x < XPF; ++x) { const mm_u32x4 v = *(const mm_u32x4 *)((FAR ? xfar[FAR ? x : 0] : Xb + xo[x]) + k); reg[0][x] = in ? v : zero; }
#pragma unroll
        for (int x = 0; x < WPF; ++x) { const mm_u32x4 v = *(const mm_u32x4 *)(w_base(x) + wo[x] + k); reg[0][XPF + x] = in ? v : zero; }
        stash(reg[0]);
        products();
    }
    // the shares meet: the first wavefront adds them in order
    sync();
    ls_f32x4 *mine = (ls_f32x4 *)Xs;
    if (wave > 0)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) mine[(4 * t + g) * 64 + lane] = ls_f32x4{acc[0][t][4 * g], acc[0][t][4 * g + 1], acc[0][t][4 * g + 2], acc[0][t][4 * g + 3]};
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 1; w < MF_NW; ++w)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const ls_f32x4 v = ((const ls_f32x4 *)(smem + w * OWN))[(4 * t + g) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[0][t][4 * g + i] += v[i];
            }
    moe_store<T, 1, NT, GATED, !GATED>(a, acc, nr, n0, [&](int, int k, int &p, float &w) { p = rows_out[k]; w = rows_weight[k]; }, [](int) { return 0; },
                                       [&](int t) { return 32 * t; }, lane, [&](int m) { return LIST ? rows_out[m] : r0 + m; });
}

// ---- the same product in tiles of 256 rows by 256 weight rows (bfloat16, depths in whole stages of 64) ----------------------------------------
// What bounds the tiles of 128 rows where experts have hundreds of rows each is not the matrix cores but the way from L2 into LDS (without their products they take 335 of 395 us for the gated product at 8192 x 4
// of 32 experts of 2048 x 1024: 3.4 GB at 10 TB/s).  Tiles of 256 x 256 move a third less, in whole lines of 128 bytes.  One workgroup of eight wavefronts (128 rows x 64 weight rows each, two per SIMD) per CU
// walks tile after tile: the next tile's first stage travels while the last stage of this one is multiplied, and this one's results leave while the next is multiplied.  A tile of at most 128 rows
// (an expert's last) takes half the products: the row blocks of 32 alternate between the two rows of wavefronts.
// Gated product of 8192 x 4 of 32 experts of 2048 x 1024: 395 -> 330 us (830 TFLOP/s); without loads 229, without products 235, without results 300.  Three stages of W in LDS instead of two,
// so that its lines from memory have twice the time, change nothing, nor do other orders of the depths per column; on the way down the results of a whole round (67 MB) leave at once and
// make up for the rest: 245 us against 236 of three smaller workgroups per CU.
template <bool GATED>
__global__ __launch_bounds__(512, 2) void moe_big_kernel(MoeMM a) {
    constexpr int TKU = 8, STAGE = 64, XT = 4, NT = 2, TN = GATED ? 128 : 256, BUF = 512 * TKU;
    __shared__ uint4 smem[2 * BUF];                                 // [2][rows of X, rows of W][8 units]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hi = lane >> 5, wm = wave >> 2, wn = wave & 3;
    const int K = a.K, n_out = a.n_out, full = K / STAGE, in_use = __builtin_amdgcn_readfirstlane(a.offsets[a.E + 1]), tiles = in_use < a.max_tiles ? in_use : a.max_tiles;
    const int per_xcd = (tiles + 7) / 8, first = (blockIdx.x & 7) * per_xcd, slots = gridDim.x / 8;      // workgroups with the same remainder by 8 share an XCD: neighbouring tiles and all their columns
    const int here = tiles - first < per_xcd ? tiles - first : per_xcd;
    auto at = [](int row, int u) { return row * TKU + (u ^ ((row >> 1) & 7)); };
    auto w_row = [&](int t) { return GATED ? t * TN + wn * 32 : wn * 64 + 32 * t; };
    struct Tile { int e, r0, nr, n0; };
    auto tile_at = [&](int q) {
        const int t = first + q / a.col_blocks, e = __builtin_amdgcn_readfirstlane(a.tile_expert[t]), r0 = __builtin_amdgcn_readfirstlane(a.tile_row0[t]);
        const int left = __builtin_amdgcn_readfirstlane(a.offsets[e + 1]) - r0;
        return Tile{e, r0, left < 256 ? left : 256, (q % a.col_blocks) * TN};
    };
    // loaders: the unit that belongs into this thread's place of LDS, of rows tid / 8 + 64 x of X and of W; a row that does not exist repeats another and is not stored
    const int lr = tid >> 3, unit = (tid & 7) ^ ((lr >> 1) & 7);
    uint32_t xo[XT], wo[4];
    const char *const Xb = (const char *)a.X, *Wb, *Wl;
    bool half;                                                      // at most 128 rows
    auto aim = [&](const Tile &t, const int (&row)[XT]) {
        Wb = (const char *)a.Wt + ((int64_t)t.e * (GATED ? 2 : 1) * n_out + t.n0) * K * 2;
        Wl = Wb + (int64_t)(GATED ? n_out : 0) * K * 2;
        half = t.nr <= 128;
#pragma unroll
        for (int x = 0; x < XT; ++x) {
            xo[x] = (uint32_t)(row[x] / a.top) * (uint32_t)(K * 2) + unit * 16;
            const int j = lr + 64 * x, c = GATED ? j % TN : j;
            wo[x] = (uint32_t)(t.n0 + c < n_out ? c : n_out - 1 - t.n0) * (uint32_t)(K * 2) + unit * 16;
        }
    };
    auto rows_of = [&](const Tile &t, int (&row)[XT]) {
#pragma unroll
        for (int x = 0; x < XT; ++x) {
            const int m = lr + 64 * x < t.nr ? lr + 64 * x : 0;
            row[x] = a.perm[t.r0 + m];                              // divided by `top` where it is used: the load need not be waited for here
        }
    };
    const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)(smem + wave * 64));
    auto issue = [&](int i, int sel, int part) {                     // the rows of X (part 0) or of W (1) of stage i into buffer `sel`
        const int64_t k = (int64_t)i * STAGE * 2;
        const uint32_t dst = lds + sel * BUF * 16;
        if (part == 0) {
#pragma unroll
            for (int x = 0; x < XT; ++x)
                if (x < XT / 2 || !half) jl_load_lds(Xb + k, xo[x], dst + x * 512 * 16);
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x) jl_load_lds((GATED && x >= 2 ? Wl : Wb) + k, wo[x], dst + (XT + x) * 512 * 16);
        }
    };
    auto products = [&](int sel, auto &acc, auto beside) {
        constexpr int NX = sizeof(acc) / sizeof(acc[0]);
        const uint4 *Xs = smem + sel * BUF, *Ws = Xs + 256 * TKU;
#pragma unroll
        for (int s = 0; s < TKU / 2; ++s) {
            uint4 xf[NX], wf[NT];
#pragma unroll
            for (int x = 0; x < NX; ++x) xf[x] = Xs[at(64 * x + 32 * wm + l32, 2 * s + hi)];
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t] = Ws[at(w_row(t) + l32, 2 * s + hi)];
            beside(s);
            __builtin_amdgcn_s_setprio(1);                          // whoever has its operands multiplies; the SIMD's other wavefront reads meanwhile
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int x = 0; x < NX; ++x) acc[x][t] = mm_type<bf16_t>::mma(xf[x], wf[t], acc[x][t]);
            __builtin_amdgcn_s_setprio(0);
        }
    };
    const int n_q = here * a.col_blocks;
    int q = blockIdx.x >> 3;
    if (q >= n_q) return;                                           // the whole workgroup
    Tile now = tile_at(q);
    int row[XT], sel = 0;
    rows_of(now, row);
    aim(now, row);
    issue(0, 0, 0);
    issue(0, 0, 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // one tile: stage 0 of it is in buffer `sel`, as far as this wavefront loaded it.  False behind the last
    auto walk = [&](auto n_x) {
        constexpr int NX = decltype(n_x)::value;
        const bool more = q + slots < n_q;
        Tile next = now;
        if (more) {
            next = tile_at(q + slots);
            rows_of(next, row);
        }
        mm_f32x16 acc[NX][NT];
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[x][t][i] = 0.f;
        for (int i = 0; i + 1 < full; ++i) {
            if (i > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();                                        // stage i is in LDS; everybody has read what the other buffer held
            products(sel, acc, [&](int s) { if (s < 2) issue(i + 1, sel ^ 1, s); });
            sel ^= 1;
        }
        if (full > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (more) {
            aim(next, row);
            issue(0, sel ^ 1, 0);
            issue(0, sel ^ 1, 1);
        }
        products(sel, acc, [](int) {});
        sel ^= 1;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // the next tile's first stage, before the results: what this wavefront loaded of it is there
        moe_store<bf16_t, NX, NT, GATED, false>(a, acc, now.nr, now.n0, [](int, int, int &, float &) {}, [&](int x) { return 64 * x + 32 * wm; }, w_row, lane, [&](int m) { return now.r0 + m; });
        now = next;
        q += slots;
        return more;
    };
    while (half ? walk(std::integral_constant<int, XT / 2>()) : walk(std::integral_constant<int, XT>())) {}
}

// ---- the same product of floats for experts with many rows, on the bfloat16 matrix instructions in three terms per operand (jl_split.h) -----------------------------------------------
// 64 rows by 256 weight rows (four wavefronts), 128 by 128 (eight) where experts fill them (jl_moe_float_tiles).  us of the experts on the float instructions (64 x 256) / so: 2553 x 4 of 16 of 1024 x 512
// gated 348 / 248, plain 258 / 182, 1021 x 3 of 24 of 1024 x 1024 254 / 210, 2042 x 2 of 16 of 1024 x 512 221 / 167; error against 64 bits 9.7e-7 / 8.3e-7.
template <int TM, int WR, int NW, int WM, int TKU, bool GATED>
__global__ __launch_bounds__(64 * NW, NW / 2) void moe_split_kernel(MoeMM a) {
    constexpr int WN = NW / WM, XT = TM / WM / 32, NT = WR / WN / 32, TN = GATED ? WR / 2 : WR;
    __shared__ uint4 smem[split_units(TM, WR, TKU)];
    __shared__ int rows_out[TM];                                    // way down: the flat indices and weights of the tile's rows
    __shared__ float rows_weight[TM];
    // workgroups with the same remainder by 8 share an XCD
    const int per_xcd = (a.offsets[a.E + 1] + 7) / 8, xcd = blockIdx.x & 7, s = blockIdx.x >> 3;
    if (s >= per_xcd * a.col_blocks * a.parts) return;
    const int tile = xcd * per_xcd + s / (a.col_blocks * a.parts), part = s / a.col_blocks % a.parts, col = s % a.col_blocks;
    if (tile >= a.max_tiles) return;
    const int e = a.tile_expert[tile];
    if (e < 0) return;
    const int r0 = a.tile_row0[tile] + part * TM, K = a.K, n_out = a.n_out, n0 = col * TN, left = a.offsets[e + 1] - r0, nr = left < TM ? left : TM;
    if (nr <= 0) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, wm = wave / WN, wn = wave % WN;
    if (!GATED && a.mode == 1 && tid < nr) {
        const int p = a.perm[r0 + tid];
        rows_out[tid] = p;
        rows_weight[tid] = a.weights[p];
    }
    const float *W = (const float *)a.Wt + (int64_t)e * (GATED ? 2 : 1) * n_out * K;
    // the first half of a gated tile's rows are the gate's, the others the linear branch's, n_out further on; rows that do not exist repeat others and are not stored
    auto x_at = [&](int m) { const int row = m < nr ? m : 0; return (const float *)a.X + (int64_t)(a.mode != 1 ? a.perm[r0 + row] / a.top : r0 + row) * K; };
    auto w_at = [&](int j) { const int c = n0 + (GATED ? j % TN : j); return W + ((c < n_out ? c : n_out - 1) + (int64_t)(GATED && j >= TN ? n_out : 0)) * K; };
    auto x_row = [&](int x) { return wm * (TM / WM) + 32 * x; };
    auto w_row = [&](int t) { return GATED ? (t < NT / 2 ? 0 : TN) + wn * (TN / WN) + 32 * (t % (NT / 2 > 0 ? NT / 2 : 1)) : wn * (WR / WN) + 32 * t; };
    mm_f32x16 acc[XT][NT];
    split_products<TM, WR, NW, WM, TKU>(acc, smem, K, x_at, w_at, x_row, w_row);
    moe_store<float, XT, NT, GATED, !GATED>(a, acc, nr, n0, [&](int x, int k, int &p, float &w) { const int m = x_row(x) + k; p = rows_out[m]; w = rows_weight[m]; }, x_row, w_row, lane, [&](int m) { return r0 + m; });
}

template <typename T, int TM, int NW, int WR, int TKU> static int moe_mm_launch(MoeMM &a, bool gated, hipStream_t st) {
    const int tn = gated ? WR / 2 : WR;
    a.col_blocks = (a.n_out + tn - 1) / tn;
    const int64_t groups = (int64_t)(a.max_tiles + 7) / 8 * 8 * a.col_blocks * a.parts;
    if (groups > 0x7fffffff) return jl_fail(JL_E_INVALID, "jl_moe_gemm: too many tiles");
    const bool far = a.mode != 1 && ((int64_t)a.max_tiles * a.parts * TM / a.top + 1) * a.K * (int64_t)sizeof(T) > UINT32_MAX;      // gathered rows beyond what 32 bits reach
    auto kern = gated ? (far ? moe_mm_kernel<T, TM, NW, WR, TKU, true, true> : moe_mm_kernel<T, TM, NW, WR, TKU, true, false>)
                      : (far ? moe_mm_kernel<T, TM, NW, WR, TKU, false, true> : moe_mm_kernel<T, TM, NW, WR, TKU, false, false>);
    kern<<<dim3((unsigned)groups), 64 * NW, 0, st>>>(a);
    return jl_check_launch("moe_mm_kernel");
}
template <typename T> static int moe_mm_rows(MoeMM &a, int tile_rows, bool gated, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        if (tile_rows == 256) {
            a.parts = 2;
            if (a.mode == 1 || !moe_big_sizes(a.K, (int64_t)a.max_tiles * 256)) return moe_mm_launch<T, 128, 4, 256, 4>(a, gated, st);
            a.col_blocks = (a.n_out + (gated ? 127 : 255)) / (gated ? 128 : 256);
            const int64_t groups = (int64_t)(a.max_tiles + 7) / 8 * 8 * a.col_blocks;
            if (groups > 0x7fffffff) return jl_fail(JL_E_INVALID, "jl_moe_gemm: too many tiles");
            (gated ? moe_big_kernel<true> : moe_big_kernel<false>)<<<dim3((unsigned)(groups < 256 ? groups : 256)), 512, 0, st>>>(a);      // one workgroup per CU
            return jl_check_launch("moe_big_kernel");
        }
        if (tile_rows == 128) return moe_mm_launch<T, 128, 4, 256, 4>(a, gated, st);
    } else if (tile_rows == 128) return jl_fail(JL_E_INVALID, "jl_moe_gemm: float tiles have 32, 64 or 256 rows");
    if (tile_rows == 64 || tile_rows == 256) {
        if constexpr (sizeof(T) == 2) return moe_mm_launch<T, 64, 4, 256, 4>(a, gated, st);
        const int tm = tile_rows == 256 ? 128 : 64, tn = (tile_rows == 256 ? 128 : 256) / (gated ? 2 : 1);
        a.parts = tile_rows / tm;
        a.col_blocks = (a.n_out + tn - 1) / tn;
        const int64_t groups = (int64_t)(a.max_tiles + 7) / 8 * 8 * a.col_blocks * a.parts;
        if (groups > 0x7fffffff) return jl_fail(JL_E_INVALID, "jl_moe_gemm: too many tiles");
        if (tm == 128) (gated ? moe_split_kernel<128, 128, 8, 4, 4, true> : moe_split_kernel<128, 128, 8, 4, 4, false>)<<<dim3((unsigned)groups), 512, 0, st>>>(a);
        else (gated ? moe_split_kernel<64, 256, 4, 1, 4, true> : moe_split_kernel<64, 256, 4, 1, 4, false>)<<<dim3((unsigned)groups), 256, 0, st>>>(a);
        return jl_check_launch("moe_split_kernel");
    }
    a.col_blocks = (a.n_out + (gated ? 31 : 63)) / (gated ? 32 : 64);
    const int64_t groups = (int64_t)a.max_tiles * a.col_blocks;
    if (groups > 0x7fffffff) return jl_fail(JL_E_INVALID, "jl_moe_gemm: too many tiles");
    const bool far = a.mode != 1 && ((int64_t)a.max_tiles * 32 / a.top + 1) * a.K * (int64_t)sizeof(T) > UINT32_MAX;
    // four wavefronts where experts have up to about eight rows, and for float (twice the bytes, a sixteenth of the matrix rate); two where more tiles fill the chip
    const bool four = sizeof(T) == 4 || a.max_tiles - a.E <= a.E / 4;
#define MF_KERNEL(NW) (gated ? (far ? moe_few_kernel<T, NW, true, true> : moe_few_kernel<T, NW, true, false>) : (far ? moe_few_kernel<T, NW, false, true> : moe_few_kernel<T, NW, false, false>))
    if (four) MF_KERNEL(4)<<<dim3((unsigned)groups), 256, 0, st>>>(a);
    else MF_KERNEL(2)<<<dim3((unsigned)groups), 128, 0, st>>>(a);
#undef MF_KERNEL
    return jl_check_launch("moe_few_kernel");
}

static int moe_gemm_launch(const void *X, const void *Wt, int dtype, int32_t mode, int32_t K, int32_t n_out, int32_t top, const int32_t *perm,
                           const int32_t *offsets, const int32_t *tile_expert, const int32_t *tile_row0, int32_t max_tiles, int32_t E, int32_t tile_rows,
                           const float *weights, void *out, const MoeAct *act, void *stream) {
    static const bool no_mfma = getenv("JL_MOE_NO_MFMA") != nullptr;      // A/B switch for measurements
    if (E <= 0 || (tile_rows != 32 && tile_rows != 64 && tile_rows != 128 && tile_rows != 256)) return jl_fail(JL_E_INVALID, "jl_moe_gemm: tiles of 32, 64, 128 or 256 rows");
    const int64_t dtype_bytes = dtype == JL_BF16 ? 2 : 4;
    MoeMM a = {X, Wt, perm, offsets, tile_expert, tile_row0, weights, out, mode, K, n_out, top, E, 0, max_tiles, 1, act ? *act : MoeAct{0, 0.f, 0.f, 0.f}, nullptr, 0};
    if (!no_mfma && moe_mm_sizes(dtype, K) && ((uintptr_t)X % 16) == 0 && ((uintptr_t)Wt % 16) == 0 && ((uintptr_t)out % 16) == 0 &&
        256 * (int64_t)K * dtype_bytes <= UINT32_MAX) {                     // a tile's rows, of X or of W
        if (dtype == JL_BF16) return moe_mm_rows<bf16_t>(a, tile_rows, act != nullptr, (hipStream_t)stream);
        return moe_mm_rows<float>(a, tile_rows, act != nullptr, (hipStream_t)stream);
    }
    const dim3 grid((unsigned)max_tiles, (unsigned)((n_out + MOE_TN - 1) / MOE_TN), (unsigned)((tile_rows + MOE_TM - 1) / MOE_TM));
    if (act)
        JL_DISPATCH(dtype, moe_gemm_kernel<T, true><<<grid, 256, 0, (hipStream_t)stream>>>((const T *)X, (const T *)Wt, mode, K, n_out, top, perm, offsets,
                                                                                           tile_expert, tile_row0, weights, out, a.act, tile_rows));
    else
        JL_DISPATCH(dtype, moe_gemm_kernel<T, false><<<grid, 256, 0, (hipStream_t)stream>>>((const T *)X, (const T *)Wt, mode, K, n_out, top, perm, offsets,
                                                                                            tile_expert, tile_row0, weights, out, a.act, tile_rows));
    return jl_check_launch("moe_gemm_kernel");
}

extern "C" int jl_moe_gemm(const void *X, const void *Wt, int dtype, int32_t mode, int32_t K, int32_t n_out, int32_t top,
                           const int32_t *perm, const int32_t *offsets, const int32_t *tile_expert, const int32_t *tile_row0,
                           int32_t max_tiles, int32_t E, int32_t tile_rows, const float *weights, void *out, void *stream) {
    if (max_tiles <= 0) return JL_OK;
    if (!X || !Wt || !perm || !offsets || !tile_expert || !tile_row0 || !out || (mode == 1 && !weights))
        return jl_fail(JL_E_INVALID, "jl_moe_gemm: null pointer");
    if (K <= 0 || n_out <= 0 || top <= 0 || (mode != 0 && mode != 1 && mode != JL_MOE_UP_PLAIN)) return jl_fail(JL_E_INVALID, "jl_moe_gemm: bad sizes or mode");
    return moe_gemm_launch(X, Wt, dtype, mode, K, n_out, top, perm, offsets, tile_expert, tile_row0, max_tiles, E, tile_rows, weights, out, nullptr, stream);
}

extern "C" int jl_moe_gemm_gated(const void *X, const void *Wt, int dtype, int32_t K, int32_t ff, int32_t top, const int32_t *perm,
                                 const int32_t *offsets, const int32_t *tile_expert, const int32_t *tile_row0, int32_t max_tiles, int32_t E,
                                 int32_t tile_rows, int32_t kind, float limit, float alpha, float shift, void *out, void *stream) {
    if (max_tiles <= 0) return JL_OK;
    if (!X || !Wt || !perm || !offsets || !tile_expert || !tile_row0 || !out) return jl_fail(JL_E_INVALID, "jl_moe_gemm_gated: null pointer");
    if (K <= 0 || ff <= 0 || top <= 0 || kind < JL_ACT_GELU_TANH || kind > JL_ACT_GELU_ERF)
        return jl_fail(JL_E_INVALID, "jl_moe_gemm_gated: bad sizes or kind");
    const MoeAct act = {kind, limit, alpha, shift};
    return moe_gemm_launch(X, Wt, dtype, JL_MOE_UP_PLAIN, K, ff, top, perm, offsets, tile_expert, tile_row0, max_tiles, E, tile_rows, nullptr, out, &act, stream);
}

// A decode's experts without a grouping: three launches, the choice with a workgroup per token and the products in tiles of 32 of an expert's rows, whose number is not known: every expert gets as many as
// all tokens could fill.  A product that is not gated goes in 32 columns at a time, three workgroups to a CU (64 columns, two: 9.0 us instead of 7.4, of 32 x 4 rows of 16 of 1024 x 512).
// us, experts with choice, weights from memory, grouped / so: 16 of 1024 x 512, 1 token x 4 20.9 / 15.4, 32 31.2 / 20.8, 64 35.1 / 21.9, 96 36.0 / 23.9; 32 of 2048 x 1024, gated, 1 33.1 / 31.6, 32
// 102 / 94, 64 105 / 94, 96 105 / 103; 64 of 1024 x 512, gated, 96 72 / 67; float, 16 of 1024 x 512, 32 45 / 39.  Beyond the line the tiles that have no rows cost more than the grouping: 128 of 32 106 / 108,
// of 64 73 / 73, 191 of 32 107 / 133.
static bool moe_few_sizes(int dtype, int64_t N, int32_t Er, int32_t top, int64_t W, int64_t ff) {
    return N > 0 && N <= JL_MOE_FEW_TOKENS && Er > 0 && Er <= MR_MAX_E && top > 0 && N * top <= JL_MOE_FEW_ROWS && moe_mm_sizes(dtype, W) && moe_mm_sizes(dtype, ff) && W > 0 && ff > 0 && W <= (1 << 20) &&
           ff <= (1 << 20);
}
extern "C" int jl_moe_few_ok(int dtype, int64_t N, int32_t Er, int32_t top, int32_t W, int32_t ff) {
    static const bool no_mfma = getenv("JL_MOE_NO_MFMA") != nullptr;      // A/B switch for measurements
    return !no_mfma && moe_few_sizes(dtype, N, Er, top, W, ff);
}
extern "C" int jl_moe_few_run(const jl_moe_few *ap, void *stream) {
    if (!ap) return jl_fail(JL_E_INVALID, "jl_moe_few_run: null arguments");
    const jl_moe_few &f = *ap;
    const jl_moe_router &a = f.router;
    if (!a.x || !a.ids || !a.weights || !f.h || !f.w_up || !f.w_down || !f.act || !f.out) return jl_fail(JL_E_INVALID, "jl_moe_few_run: null pointer");
    if ((f.dtype != JL_BF16 && f.dtype != JL_F32) || !moe_few_sizes(f.dtype, a.N, a.E, a.top, f.W, f.ff) || a.experts <= 0 || a.experts > a.E || a.top > a.E || a.kind < JL_ROUTE_SIGMOID ||
        a.kind > JL_ROUTE_TOP_SOFTMAX || (f.gated && (f.unit < JL_ACT_GELU_TANH || f.unit > JL_ACT_GELU_ERF)))
        return jl_fail(JL_E_INVALID, "jl_moe_few_run: up to %d tokens, %d choices of theirs and %d router outputs, rows at 16-byte borders", JL_MOE_FEW_TOKENS, JL_MOE_FEW_ROWS, MR_MAX_E);
    if (((uintptr_t)f.h | (uintptr_t)f.w_up | (uintptr_t)f.w_down | (uintptr_t)f.act | (uintptr_t)f.out) & 15) return jl_fail(JL_E_INVALID, "jl_moe_few_run: operands at 16-byte borders");
    if (!a.w && (a.x_dtype != JL_F32 || a.bias)) return jl_fail(JL_E_INVALID, "jl_moe_few_run: logits are float and whole");
    if (a.w && ((a.x_dtype != JL_BF16 && a.x_dtype != JL_F32) || a.K <= 0 || a.K % 4 || a.x_ld < a.K || a.x_ld % (a.x_dtype == JL_BF16 ? 8 : 4) || (((uintptr_t)a.x | (uintptr_t)a.w) & 15)))
        return jl_fail(JL_E_INVALID, "jl_moe_few_run: rows of x and W at 16-byte borders");
    hipStream_t st = (hipStream_t)stream;
#define RF_CASE(outputs) JL_DISPATCH(a.x_dtype, moe_router_few_kernel<T, outputs><<<dim3((unsigned)a.N), 64 * RF_NW, 0, st>>>(a))
    if (a.E <= RF_NW) RF_CASE(1); else if (a.E <= 2 * RF_NW) RF_CASE(2); else RF_CASE(4);
#undef RF_CASE
    const int chunks = (int)((a.N + 31) / 32), rows = (int)(a.N * a.top);
    auto product = [&](const void *x, const void *w, const float *weights, void *out, int mode, int K, int n_out, bool gated) {
        const MoeMM m = {x, w, nullptr, nullptr, nullptr, nullptr, weights, out, mode, K, n_out, a.top, a.experts, (n_out + 31) / 32, 0, 1, {f.unit, f.limit, f.alpha, f.shift}, a.ids, rows};
        const dim3 grid((unsigned)(a.experts * chunks * m.col_blocks));
        if (gated) JL_DISPATCH(f.dtype, moe_few_kernel<T, 4, true, false, true><<<grid, 256, 0, st>>>(m));
        else JL_DISPATCH(f.dtype, moe_few_kernel<T, 4, false, false, true, 32><<<grid, 256, 0, st>>>(m));
    };
    product(f.h, f.w_up, nullptr, f.act, f.gated ? JL_MOE_UP_PLAIN : 0, f.W, f.ff, f.gated);
    product(f.act, f.w_down, a.weights, f.out, 1, f.ff, f.W, false);
    return jl_check_launch("moe_few_kernel");
}
