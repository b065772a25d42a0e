// jl_moe.hip — routed experts: the router's choice (sigmoid scores with a correction, a softmax renormalised over the chosen with or without
// a correction, or a softmax over the chosen logits alone), the rows grouped by expert (a choice of an expert without weights has none), and
// the grouped products: up with relu^2, plain, or with the gated unit in its epilogue, down with the routing weights.
#include "jl_common.h"
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
        be = __shfl(be, 0, 64);                                     // one winner for all lanes, whatever the values compared to (not-a-numbers)
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
// bfloat16, us at 32 / 64 / 128 rows: 8192 tokens x 4 of 32 (2048 x 1024) 1059 / 790 / 623, 1024 tokens 213 / 171 / 160, 512 tokens 147 / 140 / 155, 256 tokens 121 / 124 / 142;
// 4096 x 4 of 16 (1024 x 512) 180 / 135 / 123, 1024 tokens 75 / 66 / 79, 512 tokens 51 / 57 / 77; 4096 x 4 of 12 (768 x 512) 151 / 117 / 104, 2048 tokens 95 / 77 / 80;
// float, 2048 x 4 of 16 (1024 x 512): 341 / 311 / 401.
// Sizes the matrix-core product does not take (rows that do not start at 16-byte borders) go in tiles of MOE_TM.
static bool moe_mm_sizes(int dtype, int64_t K) { return (dtype == JL_BF16 && K % 8 == 0) || (dtype == JL_F32 && K % 4 == 0); }
extern "C" int jl_moe_tile_rows(int dtype, int64_t rows, int32_t E, int32_t W, int32_t ff) {
    if (E <= 0 || !moe_mm_sizes(dtype, W) || !moe_mm_sizes(dtype, ff)) return MOE_TM;
    auto blocks = [&](int tm, int width, int tn) { return (rows / tm + E / 2) * ((width + tn - 1) / tn); };
    if (dtype == JL_BF16 && blocks(128, ff, 128) >= 256 && blocks(128, W, 256) >= 256 && rows >= (int64_t)96 * E) return 128;
    return rows >= (int64_t)48 * E && blocks(64, ff, 128) + blocks(64, W, 256) >= 512 ? 64 : 32;
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
// rows when TM is 128) hold 32 x 32 accumulators; the weights are the A operand, the rows the B operand, so that a lane ends with four neighbouring
// output columns of ONE row and stores them together.  A lane's operand is one 16-byte unit: in bfloat16 the eight depths 8 (lane / 32) .. of
// v_mfma_f32_32x32x16_bf16; in float four v_mfma_f32_32x32x2_f32, one for each of its floats (the depths meet in the order 0, 4, 1, 5, ..: a sum of
// products rounded one by one, as a chain of multiply-adds is).  Units of a row are permuted so that 16 neighbouring rows meet different banks.
// GATED: the WR weight rows are WR / 2 of the gate and the WR / 2 of the linear branch that belong to them (rows n_out further on); both products
// of a column end in the same lane, which stores the gated unit.
// TM = 128 (an expert has about a hundred rows or more) is bound by the matrix cores and LDS: 128 x 256 reads 48 KB of LDS per 64 products.  Rows go from memory straight into LDS
// (16 bytes per lane, every lane fetching the unit that the permutation puts into its place), one stage ahead: no registers and no LDS writes for them, so that three workgroups fit a
// CU and cover each other's barriers (through registers, two of them: gated product at 8192 x 4 of 32 experts of 2048 x 1024 406 -> 363 us, the way down 290 -> 252).
// Workgroups of an XCD (every eighth) take neighbouring tiles and all their columns, so that an expert's weights are read into one L2.  TM = 32 (decoding) is bound by reading
// the weights: single wavefronts, many per CU, 12 KB on the way each, in registers.
// Loads carry no branch and no 64-bit address arithmetic of their own: offsets of 32 bits from a base (of the tile where its rows lie together; FAR: rows gathered from more than
// 4 GiB have 64-bit addresses), rows that do not exist repeat another, stages behind the last repeat the
// first, depths beyond the last whole stage come after the loop (a condition per load had cost six vector instructions per product: 431 us instead of 406 for the gated product
// above; us for up and down at 32 rows x 4 of 16 of 1024 x 512: 49 -> 41, float 16 rows 100 -> 79, 400 rows 53 -> 45).
struct MoeMM {
    const void *X, *Wt;
    const int32_t *perm, *offsets, *tile_expert, *tile_row0;
    const float *weights;
    void *out;
    int mode, K, n_out, top, E, col_blocks, max_tiles;
    MoeAct act;
};
typedef __bf16 mm_bf16x8 __attribute__((ext_vector_type(8)));
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

template <typename T, int TM, int NW, int WR, int TKU, bool GATED, bool FAR>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 3 : 1) void moe_mm_kernel(MoeMM a) {
    constexpr int THREADS = 64 * NW, UNIT = mm_type<T>::UNIT, WM = TM == 128 ? 2 : 1, WN = NW / WM, XT = TM / WM / 32, NT = WR / WN / 32;
    constexpr int XPF = TM * TKU / THREADS, WPF = WR * TKU / THREADS, TN = GATED ? WR / 2 : WR, STAGE = TKU * UNIT;
    static_assert(XPF * THREADS == TM * TKU && WPF * THREADS == WR * TKU && (!GATED || NT % 2 == 0), "tile");
    __shared__ uint4 smem[2 * (TM + WR) * TKU];
    int tile, col;
    if (TM >= 64) {                                                 // workgroups with the same remainder by 8 share an XCD
        const int per_xcd = (a.offsets[a.E + 1] + 7) / 8, xcd = blockIdx.x & 7, s = blockIdx.x >> 3;
        if (s >= per_xcd * a.col_blocks) return;
        tile = xcd * per_xcd + s / a.col_blocks;
        col = s % a.col_blocks;
        if (tile >= a.max_tiles) return;
    } else {
        tile = blockIdx.x / a.col_blocks;
        col = blockIdx.x - tile * a.col_blocks;
    }
    const int e = a.tile_expert[tile];
    if (e < 0) return;
    const int r0 = a.tile_row0[tile], K = a.K, n_out = a.n_out, n0 = col * TN;
    const int nr = a.offsets[e + 1] - r0 < TM ? a.offsets[e + 1] - r0 : TM;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, hi = lane >> 5, wm = wave / WN, wn = wave % WN;
    auto at = [](int row, int u) { return row * TKU + (u ^ (TKU == 4 ? (row >> 2) & 3 : (row >> 1) & 7)); };
    // loaders: unit tid % TKU of rows tid / TKU + x * THREADS / TKU; a row that does not exist repeats another and is not stored
    const int lr = tid / TKU;
    constexpr bool DMA = NW > 1;
    auto unit_of = [&](int x) { return DMA ? at(lr + x * (THREADS / TKU), tid % TKU) % TKU : tid % TKU; };      // DMA: what belongs into this thread's place of LDS
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
    mm_u32x4 reg[DMA ? 1 : 2][XPF + WPF];                                     // stages on their way: even ones in reg[0], odd ones in reg[1]
    const int full = K / STAGE;                                     // whole stages; what is left of K comes last
    auto fetch = [&](mm_u32x4 (&r)[XPF + WPF], int i) {             // without branches: behind the last stage, stage 0 again (never used)
        const int64_t k = i < full ? (int64_t)i * STAGE * sizeof(T) : 0;
        const char *xb = Xb + k;
#pragma unroll
        for (int x = 0; x < XPF; ++x) {
            if constexpr (FAR) r[x] = *(const mm_u32x4 *)(xfar[x] + k);
            else r[x] = *(const mm_u32x4 *)(xb + xo[x]);
        }
#pragma unroll
        for (int x = 0; x < WPF; ++x) r[XPF + x] = *(const mm_u32x4 *)(w_base(x) + k + wo[x]);
    };
    auto stash = [&](const mm_u32x4 (&r)[XPF + WPF], int sel) {
        uint4 *Xs = smem + sel * (TM + WR) * TKU, *Ws = Xs + TM * TKU;
#pragma unroll
        for (int x = 0; x < XPF; ++x) Xs[at(lr + x * (THREADS / TKU), unit_of(x))] = __builtin_bit_cast(uint4, r[x]);
#pragma unroll
        for (int x = 0; x < WPF; ++x) Ws[at(lr + x * (THREADS / TKU), unit_of(x))] = __builtin_bit_cast(uint4, r[XPF + x]);
    };
    mm_f32x16 acc[XT][NT];
#pragma unroll
    for (int x = 0; x < XT; ++x)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[x][t][i] = 0.f;
    // weight row (within the tile) of this wavefront's tile t: gate tiles first, then the linear branch's
    auto w_row = [&](int t) { return GATED ? (t < NT / 2 ? 0 : TN) + wn * (TN / WN) + 32 * (t % (NT / 2 > 0 ? NT / 2 : 1)) : wn * (WR / WN) + 32 * t; };
    auto products = [&](auto sel_c) {
        constexpr int sel = decltype(sel_c)::value;
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
                for (int x = 0; x < XT; ++x) acc[x][t] = mm_type<T>::mma(wf[t], xf[x], acc[x][t]);

        }
    };
    std::integral_constant<int, 0> even;
    std::integral_constant<int, 1> odd;
    if (DMA && full > 0) {
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
        auto arrived = [&]() {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        };
        issue(0, 0);
        int i = 0;
        for (; i + 1 < full; i += 2) {
            arrived();
            issue(i + 1, 1);
            products(even);
            arrived();
            issue(i + 2, 0);
            products(odd);
        }
        arrived();
        if (i < full) {
            products(even);
            __syncthreads();
        }
    } else if (full > 0) {
        fetch(reg[0], 0);
        constexpr int R1 = DMA ? 0 : 1;
        fetch(reg[R1], 1);
        stash(reg[0], 0);
        __syncthreads();
        int i = 0;
        for (; i + 1 < full; i += 2) {                              // two stages ahead: a trip to memory takes longer than one stage's products
            fetch(reg[0], i + 2);
            products(even);
            stash(reg[R1], 1);
            __syncthreads();
            fetch(reg[R1], i + 3);
            products(odd);
            stash(reg[0], 0);
            __syncthreads();
        }
        if (i < full) {
            products(even);
            __syncthreads();
        }
    }
    if (full * STAGE < K) {                                         // depths beyond K are zero
        const mm_u32x4 zero = {0, 0, 0, 0};
        auto last = [&](const char *from, int u) {                  // a lane beyond K reads its row's first unit: a row may be shorter than a stage
            const bool in = full * STAGE + u * UNIT < K;
            const mm_u32x4 v = *(const mm_u32x4 *)(from + (in ? (int64_t)full * STAGE * sizeof(T) : -(int64_t)(u * UNIT * sizeof(T))));
            return in ? v : zero;
        };
#pragma unroll
        for (int x = 0; x < XPF; ++x) reg[0][x] = last(FAR ? xfar[FAR ? x : 0] : Xb + xo[x], unit_of(x));
#pragma unroll
        for (int x = 0; x < WPF; ++x) reg[0][XPF + x] = last(w_base(x) + wo[x], unit_of(x));
        stash(reg[0], 0);
        __syncthreads();
        products(even);
    }
    constexpr int OT = GATED ? NT / 2 : NT;
    const bool whole = n_out % 4 == 0;
#pragma unroll
    for (int x = 0; x < XT; ++x) {
        const int m = wm * (TM / WM) + 32 * x + l32;
        if (m >= nr) continue;
        const int64_t r = r0 + m;
        const int64_t p = a.mode == 1 ? a.perm[r] : r;
        const float w = a.mode == 1 ? a.weights[p] : 1.0f;
#pragma unroll
        for (int t = 0; t < OT; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + w_row(t) + 8 * g + 4 * hi;       // four neighbouring columns
                if (n >= n_out) continue;
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float c = acc[x][t][4 * g + i];
                    if (GATED) v[i] = gated_unit_f<sizeof(T) == 2>(c, acc[x][t + (GATED ? OT : 0)][4 * g + i], a.act.kind, a.act.limit, a.act.alpha, a.act.shift);
                    else if (a.mode == JL_MOE_UP_PLAIN) v[i] = c;
                    else if (a.mode == 0) { const float q = fmaxf(c, 0.f); v[i] = q * q; }
                    else v[i] = c * w;
                }
                const int64_t o = p * n_out + n;
                if (!GATED && a.mode == 1) {
                    if (whole) st4_f((float *)a.out + o, v);
                    else for (int i = 0; i < 4 && n + i < n_out; ++i) ((float *)a.out)[o + i] = v[i];
                } else {
                    if (whole) st4_f((T *)a.out + o, v);
                    else for (int i = 0; i < 4 && n + i < n_out; ++i) st_f((T *)a.out + o + i, v[i]);
                }
            }
    }
}

template <typename T, int TM, int NW, int WR, int TKU> static int moe_mm_launch(MoeMM &a, bool gated, hipStream_t st) {
    const int tn = gated ? WR / 2 : WR;
    a.col_blocks = (a.n_out + tn - 1) / tn;
    const int64_t groups = (int64_t)(TM >= 64 ? (a.max_tiles + 7) / 8 * 8 : a.max_tiles) * a.col_blocks;
    if (groups > 0x7fffffff) return jl_fail(JL_E_INVALID, "jl_moe_gemm: too many tiles");
    const bool far = a.mode != 1 && ((int64_t)a.max_tiles * TM / a.top + 1) * a.K * (int64_t)sizeof(T) > UINT32_MAX;      // gathered rows beyond what 32 bits reach
    auto kern = gated ? (far ? moe_mm_kernel<T, TM, NW, WR, TKU, true, true> : moe_mm_kernel<T, TM, NW, WR, TKU, true, false>)
                      : (far ? moe_mm_kernel<T, TM, NW, WR, TKU, false, true> : moe_mm_kernel<T, TM, NW, WR, TKU, false, false>);
    kern<<<dim3((unsigned)groups), 64 * NW, 0, st>>>(a);
    return jl_check_launch("moe_mm_kernel");
}
template <typename T> static int moe_mm_rows(MoeMM &a, int tile_rows, bool gated, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        if (tile_rows == 128) return moe_mm_launch<T, 128, 4, 256, 4>(a, gated, st);
    } else if (tile_rows == 128) return jl_fail(JL_E_INVALID, "jl_moe_gemm: float tiles have 32 or 64 rows");
    if (tile_rows == 64) return moe_mm_launch<T, 64, 4, 256, 4>(a, gated, st);
    return moe_mm_launch<T, 32, 1, 64, 8>(a, gated, st);
}

static int moe_gemm_launch(const void *X, const void *Wt, int dtype, int32_t mode, int32_t K, int32_t n_out, int32_t top, const int32_t *perm,
                           const int32_t *offsets, const int32_t *tile_expert, const int32_t *tile_row0, int32_t max_tiles, int32_t E, int32_t tile_rows,
                           const float *weights, void *out, const MoeAct *act, void *stream) {
    static const bool no_mfma = getenv("JL_MOE_NO_MFMA") != nullptr;      // A/B switch for measurements
    if (E <= 0 || (tile_rows != 32 && tile_rows != 64 && tile_rows != 128)) return jl_fail(JL_E_INVALID, "jl_moe_gemm: tiles of 32, 64 or 128 rows");
    const int64_t dtype_bytes = dtype == JL_BF16 ? 2 : 4;
    MoeMM a = {X, Wt, perm, offsets, tile_expert, tile_row0, weights, out, mode, K, n_out, top, E, 0, max_tiles, act ? *act : MoeAct{0, 0.f, 0.f, 0.f}};
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
