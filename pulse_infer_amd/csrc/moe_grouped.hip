// The experts of a routed feed-forward on the matrix cores (bfloat16): the (token, choice) pairs of a step are
// grouped by expert on the device, and every expert multiplies its own rows.
//
// pulse_moe_group (one workgroup): counts the pairs of every expert, gives each pair its place among its expert's
// (`order`: places -> pairs, the experts one after the other) and cuts every expert's pairs into tiles of TM rows:
// tile_expert, tile_row0 (first place), tile_rows, and their number.  Pairs that chose an identity expert
// (index >= experts) are in no tile.  Which place a pair gets among its expert's depends on the order in which the
// threads arrive; no result depends on it, since every row of a product is computed by itself.
//
// pulse_moe_gate_up_grouped and pulse_moe_down_grouped run on the loop of tile_loop.h (moe_tile_kernel) where the inner
// dimension is a multiple of 64.  Else:
// pulse_moe_gate_up_grouped: a workgroup of four wavefronts per (tile, 64 inner columns); a wavefront owns 16 gate
// rows and the 16 up rows beside them and walks the hidden size in steps of 32 with v_mfma_f32_16x16x32_bf16, the
// weight rows as the row operand, up to RB blocks of 16 gathered token rows as the column operand;
// act[pair, j] = silu(g) * u.
// pulse_moe_down_grouped: the same walk over the inner width with the down weights; y[pair, :] in float32.
// pulse_moe_combine: out[t] = sum over the token's choices, in their order, of weight * y[pair] (or weight * x[t]
// for an identity expert), float32.
// The launches are sized by the step's shape alone (the most tiles it can have); workgroups behind the number of
// tiles leave at once.
#include "common.h"
#include "tile_loop.h"

#include <math.h>

#include <algorithm>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ bf16x8 zeros8() {
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (__bf16)0.0f;
    return z;
}

constexpr int GROUP_THREADS = 1024;
constexpr int MAX_EXPERTS = 1024;

__global__ __launch_bounds__(GROUP_THREADS) void moe_group_kernel(const int* __restrict__ idx, int pairs, int experts,
                                                                  int tile_rows_max, int max_tiles,
                                                                  int* __restrict__ rank, int* __restrict__ order,
                                                                  int* __restrict__ tile_expert,
                                                                  int* __restrict__ tile_row0,
                                                                  int* __restrict__ tile_rows,
                                                                  int* __restrict__ num_tiles) {
    __shared__ int count[MAX_EXPERTS];
    __shared__ int first[MAX_EXPERTS];       // an expert's first place
    __shared__ int first_tile[MAX_EXPERTS + 1];
    const int tid = threadIdx.x;
    for (int e = tid; e < experts; e += GROUP_THREADS) count[e] = 0;
    __syncthreads();
    // (the choices of eight rounds are asked for together: a round by itself waits out a trip to memory)
    constexpr int AHEAD = 8;
    for (int a0 = tid; a0 < pairs; a0 += AHEAD * GROUP_THREADS) {
        int es[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) es[u] = a0 + u * GROUP_THREADS < pairs ? idx[a0 + u * GROUP_THREADS] : -1;
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (es[u] >= 0 && es[u] < experts) rank[a0 + u * GROUP_THREADS] = atomicAdd(&count[es[u]], 1);
    }
    __syncthreads();
    if (tid < PULSE_WAVE) {       // places and tiles before an expert: sums over the experts, 64 at a time
        int at = 0, tiles = 0;
        for (int e0 = 0; e0 < experts; e0 += PULSE_WAVE) {
            const int e = e0 + tid;
            const int c = e < experts ? count[e] : 0, n = (c + tile_rows_max - 1) / tile_rows_max;
            int pre_c = c, pre_n = n;
#pragma unroll
            for (int off = 1; off < PULSE_WAVE; off <<= 1) {
                const int uc = __shfl_up(pre_c, off, PULSE_WAVE), un = __shfl_up(pre_n, off, PULSE_WAVE);
                if (tid >= off) { pre_c += uc; pre_n += un; }
            }
            if (e < experts) {
                first[e] = at + pre_c - c;
                first_tile[e] = tiles + pre_n - n;
            }
            at += __shfl(pre_c, PULSE_WAVE - 1, PULSE_WAVE);
            tiles += __shfl(pre_n, PULSE_WAVE - 1, PULSE_WAVE);
        }
        if (tid == 0) *num_tiles = min(tiles, max_tiles);
    }
    __syncthreads();
    for (int e = tid / 16; e < experts; e += GROUP_THREADS / 16) {      // sixteen threads an expert write its tiles
        const int c = count[e];
        for (int m = tid % 16; m * tile_rows_max < c; m += 16) {
            const int t = first_tile[e] + m;
            if (t >= max_tiles) break;
            tile_expert[t] = e;
            tile_row0[t] = first[e] + m * tile_rows_max;
            tile_rows[t] = min(tile_rows_max, c - m * tile_rows_max);
        }
    }
    for (int a0 = tid; a0 < pairs; a0 += AHEAD * GROUP_THREADS) {
        int es[AHEAD], at[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int a = a0 + u * GROUP_THREADS;
            es[u] = a < pairs ? idx[a] : -1;
            at[u] = es[u] >= 0 && es[u] < experts ? rank[a] : -1;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (at[u] >= 0) order[first[es[u]] + at[u]] = a0 + u * GROUP_THREADS;
    }
}

// Tiles of 32 rows (decoding: few rows an expert) give few workgroups, each with a long walk: there the four
// wavefronts of a workgroup own the SAME 16 weight rows and a quarter of the k-steps each, and their sums meet in LDS in
// wavefront order (four times the workgroups, four times the loads in flight, the same result from run to run).
template <int NW, int RB>
__device__ __forceinline__ bool meet(f32x4 (&acc)[NW][RB], float* red, int wave, int lane) {
    // red: [4][NW * RB][64][4] floats
#pragma unroll
    for (int s = 0; s < NW; ++s)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[((wave * NW * RB + s * RB + rb) * 64 + lane) * 4 + i] = acc[s][rb][i];
    __syncthreads();
    if (wave != 0) return false;
#pragma unroll
    for (int w = 1; w < 4; ++w)
#pragma unroll
        for (int s = 0; s < NW; ++s)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[s][rb][i] += red[((w * NW * RB + s * RB + rb) * 64 + lane) * 4 + i];
    return true;
}

// One tile of one expert against 64 weight rows: acc[rb] += W[16 rows of this wavefront] . X[16 rows of block rb]^T.
// wrow: this lane's weight row (null: beyond the weight), xrow[rb]: this lane's row of block rb (null: no such row).
template <int RB, int NW>
__device__ __forceinline__ void walk(const bf16_t* const (&wrow)[NW], const bf16_t* const (&xrow)[RB], int blocks, int K,
                                     int kg, f32x4 (&acc)[NW][RB], int share = 0, int shares = 1) {
    constexpr int U = 4;   // k-steps whose loads are asked for before the first of them is used
    // (`share` of `shares`: this wavefront takes every shares-th group of U k-steps, from group `share` on)
    for (int k0 = share * 32 * U; k0 < K; k0 += shares * 32 * U) {
        bf16x8 wa[U][NW], xb[U][RB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kc = k0 + 32 * u + kg * 8;
            const bool kok = kc < K;   // K is a multiple of 8
#pragma unroll
            for (int s = 0; s < NW; ++s)
                wa[u][s] = (kok && wrow[s]) ? *reinterpret_cast<const bf16x8*>(wrow[s] + kc) : zeros8();
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                xb[u][rb] = (kok && rb < blocks && xrow[rb]) ? *reinterpret_cast<const bf16x8*>(xrow[rb] + kc) : zeros8();
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if (rb < blocks) {
#pragma unroll
                    for (int s = 0; s < NW; ++s)
                        acc[s][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[u][s], xb[u][rb], acc[s][rb], 0, 0, 0);
                }
            }
        }
    }
}

// The same walk for tiles of 128 rows (RB = 8): the tile's rows go through LDS in pieces of 64 values of k, fetched
// once by the workgroup's 256 threads (a thread half a row's piece: 64 bytes) instead of once by every wavefront, the
// next piece travelling while this one is multiplied.  src[t]: the row that thread t fetches half of (null: none).
constexpr int STAGE_K = 64;
constexpr int STAGE_ROW = STAGE_K + 8;   // values a row takes in LDS (the 8 more keep rows off each other's banks)

template <int NW>
__device__ __forceinline__ void walk_staged(const bf16_t* const (&wrow)[NW], const bf16_t* src, bf16_t* stage, int blocks,
                                            int K, int r, int kg, f32x4 (&acc)[NW][8]) {
    const int tid = threadIdx.x;
    const int frow = tid / 2, fk = (tid % 2) * 32;   // this thread fetches values fk .. fk + 31 of row frow's piece
    bf16x8 held[4];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kc = k0 + fk + 8 * u;
            held[u] = (src && kc < K) ? *reinterpret_cast<const bf16x8*>(src + kc) : zeros8();
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += STAGE_K) {
        __syncthreads();   // the piece in LDS has been multiplied
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<bf16x8*>(stage + frow * STAGE_ROW + fk + 8 * u) = held[u];
        __syncthreads();
        if (k0 + STAGE_K < K) fetch(k0 + STAGE_K);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int kc = k0 + 32 * half + kg * 8;
            const bool kok = kc < K;
            bf16x8 wa[NW];
#pragma unroll
            for (int s = 0; s < NW; ++s)
                wa[s] = (kok && wrow[s]) ? *reinterpret_cast<const bf16x8*>(wrow[s] + kc) : zeros8();
#pragma unroll
            for (int rb = 0; rb < 8; ++rb) {
                if (rb < blocks) {
                    const bf16x8 xb = *reinterpret_cast<const bf16x8*>(stage + (rb * 16 + r) * STAGE_ROW + 32 * half + kg * 8);
#pragma unroll
                    for (int s = 0; s < NW; ++s)
                        acc[s][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[s], xb, acc[s][rb], 0, 0, 0);
                }
            }
        }
    }
}

template <int RB>
__global__ __launch_bounds__(256) void moe_gate_up_grouped_kernel(const bf16_t* __restrict__ x,
                                                                  const bf16_t* __restrict__ wg,
                                                                  const bf16_t* __restrict__ wu,
                                                                  const int* __restrict__ order,
                                                                  const int* __restrict__ tile_expert,
                                                                  const int* __restrict__ tile_row0,
                                                                  const int* __restrict__ tile_rows,
                                                                  const int* __restrict__ num_tiles,
                                                                  bf16_t* __restrict__ act, int hidden, int ff, int top,
                                                                  const float* __restrict__ in_weight, int act_kind,
                                                                  float limit) {
    const int tile = blockIdx.x;
    if (tile >= *num_tiles) return;
    const int e = tile_expert[tile], row0 = tile_row0[tile] + blockIdx.z * (RB * 16);   // (z: 16 RB rows of a longer tile)
    const int rows = min(tile_rows[tile] - static_cast<int>(blockIdx.z) * (RB * 16), RB * 16);
    if (rows <= 0) return;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    const int r = lane % 16, kg = lane / 16;
    constexpr bool SHARED_K = RB == 2;
    const int n0 = SHARED_K ? blockIdx.y * 16 : blockIdx.y * 64 + wave * 16;
    const int n = n0 + r;
    const bf16_t* wrow[2];
    wrow[0] = n < ff ? wg + (static_cast<int64_t>(e) * ff + n) * hidden : nullptr;
    wrow[1] = n < ff ? wu + (static_cast<int64_t>(e) * ff + n) * hidden : nullptr;
    const bf16_t* xrow[RB];
    int pair[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int i = rb * 16 + r;
        pair[rb] = i < rows ? order[row0 + i] : -1;
        xrow[rb] = pair[rb] >= 0 ? x + static_cast<int64_t>(pair[rb] / top) * hidden : nullptr;
    }
    f32x4 acc[2][RB];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[s][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (RB == 8) {
        __shared__ __attribute__((aligned(16))) bf16_t stage[128 * STAGE_ROW];
        const int mine = threadIdx.x / 2;
        const int p = mine < rows ? order[row0 + mine] : -1;
        walk_staged<2>(wrow, p >= 0 ? x + static_cast<int64_t>(p / top) * hidden : nullptr, stage, (rows + 15) / 16, hidden,
                       r, kg, acc);
    } else {
        __shared__ float red[4 * 2 * RB * 64 * 4];
        walk<RB, 2>(wrow, xrow, (rows + 15) / 16, hidden, kg, acc, wave, 4);
        if (!meet<2, RB>(acc, red, wave, lane)) return;
    }
    // lane l holds inner columns 4 * (l / 16) + i of this wavefront's 16, for row l % 16 of every block
    const int j0 = n0 + 4 * kg;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        if (pair[rb] < 0) continue;
        bf16_t* dst = act + static_cast<int64_t>(pair[rb]) * ff;
        // an expert that is fed weight * x: both products are linear, so the factor goes onto their results
        const float wgt = in_weight ? in_weight[pair[rb]] : 1.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (j0 + i < ff) {
                float g = acc[0][rb][i] * wgt, u = acc[1][rb][i] * wgt;
                if (act_kind == 1) {   // clamped: min(g, limit) * sigmoid(1.702 g) * (clamp(u) + 1)
                    g = fminf(g, limit);
                    u = fminf(fmaxf(u, -limit), limit);
                    dst[j0 + i] = f32_to_bf16(g / (1.0f + expf(-1.702f * g)) * (u + 1.0f));
                } else {
                    dst[j0 + i] = f32_to_bf16(g / (1.0f + expf(-g)) * u);
                }
            }
        }
    }
}

template <int RB>
__global__ __launch_bounds__(256) void moe_down_grouped_kernel(const bf16_t* __restrict__ act,
                                                               const bf16_t* __restrict__ wd,
                                                               const int* __restrict__ order,
                                                               const int* __restrict__ tile_expert,
                                                               const int* __restrict__ tile_row0,
                                                               const int* __restrict__ tile_rows,
                                                               const int* __restrict__ num_tiles, float* __restrict__ y,
                                                               int hidden, int ff) {
    const int tile = blockIdx.x;
    if (tile >= *num_tiles) return;
    const int e = tile_expert[tile], row0 = tile_row0[tile] + blockIdx.z * (RB * 16);   // (z: 16 RB rows of a longer tile)
    const int rows = min(tile_rows[tile] - static_cast<int>(blockIdx.z) * (RB * 16), RB * 16);
    if (rows <= 0) return;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    const int r = lane % 16, kg = lane / 16;
    constexpr bool SHARED_K = RB == 2;
    const int n0 = SHARED_K ? blockIdx.y * 16 : blockIdx.y * 64 + wave * 16;
    const int n = n0 + r;
    const bf16_t* wrow[1];
    wrow[0] = n < hidden ? wd + (static_cast<int64_t>(e) * hidden + n) * ff : nullptr;
    const bf16_t* xrow[RB];
    int pair[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int i = rb * 16 + r;
        pair[rb] = i < rows ? order[row0 + i] : -1;
        xrow[rb] = pair[rb] >= 0 ? act + static_cast<int64_t>(pair[rb]) * ff : nullptr;
    }
    f32x4 acc[1][RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[0][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (RB == 8) {
        __shared__ __attribute__((aligned(16))) bf16_t stage[128 * STAGE_ROW];
        const int mine = threadIdx.x / 2;
        const int p = mine < rows ? order[row0 + mine] : -1;
        walk_staged<1>(wrow, p >= 0 ? act + static_cast<int64_t>(p) * ff : nullptr, stage, (rows + 15) / 16, ff, r, kg, acc);
    } else {
        __shared__ float red[4 * 1 * RB * 64 * 4];
        walk<RB, 1>(wrow, xrow, (rows + 15) / 16, ff, kg, acc, wave, 4);
        if (!meet<1, RB>(acc, red, wave, lane)) return;
    }
    const int c0 = n0 + 4 * kg;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        if (pair[rb] < 0) continue;
        float* dst = y + static_cast<int64_t>(pair[rb]) * hidden;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (c0 + i < hidden) dst[c0 + i] = acc[0][rb][i];
    }
}

template <typename TX>
__global__ void moe_combine_kernel(const TX* __restrict__ x, const float* __restrict__ y, const int* __restrict__ idx,
                                   const float* __restrict__ weight, float* __restrict__ out, int64_t total, int hidden,
                                   int experts, int top) {
    const int64_t at = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (at >= total) return;
    const int64_t t = at / hidden;
    const int c = static_cast<int>(at % hidden);
    float acc = 0.f;
    for (int k = 0; k < top; ++k) {
        const int e = idx[t * top + k];
        const float w = weight ? weight[t * top + k] : 1.f;
        if (e >= experts) acc = fmaf(w, to_f32<TX>(x[at]), acc);
        else if (e >= 0) acc = fmaf(w, y[(t * top + k) * hidden + c], acc);
    }
    out[at] = acc;
}

// ------------------------------------------------------------------ many rows an expert
// Tiles of 32, 64, 128 or 192 gathered rows against WR weight rows (for gate and up: slabs of 16 gate rows and the 16 up rows
// beside them, so that a lane holds both of an inner column), on the loop of tile_loop.h.
//
// What bounds it: what a compute unit copies into LDS for tiles of 192 rows, the weights' way from memory for an expert of few rows.  Neighbouring
// workgroups of a die take the tiles of a panel, which share weight rows and gathered rows in that die's L2.
struct GroupArgs {
    const bf16_t* x;             // gate and up: [tokens, K], row pair / top; down: act [pairs, K], row pair
    const bf16_t* w[2];          // stacked [experts, N, K]; down: the first
    void* out;                   // act [pairs, N] bfloat16, or y [pairs, N] float32
    const int* order;
    const int* tile_expert;
    const int* tile_row0;
    const int* tile_rows;
    const int* num_tiles;
    const float* in_weight;
    int K, N, top, tiles_n;
    int act_kind;
    float limit;
};

constexpr int GROUP_PANEL = 4;   // tiles of rows a panel of the tile order

template <bool DOWN, int WR, int XR, int WN, int WM, int S, int SX, bool NT>
__global__ __launch_bounds__(WN* WM* PULSE_WAVE) void moe_tile_kernel(GroupArgs a) {
    using Loop = TileLoop<WR, XR, WN, WM, S, NT, SX>;
    constexpr int COLS = DOWN ? WR : WR / 2;       // output columns of a tile
    __shared__ __attribute__((aligned(1024))) char lds[Loop::LDS];
    __shared__ int pair_s[XR];
    __shared__ float weight_s[XR];

    const int tiles_m = *a.num_tiles, total = tiles_m * a.tiles_n;
    const int per_die = (total + 7) / 8;
    const int t = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || t >= total) return;
    const int panel = t / (GROUP_PANEL * a.tiles_n);
    const int panel_m = min(GROUP_PANEL, tiles_m - panel * GROUP_PANEL);
    const int in_panel = t - panel * GROUP_PANEL * a.tiles_n;
    const int tile = panel * GROUP_PANEL + in_panel % panel_m;
    const int n0 = in_panel / panel_m * COLS;
    const int e = a.tile_expert[tile], row0 = a.tile_row0[tile], rows = a.tile_rows[tile];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / PULSE_WAVE);
    const int lane = tid % PULSE_WAVE;
    for (int i = tid; i < XR; i += Loop::NW * PULSE_WAVE) {
        const int p = i < rows ? a.order[row0 + i] : -1;
        pair_s[i] = p;
        weight_s[i] = p >= 0 && a.in_weight ? a.in_weight[p] : 1.f;
    }
    __syncthreads();

    // (rows past the end are the tile's first row, weight rows past the end the last one: their results are not written)
    // A chunk is eight rows of one weight: gate and up alternate in slabs of 16.
    const int64_t first_row = static_cast<int64_t>(e) * a.N + n0;
    typename Loop::Offset from[Loop::PER];
#pragma unroll
    for (int j = 0; j < Loop::PER; ++j) {
        const int row = Loop::row_of(j, wave, lane);
        int64_t at;
        if (j < Loop::PER_W) at = min(DOWN ? row : row / 32 * 16 + row % 16, a.N - 1 - n0);
        else at = (pair_s[row] < 0 ? pair_s[0] : pair_s[row]) / (DOWN ? 1 : a.top);
        from[j] = Loop::offset_of(j, at * a.K + Loop::piece_of(row, lane) * 8);
    }
    Loop loop;
    constexpr int BLOCK = DOWN ? TILE_BLOCK : TILE_BLOCK / 2;
    loop.run([&](int j) __attribute__((always_inline)) {
                 if (j >= Loop::PER_W) return a.x;
                 return (!DOWN && (wave * Loop::PER_W + j) & 2 ? a.w[1] : a.w[0]) + first_row * a.K;
             }, from, lds, wave, lane, a.K, tile_first_step(e * ((a.N + BLOCK - 1) / BLOCK) + n0 / BLOCK, a.K / Loop::BK));

    // Results leave through LDS, a wavefront's 32 rows at a time, in whole 16-byte pieces of rows.
    constexpr int TN = Loop::TN, TM = Loop::TM;
    constexpr int SIZE = DOWN ? 4 : 2, W_COLS = TN * (DOWN ? 16 : 8), PITCH = W_COLS * SIZE + 16, PCS = W_COLS * SIZE / 16;
    constexpr int WAVE_LDS = Loop::LDS / Loop::NW;
    static_assert(32 * PITCH <= WAVE_LDS && TN % 2 == 0, "a wavefront's piece of LDS holds 32 rows of its part of the tile");
    char* mine = lds + wave * WAVE_LDS;
    const int wave_n = wave % WN, wave_m = wave / WN, h = lane / 16;
    const int n_wave = n0 + wave_n * W_COLS;
#pragma unroll
    for (int g0 = 0; g0 < TM; g0 += 2) {
        const int m_base = (wave_m * TM + g0) * 16;
        if (m_base >= rows) break;
#pragma unroll
        for (int g = g0; g < g0 + 2; ++g) {
            char* at = mine + ((g - g0) * 16 + lane % 16) * PITCH + h * 4 * SIZE;
            if constexpr (DOWN) {
#pragma unroll
                for (int f = 0; f < TN; ++f)
                    *reinterpret_cast<float4*>(at + f * 64) = float4{loop.acc[f][g][0], loop.acc[f][g][1], loop.acc[f][g][2], loop.acc[f][g][3]};
            } else {
                const float wgt = weight_s[(wave_m * TM + g) * 16 + lane % 16];
#pragma unroll
                for (int f = 0; f < TN; f += 2) {
                    tile_bf16x4 v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        // an expert that is fed weight * x: both products are linear, so the factor goes onto their results
                        float gate = loop.acc[f][g][i] * wgt, up = loop.acc[f + 1][g][i] * wgt;
                        // (expf and a division, whose results are within 8 * 2^-24 of the function: the hardware's exponential and
                        // reciprocal took 12 us less, 16 experts of 1,536 x 4,096, 8,192 pairs 197 for 209 us, but were up to 30 * 2^-24 off)
                        if (a.act_kind == 1) {   // clamped: min(g, limit) * sigmoid(1.702 g) * (clamp(u) + 1)
                            gate = fminf(gate, a.limit);
                            up = fminf(fmaxf(up, -a.limit), a.limit);
                            v[i] = (__bf16)(gate / (1.0f + expf(-1.702f * gate)) * (up + 1.0f));
                        } else {
                            v[i] = (__bf16)(gate / (1.0f + expf(-gate)) * up);
                        }
                    }
                    *reinterpret_cast<tile_bf16x4*>(at + f * 16) = v;
                }
            }
        }
        tile_wave_sync();
#pragma unroll
        for (int it = 0; it < PCS / 2; ++it) {
            const int row = (it * PULSE_WAVE + lane) / PCS, pc = (it * PULSE_WAVE + lane) % PCS;
            const uint4 v = *reinterpret_cast<const uint4*>(mine + row * PITCH + pc * 16);
            const int p = pair_s[m_base + row], n = n_wave + pc * (16 / SIZE);
            if (p >= 0 && n < a.N)
                *reinterpret_cast<uint4*>(static_cast<char*>(a.out) + (static_cast<int64_t>(p) * a.N + n) * SIZE) = v;
        }
        tile_wave_sync();
    }
}

template <bool DOWN, int WR, int XR, int WN, int WM, int S, bool NT, int SX = S>
void launch_tiles(GroupArgs a, int max_tiles, hipStream_t stream) {
    constexpr int COLS = DOWN ? WR : WR / 2;
    a.tiles_n = (a.N + COLS - 1) / COLS;
    const int64_t grid = (static_cast<int64_t>(max_tiles) * a.tiles_n + 7) / 8 * 8;
    hipLaunchKernelGGL((moe_tile_kernel<DOWN, WR, XR, WN, WM, S, SX, NT>), dim3(static_cast<unsigned>(grid)), dim3(WN * WM * PULSE_WAVE), 0,
                       stream, a);
}

// Which shape a list's tiles take.  Lists of up to 128 rows are for experts of one tile mostly: bound by the weights' way from
// memory, which go past the caches; where two tiles of an expert follow each other (192 rows) they find each other's weights
// there, and the wider the tile the less a compute unit copies.  Measured, 16 experts of 1,536 x 4,096, 4 chosen a token, gate
// and up alone / with down in us, at 8, 64, 130, 211, 300, 400, 600, 1,024, 1,300, 2,048, 4,096 tokens:
//   32 rows (weights 64, 2 wavefronts, 4 stages)   68/101  70/110 105/161
//     not past the caches (weights 128, 3 stages)  79/115  84/125 109/159
//   64 rows (weights 128, 3 stages)                70/103  75/111  77/117   86/139  135/213 124/201  211/319
//     not past the caches                          79/115  85/126   89/131  88/142  108/178 101/168  148/238  215/335
//   128 rows (weights 256, 3 stages)                       90/130   94/134  95/139   95/144  97/145  163/239  143/246
//     not past the caches                                  96/138  101/147 102/150  104/154 107/158  164/236  138/241  199/309  276/452  480/786
//   192 rows (weights 192, down 256; X for down in 2 stages)                                         109/175  156/240  155/241  229/368  450/704
//     (since the loop's smaller matrix instruction and one-instruction copies: 2,048 tokens 209/331)
//   the kernels above, 32 rows, K shared           78/111 110/167  219/351
//   the kernels above, 128 rows                   150/231 150/231                                   370/688
template <bool DOWN>
void launch_tiles_for(const GroupArgs& a, int max_tiles, int rows, hipStream_t stream) {
    if (rows <= 32) launch_tiles<DOWN, 64, 32, 2, 1, 4, true>(a, max_tiles, stream);
    else if (rows <= 64) launch_tiles<DOWN, 128, 64, 4, 1, 3, true>(a, max_tiles, stream);
    else if (rows <= 128) launch_tiles<DOWN, 256, 128, 2, 2, 3, true>(a, max_tiles, stream);
    else if constexpr (DOWN) launch_tiles<DOWN, 256, 192, 2, 2, 3, false, 2>(a, max_tiles, stream);
    else launch_tiles<DOWN, 192, 192, 2, 2, 3, false>(a, max_tiles, stream);
}

}  // namespace

extern "C" int pulse_moe_group(const int* idx, int pairs, int experts, int tile_rows_max, int max_tiles, int* rank,
                               int* order, int* tile_expert, int* tile_row0, int* tile_rows, int* num_tiles,
                               hipStream_t stream) {
    PULSE_REQUIRE(pairs >= 0 && experts > 0 && experts <= MAX_EXPERTS, "moe_group: at most %d experts, got %d",
                  MAX_EXPERTS, experts);
    PULSE_REQUIRE(tile_rows_max > 0 && tile_rows_max % 16 == 0, "moe_group: tiles hold a multiple of 16 rows");
    PULSE_REQUIRE(max_tiles >= (pairs + tile_rows_max - 1) / tile_rows_max + experts,
                  "moe_group: %d tiles cannot hold %d pairs of %d experts in every case", max_tiles, pairs, experts);
    PULSE_REQUIRE(idx && rank && order && tile_expert && tile_row0 && tile_rows && num_tiles, "moe_group: null pointer");
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(GROUP_THREADS), 0, stream, idx, pairs, experts, tile_rows_max,
                       max_tiles, rank, order, tile_expert, tile_row0, tile_rows, num_tiles);
    PULSE_LAUNCH_CHECK("moe_group");
    return 0;
}

static bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Whether `rows` rows of K values, and a tile's rows of a weight (256 at most), lie as near the first as moe_tile_kernel's 32-bit offsets
// reach (with the pieces and BACK and `inside` of TileLoop).
static bool near_rows(int64_t rows, int64_t K) { return std::max<int64_t>(rows, 256) * K * 2 + 8192 < (int64_t{1} << 32); }

extern "C" int pulse_moe_gate_up_grouped(const void* x, const void* wg, const void* wu, const int* order,
                                         const int* tile_expert, const int* tile_row0, const int* tile_rows,
                                         const int* num_tiles, int max_tiles, int tile_rows_max, void* act, int hidden,
                                         int ff, int top, const float* in_weight, int act_kind, float limit,
                                         hipStream_t stream) {
    PULSE_REQUIRE(act_kind == 0 || act_kind == 1, "moe_gate_up_grouped: unknown activation %d", act_kind);
    PULSE_REQUIRE(hidden > 0 && ff > 0 && top > 0 && max_tiles > 0, "moe_gate_up_grouped: bad sizes");
    PULSE_REQUIRE(hidden % 8 == 0 && aligned16(x) && aligned16(wg) && aligned16(wu),
                  "moe_gate_up_grouped: rows must be multiples of 8 values and 16-byte aligned");
    PULSE_REQUIRE(tile_rows_max == 32 || tile_rows_max == 64 || tile_rows_max == 128 || tile_rows_max == 192, "moe_gate_up_grouped: tiles of 32, 64, 128 or 192 rows");
    PULSE_REQUIRE(x && wg && wu && order && tile_expert && tile_row0 && tile_rows && num_tiles && act,
                  "moe_gate_up_grouped: null pointer");
    PULSE_REQUIRE((ff + 15) / 16 < 65536, "moe_gate_up_grouped: an inner width of %d is too large", ff);
    // (the loop walks K in whole steps of 64; rows leave in 16-byte pieces; the tiles have room for every pair)
    if (hidden % 64 == 0 && ff % 8 == 0 && aligned16(act) && near_rows(static_cast<int64_t>(max_tiles) * tile_rows_max / top + 1, hidden)) {
        launch_tiles_for<false>({static_cast<const bf16_t*>(x), {static_cast<const bf16_t*>(wg), static_cast<const bf16_t*>(wu)},
                                 act, order, tile_expert, tile_row0, tile_rows, num_tiles, in_weight, hidden, ff, top, 0,
                                 act_kind, limit}, max_tiles, tile_rows_max, stream);
        PULSE_LAUNCH_CHECK("moe_gate_up_grouped");
        return 0;
    }
    const dim3 grid(max_tiles, (ff + 63) / 64, (tile_rows_max + 127) / 128);
    if (tile_rows_max == 32)
        hipLaunchKernelGGL(moe_gate_up_grouped_kernel<2>, dim3(max_tiles, (ff + 15) / 16), dim3(256), 0, stream, static_cast<const bf16_t*>(x),
                           static_cast<const bf16_t*>(wg), static_cast<const bf16_t*>(wu), order, tile_expert, tile_row0,
                           tile_rows, num_tiles, static_cast<bf16_t*>(act), hidden, ff, top, in_weight, act_kind, limit);
    else
        hipLaunchKernelGGL(moe_gate_up_grouped_kernel<8>, grid, dim3(256), 0, stream, static_cast<const bf16_t*>(x),
                           static_cast<const bf16_t*>(wg), static_cast<const bf16_t*>(wu), order, tile_expert, tile_row0,
                           tile_rows, num_tiles, static_cast<bf16_t*>(act), hidden, ff, top, in_weight, act_kind, limit);
    PULSE_LAUNCH_CHECK("moe_gate_up_grouped");
    return 0;
}

extern "C" int pulse_moe_down_grouped(const void* act, const void* wd, const int* order, const int* tile_expert,
                                      const int* tile_row0, const int* tile_rows, const int* num_tiles, int max_tiles,
                                      int tile_rows_max, float* y, int hidden, int ff, hipStream_t stream) {
    PULSE_REQUIRE(hidden > 0 && ff > 0 && max_tiles > 0, "moe_down_grouped: bad sizes");
    PULSE_REQUIRE(ff % 8 == 0 && aligned16(act) && aligned16(wd),
                  "moe_down_grouped: rows must be multiples of 8 values and 16-byte aligned");
    PULSE_REQUIRE(tile_rows_max == 32 || tile_rows_max == 64 || tile_rows_max == 128 || tile_rows_max == 192, "moe_down_grouped: tiles of 32, 64, 128 or 192 rows");
    PULSE_REQUIRE(act && wd && order && tile_expert && tile_row0 && tile_rows && num_tiles && y,
                  "moe_down_grouped: null pointer");
    PULSE_REQUIRE((hidden + 15) / 16 < 65536, "moe_down_grouped: a width of %d is too large", hidden);
    if (ff % 64 == 0 && hidden % 4 == 0 && aligned16(y) && near_rows(static_cast<int64_t>(max_tiles) * tile_rows_max, ff)) {
        launch_tiles_for<true>({static_cast<const bf16_t*>(act), {static_cast<const bf16_t*>(wd), nullptr}, y, order, tile_expert,
                                tile_row0, tile_rows, num_tiles, nullptr, ff, hidden, 1, 0, 0, 0.f}, max_tiles, tile_rows_max, stream);
        PULSE_LAUNCH_CHECK("moe_down_grouped");
        return 0;
    }
    const dim3 grid(max_tiles, (hidden + 63) / 64, (tile_rows_max + 127) / 128);
    if (tile_rows_max == 32)
        hipLaunchKernelGGL(moe_down_grouped_kernel<2>, dim3(max_tiles, (hidden + 15) / 16), dim3(256), 0, stream, static_cast<const bf16_t*>(act),
                           static_cast<const bf16_t*>(wd), order, tile_expert, tile_row0, tile_rows, num_tiles, y, hidden, ff);
    else
        hipLaunchKernelGGL(moe_down_grouped_kernel<8>, grid, dim3(256), 0, stream, static_cast<const bf16_t*>(act),
                           static_cast<const bf16_t*>(wd), order, tile_expert, tile_row0, tile_rows, num_tiles, y, hidden, ff);
    PULSE_LAUNCH_CHECK("moe_down_grouped");
    return 0;
}

extern "C" int pulse_moe_combine(const void* x, int x_dtype, const float* y, const int* idx, const float* weight,
                                 float* out, int tokens, int hidden, int experts, int top, hipStream_t stream) {
    PULSE_REQUIRE(tokens >= 0 && hidden > 0 && top > 0 && x && y && idx && out && pulse_dtype_ok(x_dtype),
                  "moe_combine: bad arguments");
    const int64_t total = static_cast<int64_t>(tokens) * hidden;
    if (total == 0) return 0;
    const int64_t blocks = (total + 255) / 256;
    PULSE_REQUIRE(blocks < (1ll << 31), "moe_combine: too many elements");
    PULSE_DISPATCH_DTYPE(x_dtype, TX,
        hipLaunchKernelGGL(moe_combine_kernel<TX>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,
                           static_cast<const TX*>(x), y, idx, weight, out, total, hidden, experts, top));
    PULSE_LAUNCH_CHECK("moe_combine");
    return 0;
}
