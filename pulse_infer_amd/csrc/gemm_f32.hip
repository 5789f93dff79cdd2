// C[M, N] = A[M, K] * W[N, K]^T in float32, every output added up in an order of its own that M has no part in.
//
// This is the matrix product of the true 32-bit path.  Float32 operands with a large weight are multiplied as parts on the
// bfloat16 instruction (gemm_split.hip, which is no less exact), whatever the number of rows; all others here on
// v_mfma_f32_16x16x4_f32, which multiplies and accumulates in float32 (no reduced-precision mode).  Inputs may be stored as
// bfloat16 (they are widened exactly).  (reference: cublasSgemm, src/ops/kernels/cuda/matmul_kernel.cu:70-88)
//
// The order: K is cut into blocks of 16 and the blocks into four shares, one a wavefront of the workgroup that owns the
// output; a share is added up block after block, and the four shares in their order.  The cut depends on K alone and
// every shape of tile walks a share in the same way, so a row's result does not depend on what else is in the batch.
//
// What bounds it: the matrix cores (256 float32 operations a clock and compute unit) from about 100 rows on, the weights'
// way from memory below.  Wavefronts that share K instead of the tile fetch nothing twice in a workgroup and walk without
// a barrier; the next blocks are asked for before these are multiplied.  Measured against scalar multiply-adds on a 64 x 64 tile
// in LDS (16 k a barrier): 2,048 x 8,192 at 333 rows 830 -> 105 us (106 TFLOP/s).  The error against 64 bits is half that of one sum
// (K of 2,048: 8e-7 -> 4e-7): four shorter sums.
#include "common.h"
#include "gemm_split.h"
#include "tile_loop.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int SHARES = 4;   // wavefronts a workgroup, each with a share of K
constexpr int KB = 16;      // k a block: four a lane group of the matrix instruction

struct GemmArgs {
    const void* A;
    const void* W;
    void* C;
    int c_bf16;
    int c_wide;     // float32 results can be stored four at a time
    int M, N, K;
    int64_t lda, ldw, ldc;
    int tiles_m, tiles_n;
};

// Values k .. k + 3 of a row that can be read in pieces of four, K a multiple of 4; a piece past the end is the row's last
// piece, read for nobody, so that no lane branches round a load.
template <typename T>
__device__ __forceinline__ f32x4 load4(const T* row, int k, int K) {
    f32x4 v;
    const int at = min(k, K - 4);
    if constexpr (sizeof(T) == 4) {
        v = *reinterpret_cast<const f32x4*>(row + at);
    } else {
        const uint2 raw = *reinterpret_cast<const uint2*>(row + at);
        v[0] = __uint_as_float(raw.x << 16);
        v[1] = __uint_as_float(raw.x & 0xffff0000u);
        v[2] = __uint_as_float(raw.y << 16);
        v[3] = __uint_as_float(raw.y & 0xffff0000u);
    }
    return v;
}

// Four results of row m, for weight rows n .. n + 3 (a lane of the matrix instruction's result holds weight rows
// 4 * (l / 16) + e for row l % 16 of A).
__device__ __forceinline__ void store_tile(const GemmArgs& a, int m, int n, f32x4 v) {
    if (m >= a.M) return;
    const int64_t at = static_cast<int64_t>(m) * a.ldc + n;
    if (a.c_bf16) {
        bf16_t* c = static_cast<bf16_t*>(a.C) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < a.N) c[e] = f32_to_bf16(v[e]);
    } else if (a.c_wide) {
        if (n < a.N) *reinterpret_cast<f32x4*>(static_cast<float*>(a.C) + at) = v;
    } else {
        float* c = static_cast<float*>(a.C) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < a.N) c[e] = v[e];
    }
}

// A workgroup's tile is 16 * BN weight rows (the row operand) by 16 * BM rows of A (the column operand); U blocks of k
// are a stage.
template <typename TA, typename TW, int BM, int BN, int U>
__global__ __launch_bounds__(SHARES* PULSE_WAVE) void gemm_f32_kernel(GemmArgs a) {
    constexpr int TILES = BM * BN;
    constexpr int PASS = TILES % 8 == 0 ? 8 : TILES % 6 == 0 ? 6 : TILES % 9 == 0 ? 9 : TILES;     // tiles of the matrix instruction a pass of the meeting in LDS
    __shared__ f32x4 meet[SHARES][PASS][PULSE_WAVE];

    // (the workgroups of a die, every eighth, take neighbouring tiles: those of one span of weight rows)
    const int total = a.tiles_m * a.tiles_n;
    const int per_die = (total + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || tile >= total) return;
    const int m0 = tile % a.tiles_m * (16 * BM), n0 = tile / a.tiles_m * (16 * BN);

    const int lane = threadIdx.x % PULSE_WAVE;
    const int share = threadIdx.x / PULSE_WAVE;
    const int r = lane % 16, kg = lane / 16;
    const int blocks = (a.K + KB - 1) / KB;
    const int b_end = static_cast<int>(static_cast<int64_t>(blocks) * (share + 1) / SHARES);
    int b = static_cast<int>(static_cast<int64_t>(blocks) * share / SHARES);

    // (rows past the end are the last row again: their results are not written)
    const TA* arow[BM];
    const TW* wrow[BN];
#pragma unroll
    for (int i = 0; i < BM; ++i)
        arow[i] = static_cast<const TA*>(a.A) + static_cast<int64_t>(min(m0 + 16 * i + r, a.M - 1)) * a.lda;
#pragma unroll
    for (int j = 0; j < BN; ++j)
        wrow[j] = static_cast<const TW*>(a.W) + static_cast<int64_t>(min(n0 + 16 * j + r, a.N - 1)) * a.ldw;

    f32x4 acc[BN][BM];
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
        for (int i = 0; i < BM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 av[2][U][BM], wv[2][U][BN];
    auto fetch = [&](int set, int block) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (block + u) * KB + 4 * kg;
#pragma unroll
            for (int j = 0; j < BN; ++j) wv[set][u][j] = load4<TW>(wrow[j], k, a.K);
#pragma unroll
            for (int i = 0; i < BM; ++i) av[set][u][i] = load4<TA>(arow[i], k, a.K);
        }
        __builtin_amdgcn_sched_barrier(0);   // (the loads stay ahead of the products that they hide behind)
    };
    auto multiply = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < BN; ++j)
#pragma unroll
                    for (int i = 0; i < BM; ++i)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[set][u][j][e], av[set][u][i][e], acc[j][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // What lies behind the share's end is zeros on both sides, which leaves the sums as they are.
    const int k_end = min(a.K, b_end * KB);
    auto clear_behind = [&](int set, int block) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (block + u) * KB + 4 * kg;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool in = k + e < k_end;
#pragma unroll
                for (int j = 0; j < BN; ++j) wv[set][u][j][e] = in ? wv[set][u][j][e] : 0.f;
#pragma unroll
                for (int i = 0; i < BM; ++i) av[set][u][i][e] = in ? av[set][u][i][e] : 0.f;
            }
        }
    };
    const int b_full = min(b_end, a.K / KB);    // blocks that lie inside K as a whole
    fetch(0, b);
    for (; b + 2 * U <= b_full; b += 2 * U) {
        fetch(1, b + U);
        multiply(0);
        fetch(0, b + 2 * U);
        multiply(1);
    }
    for (; b < b_end; b += 2 * U) {             // (at most twice)
        fetch(1, b + U);
        clear_behind(0, b);
        multiply(0);
        clear_behind(1, b + U);
        multiply(1);
        if (b + 2 * U < b_end) fetch(0, b + 2 * U);
    }

    // The shares meet in LDS, a few tiles at a time; wavefront t % 4 adds up the four results of tile t.
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += PASS) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) meet[share][t][lane] = acc[(t0 + t) / BM][(t0 + t) % BM];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) {
            if (t % SHARES != share) continue;
            f32x4 v = meet[0][t][lane];
#pragma unroll
            for (int s = 1; s < SHARES; ++s) v += meet[s][t][lane];
            store_tile(a, m0 + 16 * ((t0 + t) % BM) + r, n0 + 16 * ((t0 + t) / BM) + 4 * kg, v);
        }
    }
}

// The same walk for many rows of float32 operands, the operands through LDS: read straight into registers, the sixteen
// lanes that an instruction serves together touch sixteen rows, and the compute unit's cache looks up a line for 16
// bytes of each.  A wavefront copies its own share's blocks (16 rows x 64 bytes an instruction, four lanes a row) into
// S stages of its own, so the walk has no barrier here either.
template <int BM, int BN, int S>
__global__ __launch_bounds__(SHARES* PULSE_WAVE) void gemm_f32_staged_kernel(GemmArgs a) {
    constexpr int TILES = BM * BN;
    constexpr int STAGE = (BM + BN) * 1024;
    constexpr int PASS = TILES % 8 == 0 ? 8 : TILES % 6 == 0 ? 6 : TILES % 9 == 0 ? 9 : TILES;
    constexpr int MEET = SHARES * PASS * PULSE_WAVE * 16;
    __shared__ __attribute__((aligned(1024))) char lds[SHARES * S * STAGE > MEET ? SHARES * S * STAGE : MEET];

    const int total = a.tiles_m * a.tiles_n;
    const int per_die = (total + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || tile >= total) return;
    const int m0 = tile % a.tiles_m * (16 * BM), n0 = tile / a.tiles_m * (16 * BN);

    const int lane = threadIdx.x % PULSE_WAVE;
    const int share = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int r = lane % 16, kg = lane / 16;
    const int blocks = (a.K + KB - 1) / KB;
    const int b_end = static_cast<int>(static_cast<int64_t>(blocks) * (share + 1) / SHARES);
    const int b0 = static_cast<int>(static_cast<int64_t>(blocks) * share / SHARES);

    // Copies: lane i brings the piece that belongs at place i % 4 of row i / 4; piece c of row q sits at place
    // c ^ (q / 4 % 4), so that the eight lanes which LDS serves together read eight different places.
    const int crow = lane / 4, cpiece = (lane % 4) ^ (crow / 4 % 4);
    const float* from[BN + BM];
#pragma unroll
    for (int j = 0; j < BN; ++j)
        from[j] = static_cast<const float*>(a.W) + static_cast<int64_t>(min(n0 + 16 * j + crow, a.N - 1)) * a.ldw;
#pragma unroll
    for (int i = 0; i < BM; ++i)
        from[BN + i] = static_cast<const float*>(a.A) + static_cast<int64_t>(min(m0 + 16 * i + crow, a.M - 1)) * a.lda;
    char* mine = lds + share * S * STAGE;
    const uint32_t mine_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (void __attribute__((address_space(3)))*)(mine)));
    auto copy = [&](int block, int stage) __attribute__((always_inline)) {
        const int at = min(block * KB + 4 * cpiece, a.K - 4);    // (past the end: the row's last piece, for nobody)
#pragma unroll
        for (int t = 0; t < BN + BM; ++t) load_to_lds(from[t] + at, mine_at + stage * STAGE + t * 1024);
    };

    f32x4 acc[BN][BM];
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
        for (int i = 0; i < BM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int read_at = r * 64 + (kg ^ (r / 4 % 4)) * 16;
    const int k_end = min(a.K, b_end * KB);
    auto multiply = [&](int stage, int block, bool whole) __attribute__((always_inline)) {
        f32x4 v[BN + BM];
#pragma unroll
        for (int t = 0; t < BN + BM; ++t) v[t] = *reinterpret_cast<const f32x4*>(mine + stage * STAGE + t * 1024 + read_at);
        if (!whole) {    // what lies behind the share's end is zeros on both sides
#pragma unroll
            for (int t = 0; t < BN + BM; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[t][e] = block * KB + 4 * kg + e < k_end ? v[t][e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < BN; ++j)
#pragma unroll
                for (int i = 0; i < BM; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][e], v[BN + i][e], acc[j][i], 0, 0, 0);
    };
    // Block b lies in stage (b - b0) % S; S - 1 blocks are on their way while one is multiplied.
#pragma unroll
    for (int s = 0; s < S - 1; ++s) copy(b0 + s, s);
    const int b_full = min(b_end, a.K / KB);
    int stage = 0;
    for (int b = b0; b < b_end; ++b) {
        const int next = stage == 0 ? S - 1 : stage - 1;
        // (the reads of the stage that this copy goes to, those of the block before, have returned: the products that use
        // them may be placed behind the copy, and the compiler does not know that it writes there)
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        copy(b + S - 1, next);
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"((S - 1) * (BN + BM)) : "memory");
        multiply(stage, b, b < b_full);
        stage = stage == S - 1 ? 0 : stage + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // the last copies, which nobody reads, must not land in what follows
    __syncthreads();

    f32x4* meet = reinterpret_cast<f32x4*>(lds);          // [SHARES][PASS][64]
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += PASS) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) meet[(share * PASS + t) * PULSE_WAVE + lane] = acc[(t0 + t) / BM][(t0 + t) % BM];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) {
            if (t % SHARES != share) continue;
            f32x4 v = meet[t * PULSE_WAVE + lane];
#pragma unroll
            for (int s = 1; s < SHARES; ++s) v += meet[(s * PASS + t) * PULSE_WAVE + lane];
            store_tile(a, m0 + 16 * ((t0 + t) % BM) + r, n0 + 16 * ((t0 + t) / BM) + 4 * kg, v);
        }
    }
}

// The same walk for rows that cannot be read in pieces of four (their length or distance is no multiple of four values):
// a block's 16 rows are read four rows an instruction, the 16 values of each side by side, so that an instruction touches
// four to eight lines where value e of every lane's piece touches sixteen, and go through LDS of the wavefront's own into the
// operands' order.  2,050 weight rows of 1,001, float32 and bfloat16: 4,096 rows 273 and 265 us, straight into registers 734
// and 783 (scalar multiply-adds on a 64 x 64 tile in LDS 527 and 460); 17 rows 10.8 and 10.7, 21.5 and 31.3 (177 and 128).
template <typename TA, typename TW, int BM, int BN>
__global__ __launch_bounds__(SHARES* PULSE_WAVE) void gemm_f32_ragged_kernel(GemmArgs a) {
    constexpr int TILES = BM * BN, T = BM + BN;
    constexpr int PASS = TILES % 8 == 0 ? 8 : TILES % 6 == 0 ? 6 : TILES % 9 == 0 ? 9 : TILES;
    constexpr int STAGE = T * 1024, MEET = SHARES * PASS * PULSE_WAVE * 16;
    __shared__ __attribute__((aligned(1024))) char lds[SHARES * STAGE > MEET ? SHARES * STAGE : MEET];

    const int total = a.tiles_m * a.tiles_n;
    const int per_die = (total + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || tile >= total) return;
    const int m0 = tile % a.tiles_m * (16 * BM), n0 = tile / a.tiles_m * (16 * BN);

    const int lane = threadIdx.x % PULSE_WAVE;
    const int share = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int r = lane % 16, kg = lane / 16;
    const int blocks = (a.K + KB - 1) / KB;
    const int b_end = static_cast<int>(static_cast<int64_t>(blocks) * (share + 1) / SHARES);
    const int b0 = static_cast<int>(static_cast<int64_t>(blocks) * share / SHARES);

    // raw[t][e]: value lane % 16 of row 4 e + lane / 16 of the t-th sixteen rows; piece c of row q sits at place c ^ (q / 4 % 4)
    float raw[T][4];
    auto fetch = [&](int block) __attribute__((always_inline)) {
        const int k = block * KB + r;
        const bool in = k < a.K;
        const int at = in ? k : a.K - 1;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 4 * e + kg;
                if (t < BN)
                    raw[t][e] = to_f32<TW>(static_cast<const TW*>(a.W)[static_cast<int64_t>(min(n0 + 16 * t + row, a.N - 1)) * a.ldw + at]);
                else
                    raw[t][e] = to_f32<TA>(static_cast<const TA*>(a.A)[static_cast<int64_t>(min(m0 + 16 * (t - BN) + row, a.M - 1)) * a.lda + at]);
                raw[t][e] = in ? raw[t][e] : 0.f;
            }
        __builtin_amdgcn_sched_barrier(0);   // (the loads stay ahead of the products that they hide behind)
    };
    float* mine = reinterpret_cast<float*>(lds + share * STAGE);
    f32x4 v[T];
    auto turn = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[t * 256 + (4 * e + kg) * 16 + ((r / 4) ^ e) * 4 + r % 4] = raw[t][e];
        tile_wave_sync();
#pragma unroll
        for (int t = 0; t < T; ++t) v[t] = *reinterpret_cast<const f32x4*>(mine + t * 256 + r * 16 + (kg ^ (r / 4 % 4)) * 4);
        tile_wave_sync();
    };

    f32x4 acc[BN][BM];
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
        for (int i = 0; i < BM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (b0 < b_end) {
        fetch(b0);
        turn();
        for (int b = b0; b < b_end; ++b) {
            if (b + 1 < b_end) fetch(b + 1);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < BN; ++j)
#pragma unroll
                    for (int i = 0; i < BM; ++i)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][e], v[BN + i][e], acc[j][i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (b + 1 < b_end) turn();
        }
    }
    __syncthreads();

    f32x4* meet = reinterpret_cast<f32x4*>(lds);          // [SHARES][PASS][64]
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += PASS) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) meet[(share * PASS + t) * PULSE_WAVE + lane] = acc[(t0 + t) / BM][(t0 + t) % BM];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < PASS; ++t) {
            if (t % SHARES != share) continue;
            f32x4 sum = meet[t * PULSE_WAVE + lane];
#pragma unroll
            for (int s = 1; s < SHARES; ++s) sum += meet[(s * PASS + t) * PULSE_WAVE + lane];
            store_tile(a, m0 + 16 * ((t0 + t) % BM) + r, n0 + 16 * ((t0 + t) / BM) + 4 * kg, sum);
        }
    }
}

template <typename TA, typename TW, int BM, int BN>
void launch_ragged(GemmArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + 16 * BM - 1) / (16 * BM);
    a.tiles_n = (a.N + 16 * BN - 1) / (16 * BN);
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(a.tiles_m) * a.tiles_n + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_f32_ragged_kernel<TA, TW, BM, BN>), dim3(grid), dim3(SHARES * PULSE_WAVE), 0, stream, a);
}

// Up to 128 rows tiles of 16 x 32, of which there are enough (100 rows, 2,050 x 1,001: 14.5 us, 19.1 with 32 x 32); beyond, 32
// x 64 where a compute unit gets eight or more of them (4,096 rows: 273 us, 313 with 32 x 32), else 32 x 32 (1,024 rows: 81, 85
// with 32 x 64; 48 x 64 and 64 x 64 were slower throughout, 334 and 301 at 4,096 rows).
template <typename TA, typename TW>
void launch_ragged_for(const GemmArgs& a, hipStream_t stream) {
    const int64_t wide = static_cast<int64_t>((a.M + 31) / 32) * ((a.N + 63) / 64);
    if (a.M <= 128) launch_ragged<TA, TW, 1, 2>(a, stream);
    else if (wide >= 8 * static_cast<int64_t>(pulse_compute_units())) launch_ragged<TA, TW, 2, 4>(a, stream);
    else launch_ragged<TA, TW, 2, 2>(a, stream);
}

template <int BM, int BN, int S>
void launch_staged(GemmArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + 16 * BM - 1) / (16 * BM);
    a.tiles_n = (a.N + 16 * BN - 1) / (16 * BN);
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(a.tiles_m) * a.tiles_n + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_f32_staged_kernel<BM, BN, S>), dim3(grid), dim3(SHARES * PULSE_WAVE), 0, stream, a);
}

template <typename TA, typename TW, int BM, int BN, int U>
void launch(GemmArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + 16 * BM - 1) / (16 * BM);
    a.tiles_n = (a.N + 16 * BN - 1) / (16 * BN);
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(a.tiles_m) * a.tiles_n + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_f32_kernel<TA, TW, BM, BN, U>), dim3(grid), dim3(SHARES * PULSE_WAVE), 0, stream, a);
}

}  // namespace

static int gemm_f32(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype, int M, int N, int K, int64_t lda,
                    int64_t ldw, int64_t ldc, void* scratch, hipStream_t stream) {
    PULSE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
    PULSE_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: leading dimensions too small");
    PULSE_REQUIRE(pulse_dtype_ok(a_dtype) && pulse_dtype_ok(w_dtype) && pulse_dtype_ok(c_dtype), "gemm_f32: bad dtype tag");
    PULSE_REQUIRE(A && W && C, "gemm_f32: null pointer");
    if (M == 0) return 0;
    PULSE_REQUIRE((M + 63) / 64 < 65536, "gemm_f32: M=%d is too large for one launch", M);
    PULSE_REQUIRE(static_cast<int64_t>((M + 15) / 16) * ((N + 15) / 16) < (1ll << 30), "gemm_f32: %d x %d outputs are too many",
                  M, N);
    const bool wide = c_dtype == PULSE_F32 && ldc % 4 == 0 && N % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
    GemmArgs a{A, W, C, c_dtype == PULSE_BF16 ? 1 : 0, wide ? 1 : 0, M, N, K, lda, ldw, ldc, 0, 0};
    const int a_size = a_dtype == PULSE_BF16 ? 2 : 4, w_size = w_dtype == PULSE_BF16 ? 2 : 4;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && reinterpret_cast<uintptr_t>(A) % (4 * a_size) == 0 &&
                     reinterpret_cast<uintptr_t>(W) % (4 * w_size) == 0;
    if (a_size == 4 && w_size == 4 && vec && pulse_split_takes(N, K)) {
        pulse_split_launch(static_cast<const float*>(A), static_cast<const float*>(W), C, a.c_bf16 != 0, wide, M, N, K, lda, ldw, ldc,
                           ldw < (1 << 25) ? scratch : nullptr, stream);
        PULSE_LAUNCH_CHECK("gemm_f32");
        return 0;
    }
    // Up to 16 rows a product is the weights' way from memory: tiles of one block of weight rows with four blocks of k a
    // stage, four blocks of weight rows where there are enough of them for every compute unit (16,384 x 2,048 at 12 rows
    // 38 -> 30 us; 2,048 x 8,192 29 -> 74).
    if (M <= 16 || !vec || a_size != 4 || w_size != 4) {
        PULSE_DISPATCH_DTYPE(a_dtype, TA, PULSE_DISPATCH_DTYPE(w_dtype, TW,
            if (!vec) launch_ragged_for<TA, TW>(a, stream);
            else if (M > 16) launch<TA, TW, 2, 2, 2>(a, stream);
            else if (N >= 64 * pulse_compute_units()) launch<TA, TW, 1, 4, 2>(a, stream);
            else launch<TA, TW, 1, 1, 4>(a, stream)));
    } else {
        // The tile whose fullest compute unit ends first: workgroups on it x (pairs of blocks in a tile + 2, what a
        // workgroup costs beside its products).  Measured at 333 rows: 2,048 weight rows of 8,192 133 / 144 / 105 / 134 us
        // with tiles of 2 x 2, 2 x 4, 3 x 4, 4 x 4 blocks, the rule's 18 / 20 / 14 / 18; 16,384 of 2,048 248 / 225 / 202 /
        // 220 us, 132 / 110 / 98 / 108.
        static constexpr int shapes[][2] = {{4, 4}, {3, 4}, {2, 4}, {2, 2}};
        const int64_t units = pulse_compute_units();
        int best = 0;
        int64_t least = 0;
        for (int i = 0; i < 4; ++i) {
            const int64_t tiles = static_cast<int64_t>((M + 16 * shapes[i][0] - 1) / (16 * shapes[i][0])) *
                                  ((N + 16 * shapes[i][1] - 1) / (16 * shapes[i][1]));
            const int64_t cost = (tiles + units - 1) / units * (shapes[i][0] * shapes[i][1] + 2);
            if (i == 0 || cost < least) { best = i; least = cost; }
        }
        if (best == 0) launch_staged<4, 4, 3>(a, stream);
        else if (best == 1) launch_staged<3, 4, 3>(a, stream);
        else if (best == 2) launch_staged<2, 4, 3>(a, stream);
        else launch_staged<2, 2, 3>(a, stream);
    }
    PULSE_LAUNCH_CHECK("gemm_f32");
    return 0;
}

extern "C" int pulse_gemm_f32(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                              int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc, hipStream_t stream) {
    return gemm_f32(A, a_dtype, W, w_dtype, C, c_dtype, M, N, K, lda, ldw, ldc, nullptr, stream);
}

// How many bytes of scratch make the product of float32 operands of these sizes fastest (0: none).
extern "C" int64_t pulse_gemm_f32_scratch(int M, int N, int K) { return M > 0 && N > 0 && K > 0 && K % 4 == 0 ? pulse_split_scratch(M, N, K) : 0; }

// The same product, bit for bit, with that many bytes of scratch.
extern "C" int pulse_gemm_f32_scratched(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype, int M, int N, int K,
                                        int64_t lda, int64_t ldw, int64_t ldc, void* scratch, int64_t scratch_bytes, hipStream_t stream) {
    PULSE_REQUIRE(scratch != nullptr && reinterpret_cast<uintptr_t>(scratch) % 16 == 0, "gemm_f32: the scratch must be 16-byte aligned");
    PULSE_REQUIRE(scratch_bytes >= pulse_gemm_f32_scratch(M, N, K), "gemm_f32: %lld bytes of scratch, %lld are needed",
                  static_cast<long long>(scratch_bytes), static_cast<long long>(pulse_gemm_f32_scratch(M, N, K)));
    return gemm_f32(A, a_dtype, W, w_dtype, C, c_dtype, M, N, K, lda, ldw, ldc, scratch, stream);
}
