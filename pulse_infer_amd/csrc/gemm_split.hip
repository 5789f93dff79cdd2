// C[M, N] = A[M, K] * W[N, K]^T of float32 operands on the bfloat16 matrix instruction, no less exact than on the float32 one.
// (reference: cublasSgemm, src/ops/kernels/cuda/matmul_kernel.cu:70-88)
//
// A float32 value is the sum of three bfloat16 parts, exactly: the value rounded, what that leaves rounded, the rest (8 + 8 + 8
// bits).  Of the nine products of two values' parts the six largest are made (second x third, third x second and third x third are
// not: at most 2^-26 of the product are left out, a quarter of a float32 rounding), each exact, on v_mfma_f32_16x16x32_bf16
// with float32 sums.  That instruction does sixteen times the arithmetic of v_mfma_f32_16x16x4_f32, so six of it take 3/8 of the
// time.  Error against 64 bits, relative, normal operands, K of 2,048 / 8,192: 2.4e-7 / 5.1e-7, the float32 instruction with
// four shares of K 4.1e-7 / 8.1e-7; largest difference over the result's root mean square 1.7e-6 / 3.1e-6 against 3.3e-6 /
// 6e-6; positive operands, and operands whose sizes spread over e^3, likewise smaller.
//
// The order: K is cut into blocks of 32 and the blocks into eight shares.  A share is added up block after block, in a block
// product after product as `w_part` and `x_part` say, and the shares in their order.  The cut depends on K alone and every way
// below does the same, so a row's result does not depend on what else is in the batch, bit for bit.
//
// Range: so exact for rows (of a share) whose largest value is at least 2^-100 and below 2^60, or that are zeros.  Any other row,
// one with an infinity or NaN among them, is flagged, and results of flagged rows are made anew on the float32 instruction
// (`replace_flagged`): products of parts would overflow, or make a NaN of an infinity times zero.  In a row that is not flagged what is
// lost of a value is below 2^-126: a value below 2^-110 loses of its third part, which shows only where every larger value of
// the row meets a zero (values of 2^-110 / 2^-115 / 2^-118 alone: 2.9e-7 / 4.9e-7 / 3.1e-6, the float32 instruction 4.1e-7).
//
// Ways: up to some hundreds of rows both operands are taken apart as they go (gemm_split_staged_kernel); from there on X once
// (gemm_split_prepare_kernel), multiplied in tiles of 64 or 96 x 256 whose wavefronts take the weights apart
// (gemm_split_tile_kernel), K in one go or its shares over workgroups, added up by gemm_split_sum_kernel.  `way_for` chooses.
// What bounds the tiles: 333 x 16,384 x 2,048 takes 125 us, its matrix instructions alone 91 (the power limit: 1.47 PFLOP/s);
// the difference is the issue of the weights' arithmetic, 104 instructions a wavefront and block beside 72 products.  Two
// wavefronts a SIMD are what hides it: with one, 160 us.  Taking X apart in the tiles, as its weights, 146 to 160.  What bounds the
// staged way: the weights' way from memory up to 32 rows (5.3 TB/s at 16,384 x 2,048), the issue of that arithmetic beyond.
// Measured, weight rows x K from memory, us, float32 instruction -> parts:
//                     1 row         12 rows       24            64            97            200           333           1,024
//   16,384 x 2,048    28 -> 25      30 -> 26      31 -> 29      44 -> 39      77 -> 66      144 -> 96     203 -> 123    584 -> 346
//   3,072 x 2,048     7.8 -> 8.3    10.0 -> 8.9   14.4 -> 11.2  14.8 -> 14.3  22 -> 22      30 -> 27      58 -> 42      110 -> 87
//   2,048 x 8,192     21 -> 23      30 -> 25      49 -> 25      50 -> 34      45 -> 42      76 -> 57      106 -> 73     270 -> 200
//   12,288 x 4,096    40 -> 36      52 -> 38      56 -> 50      74 -> 61      126 -> 96     209 -> 155    324 -> 198    828 -> 532
//   6,144 x 1,024     8.9 -> 8.8    11.4 -> 9.8   9.4 -> 10.1   14.2 -> 14.9  22 -> 21      33 -> 33      49 -> 47      122 -> 99
// (Read straight into registers by eight wavefronts a workgroup, up to 64 rows took 1.1 to 1.4 times the float32 instruction's time,
// and tiles at 40 to 200 rows of the smallest weights 1.1 to 1.7 times, by the two kernels beside them.)
#include "gemm_split.h"
#include "tile_loop.h"
#include <algorithm>
#include <cmath>

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;

constexpr int SHARES = 8;
constexpr int KB = 32;            // k a block: two of the matrix instruction's
constexpr uint32_t LOW = 0x0d80, HIGH = 0x5d80;   // 2^-100 and 2^60 as the upper half of a float32

// f(0) .. f(N - 1), each with its number as a constant.
template <int N> struct Number { static constexpr int value = N; };
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
    if constexpr (I < N) {
        f(Number<I>{});
        each<N, I + 1>(f);
    }
}

struct SplitArgs {
    const float* A;
    const float* W;
    void* C;
    int c_bf16;
    int c_wide;           // results can be stored four at a time
    int M, N, K;
    int64_t lda, ldw, ldc;
    int tiles_m, tiles_n;
    int groups;           // 1: a workgroup walks all shares; more: SHARES / groups of them each, with a float32 result a share
    int64_t part_stride;  // elements between the shares' results
    const char* xparts;   // X's parts (gemm_split_prepare_kernel) and, a byte a share and row, which rows are outside their range
    const uint8_t* xflags;
};

__device__ __forceinline__ int share_end(int blocks, int s) { return static_cast<int>(static_cast<int64_t>(blocks) * (s + 1) / SHARES); }

// Four pairs of values as the sums of three bfloat16 parts each, in steps of a few independent instructions, so that they can be
// spread over the matrix instructions: `x` holds what is left of the values, `part` two of a part side by side, `most` the
// largest magnitude of a first part so far (two of them).
constexpr int SPLIT_STEPS = 13;
template <int STEP>
__device__ __forceinline__ void split_step(f32x4 (&x)[2], uint32_t (&part)[3][4], uint32_t& most) {
    constexpr int P = STEP < 7 ? 0 : STEP < 12 ? 1 : 2;
    if constexpr (STEP == 0 || STEP == 7 || STEP == 12) {           // round
#pragma unroll
        for (int e = 0; e < 4; ++e)
            part[P][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x[e / 2][e % 2 * 2], x[e / 2][e % 2 * 2 + 1]}, bf16x2));
    } else if constexpr (STEP == 1 || STEP == 2) {
#pragma unroll
        for (int e = STEP * 2 - 2; e < STEP * 2; ++e)
            most = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, most), __builtin_bit_cast(u16x2, part[0][e] & 0x7fff7fffu)));
    } else {                                                        // subtract, a pair's values a step
        constexpr int e = STEP < 7 ? STEP - 3 : STEP - 8;
        x[e / 2][e % 2 * 2] -= __uint_as_float(part[P][e] << 16);
        x[e / 2][e % 2 * 2 + 1] -= __uint_as_float(part[P][e] & 0xffff0000u);
    }
}

__device__ __forceinline__ bool outside(uint32_t most) {
    const uint32_t top = max(most & 0xffffu, most >> 16);
    return top >= HIGH || (top != 0 && top < LOW);
}

__device__ __forceinline__ f32x4 load4(const float* row, int k, int K) {
    return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));
}

// The part of W and of X that product q of a block takes: second x second, third x first, first x third, second x first, first x
// second, first x first.
__device__ constexpr int w_part(int q) { return q == 1 ? 2 : q == 0 || q == 3 ? 1 : 0; }
__device__ constexpr int x_part(int q) { return q == 2 ? 2 : q == 0 || q == 4 ? 1 : 0; }

// A share's 16 x 16 results of which rows (of W, of X: a bit each) hold values outside the range of the parts, anew on the
// float32 instruction.
__device__ __forceinline__ void replace_flagged(f32x4& acc, uint32_t wbad, uint32_t xbad, const float* xrow, const float* wrow,
                                                int k0, int k1, int lane) {
    const int kg = lane / 16;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = k0; k < k1; k += 4) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wrow[k + kg], xrow[k + kg], sum, 0, 0, 0);
    const bool mine = (xbad >> (lane % 16)) & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = mine || ((wbad >> (4 * kg + i)) & 1) ? sum[i] : acc[i];
}

__device__ __forceinline__ void store_four(const SplitArgs& a, char* out, int m, int n, f32x4 v) {
    if (m >= a.M) return;
    const int64_t at = static_cast<int64_t>(m) * a.ldc + n;
    if (a.c_bf16) {
        bf16_t* c = reinterpret_cast<bf16_t*>(out) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < a.N) c[e] = f32_to_bf16(v[e]);
    } else if (a.c_wide) {
        if (n < a.N) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + at) = v;
    } else {
        float* c = reinterpret_cast<float*>(out) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < a.N) c[e] = v[e];
    }
}

// X's parts in the matrix instruction's operand order: for sixteen rows and a block of k, 1 KB a part, lane l's piece (row l %
// 16, values 8 (l / 16) ..) at 16 l.  A workgroup has sixteen rows and a share of K; rows past the end and values behind K are
// zeros.
constexpr int PREPARE_WAVES = 8;
__global__ __launch_bounds__(PREPARE_WAVES* PULSE_WAVE) void gemm_split_prepare_kernel(SplitArgs a, char* parts, uint8_t* flags) {
    __shared__ uint32_t tops[PREPARE_WAVES][16];
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    const int share = blockIdx.y, m = blockIdx.x * 16 + lane % 16;
    const int blocks = (a.K + KB - 1) / KB;
    const float* row = a.A + static_cast<int64_t>(min(m, a.M - 1)) * a.lda;
    uint32_t most = 0;
    for (int b = (share > 0 ? share_end(blocks, share - 1) : 0) + wave; b < share_end(blocks, share); b += PREPARE_WAVES) {
        const int k = b * KB + 8 * (lane / 16);
        f32x4 x[2] = {load4(row, k, a.K), load4(row, k + 4, a.K)};
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (m >= a.M || k + 4 * q >= a.K) x[q] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint32_t v[3][4];
        each<SPLIT_STEPS>([&](auto n) __attribute__((always_inline)) { split_step<decltype(n)::value>(x, v, most); });
        char* to = parts + (static_cast<int64_t>(blockIdx.x) * blocks + b) * 3072 + lane * 16;
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(to + p * 1024) = uint4{v[p][0], v[p][1], v[p][2], v[p][3]};
    }
    most = max(most & 0xffffu, most >> 16);
    most = max(most, static_cast<uint32_t>(__shfl_xor(most, 16)));
    most = max(most, static_cast<uint32_t>(__shfl_xor(most, 32)));
    if (lane < 16) tops[wave][lane] = most;
    __syncthreads();
    if (threadIdx.x < 16) {
        for (int w = 1; w < PREPARE_WAVES; ++w) most = max(most, tops[w][threadIdx.x]);
        flags[(static_cast<int64_t>(share) * gridDim.x + blockIdx.x) * 16 + threadIdx.x] = outside(most);
    }
}

// A workgroup's tile: 16 * TM rows of X by 256 weight rows, 32 a wavefront, which brings its own rows' values into LDS and takes
// them apart in registers for the next block between the products of this one; X's parts come to LDS as they are, for all.
constexpr int TILE_WAVES = 8, TILE_N = 32 * TILE_WAVES;
template <int TM, bool ALL>
__global__ __launch_bounds__(TILE_WAVES* PULSE_WAVE) void gemm_split_tile_kernel(SplitArgs a) {
    constexpr int SLOTS = 3;                                                       // of LDS, for X's parts and for the weights' values
    constexpr int TN = 2, PAIRS = TM / 2, EACH = 6 * TN * 2, G = PAIRS * EACH;     // products a pair of X's tiles, a block
    constexpr int XCHUNKS = 3 * TM, PX = (XCHUNKS + TILE_WAVES - 1) / TILE_WAVES, PW = 4, PC = PX + PW;  // copies of 1 KB a wavefront and block
    constexpr int XSLOT = XCHUNKS * 1024, WSLOT = PW * 1024, W0 = SLOTS * XSLOT;
    static_assert(TM % 2 == 0, "pairs of tiles");
    __shared__ __attribute__((aligned(1024))) char lds[W0 + TILE_WAVES * SLOTS * WSLOT];

    const int tiles = a.tiles_m * a.tiles_n, total = tiles * (ALL ? 1 : a.groups);
    const int per_die = (total + 7) / 8;
    const int t_all = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || t_all >= total) return;
    const int group = ALL ? 0 : t_all / tiles, t = t_all - group * tiles;
    const int share0 = ALL ? 0 : group * SHARES / a.groups, share1 = ALL ? SHARES : (group + 1) * SHARES / a.groups;
    const int m0 = t % a.tiles_m * (16 * TM);

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int lane = threadIdx.x % PULSE_WAVE, kg = lane / 16, r = lane % 16;
    const int n0 = t / a.tiles_m * TILE_N + wave * 32;
    const int blocks = (a.K + KB - 1) / KB, row_blocks = (a.M + 15) / 16;
    const int first = share0 > 0 ? share_end(blocks, share0 - 1) : 0, last = share_end(blocks, share1 - 1);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((void __attribute__((address_space(3)))*)(lds)));

    // Copies of X: chunk c of the tile is part c % 3 of its row block c / 3 (behind the last row block it again; the last chunks
    // of some wavefronts are the last one again: the same bytes at the same place).
    uint32_t xfrom[PX], xto[PX];
#pragma unroll
    for (int j = 0; j < PX; ++j) {
        const int c = min(j * TILE_WAVES + wave, XCHUNKS - 1);
        xto[j] = lds0 + c * 1024;
        xfrom[j] = static_cast<uint32_t>(min(m0 / 16 + c / 3, row_blocks - 1) * blocks) * 3072u + c % 3 * 1024 + lane * 16;
    }
    // Copies of W: chunk j is rows 8 j .. 8 j + 7 of the wavefront's, 128 bytes each; piece c of row q sits at place c ^ (q % 8).
    // A piece behind K is the row's last (times zeros).
    const int n_base = min(n0, a.N - 1), wpiece = (lane % 8) ^ (lane / 8);
    uint32_t wfrom[PW];
#pragma unroll
    for (int j = 0; j < PW; ++j)
        wfrom[j] = (static_cast<uint32_t>(min(n0 + 8 * j + lane / 8, a.N - 1) - n_base) * static_cast<uint32_t>(a.ldw) + 4 * wpiece) * 4;
    const char* const wbase = reinterpret_cast<const char*>(a.W + static_cast<int64_t>(n_base) * a.ldw);
    const uint32_t behind = static_cast<uint32_t>(min(0, a.K - 4 - ((blocks - 1) * KB + 4 * wpiece)) * 4);
    const uint32_t wto = lds0 + W0 + wave * SLOTS * WSLOT;
    const char* const wmine = lds + W0 + wave * SLOTS * WSLOT;
    // A batch of copies: the weights' values of a block, X's parts of the one before.
    const char *xsrc, *wsrc;
    uint32_t xslot, wslot, wmore;
    auto batch = [&](int bw, int sw, int sx) __attribute__((always_inline)) {
        xsrc = a.xparts + static_cast<int64_t>(min(bw - 1, last - 1)) * 3072;
        wsrc = wbase + static_cast<int64_t>(min(bw, last - 1)) * (KB * 4);
        wmore = min(bw, last - 1) == blocks - 1 ? behind : 0;
        xslot = sx * XSLOT;
        wslot = wto + sw * WSLOT;
    };
    auto copy = [&](auto number) __attribute__((always_inline)) {
        constexpr int j = decltype(number)::value;
        if constexpr (j < PW) load_to_lds(wsrc, wfrom[j] + wmore, wslot + j * 1024);
        else load_to_lds(xsrc, xfrom[j - PW], xto[j - PW] + xslot);
    };

    f32x4 acc[TN][TM], sum[ALL ? TN : 1][TM];
#pragma unroll
    for (int f = 0; f < TN; ++f)
#pragma unroll
        for (int g = 0; g < TM; ++g) {
            acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (ALL) sum[f][g] = acc[f][g];
        }
    uint32_t wp[2][TN][3][4], most[TN], top[TN];   // the weights' parts of a block and the next
    tile_bf16x8 xp[2][2][3];                       // X's parts, two tiles at a time
    f32x4 raw[TN][2];
#pragma unroll
    for (int f = 0; f < TN; ++f) most[f] = top[f] = 0;
    auto read_w = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < TN; ++f)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                raw[f][q] = *reinterpret_cast<const f32x4*>(wmine + slot * WSLOT + f * 2048 + r * 128 + ((2 * kg + q) ^ (r % 8)) * 16);
    };
    auto read_x = [&](int slot, auto pair, auto set) __attribute__((always_inline)) {
        constexpr int i = decltype(pair)::value, S = decltype(set)::value;
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int p = 0; p < 3; ++p)
                xp[S][g][p] = *reinterpret_cast<const tile_bf16x8*>(lds + slot * XSLOT + ((2 * i + g) * 3 + p) * 1024 + lane * 16);
    };
    int slot = 0;            // of block b
    // Block b, whose weights' parts are in set SET and whose first pair of X's tiles is read; `ends`: where its share ends.
    auto step = [&](auto set, int b, int ends) __attribute__((always_inline)) {
        constexpr int S = decltype(set)::value;
        const int slot1 = slot == SLOTS - 1 ? 0 : slot + 1;
        each<G>([&](auto product) __attribute__((always_inline)) {
            constexpr int p = decltype(product)::value, i = p / EACH, q = p % EACH / 4, f = p % 4 / 2, g = p % 2;
            constexpr int X = (i + S * PAIRS) & 1;
            if constexpr (p == 0) {
                read_w(slot1);
                const bool another = b + 1 == ends;      // the next block's weights are another share's
#pragma unroll
                for (int w = 0; w < TN; ++w) {
                    top[w] = another ? most[w] : top[w];
                    most[w] = another ? 0 : most[w];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (p % EACH == 0) {
                if constexpr (i + 1 < PAIRS) {
                    read_x(slot, Number<i + 1>{}, Number<X ^ 1>{});
                } else {
                    // this wavefront's copies of the next block have landed (all but the last batch) and its operands are here;
                    // behind the barrier that holds for everyone: the next block's parts of X are whole, this one's slot is free
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PC) : "memory");
                    read_x(slot1, Number<0>{}, Number<X ^ 1>{});
                    batch(b + 1 + SLOTS, slot1, slot);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const tile_bf16x8 wv = __builtin_bit_cast(tile_bf16x8, uint4{wp[S][f][w_part(q)][0], wp[S][f][w_part(q)][1], wp[S][f][w_part(q)][2], wp[S][f][w_part(q)][3]});
            acc[f][2 * i + g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xp[X][g][x_part(q)], acc[f][2 * i + g], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // a batch of copies from one barrier to the next, spread evenly
            constexpr int at = i == PAIRS - 1 ? p % EACH : p + EACH, c0 = at * PC / G, c1 = (at + 1) * PC / G;
            each<c1 - c0>([&](auto c) __attribute__((always_inline)) { copy(Number<c0 + decltype(c)::value>{}); });
            // the next block's weights, taken apart
            constexpr int STEPS = TN * SPLIT_STEPS, P0 = EACH / 4, u0 = p < P0 ? 0 : (p - P0) * STEPS / (G - P0), u1 = p < P0 ? 0 : (p - P0 + 1) * STEPS / (G - P0);
            each<u1 - u0>([&](auto u) __attribute__((always_inline)) {
                constexpr int n = u0 + decltype(u)::value;
                split_step<n % SPLIT_STEPS>(raw[n / SPLIT_STEPS], wp[S ^ 1][n / SPLIT_STEPS], most[n / SPLIT_STEPS]);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        slot = slot1;
    };

    if (first < last) {
        // before the first barrier: the weights of three blocks, X's parts of two
        each<3>([&](auto n) __attribute__((always_inline)) {
            constexpr int N = decltype(n)::value;
            batch(first + N, N, N - 1);
            each<N == 0 ? PW : PC>([&](auto j) __attribute__((always_inline)) {
                copy(j);
            });
        });
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(PC) : "memory");
        read_w(0);
        read_x(0, Number<0>{}, Number<0>{});
        each<TN * SPLIT_STEPS>([&](auto u) __attribute__((always_inline)) {
            constexpr int n = decltype(u)::value;
            split_step<n % SPLIT_STEPS>(raw[n / SPLIT_STEPS], wp[0][n / SPLIT_STEPS], most[n / SPLIT_STEPS]);
        });
        // what the last pair of a step before would have sent out (the values of the first block's weights are here)
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        batch(first + SLOTS, 0, SLOTS - 1);
        each<EACH * PC / G>([&](auto c) __attribute__((always_inline)) { copy(c); });

        int share = share0, b = first;
        while (share_end(blocks, share) <= first) ++share;
        while (b < last) {              // share after share
            const int ends = share_end(blocks, share);
#pragma unroll
            for (int f = 0; f < TN; ++f)
#pragma unroll
                for (int g = 0; g < TM; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (; b + 1 < ends; b += 2) {
                step(Number<0>{}, b, ends);
                step(Number<1>{}, b + 1, ends);
            }
            if (b < ends) {
                step(Number<0>{}, b++, ends);
#pragma unroll
                for (int f = 0; f < TN; ++f)
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int e = 0; e < 4; ++e) wp[0][f][p][e] = wp[1][f][p][e];
                if constexpr (PAIRS % 2 == 1) {
#pragma unroll
                    for (int g = 0; g < 2; ++g)
#pragma unroll
                        for (int p = 0; p < 3; ++p) xp[0][g][p] = xp[1][g][p];
                }
            }
            uint32_t xbad[TM], wbad[TN], any = 0;
#pragma unroll
            for (int g = 0; g < TM; ++g) {
                const int block = share * row_blocks + min(m0 / 16 + g, row_blocks - 1);
                any |= xbad[g] = static_cast<uint32_t>(__ballot(a.xflags[static_cast<int64_t>(block) * 16 + r] != 0)) & 0xffffu;
            }
#pragma unroll
            for (int f = 0; f < TN; ++f) {
                uint32_t m = max(top[f] & 0xffffu, top[f] >> 16);
                m = max(m, static_cast<uint32_t>(__shfl_xor(m, 16)));
                m = max(m, static_cast<uint32_t>(__shfl_xor(m, 32)));
                any |= wbad[f] = static_cast<uint32_t>(__ballot(outside(m))) & 0xffffu;
            }
            if (any != 0) {
                const int k0 = (share > 0 ? share_end(blocks, share - 1) : 0) * KB, k1 = min(ends * KB, a.K);
#pragma unroll
                for (int f = 0; f < TN; ++f)
#pragma unroll
                    for (int g = 0; g < TM; ++g)
                        if ((xbad[g] | wbad[f]) != 0)
                            replace_flagged(acc[f][g], wbad[f], xbad[g],
                                            a.A + static_cast<int64_t>(min(m0 + g * 16 + r, a.M - 1)) * a.lda,
                                            a.W + static_cast<int64_t>(min(n0 + f * 16 + r, a.N - 1)) * a.ldw, k0, k1, lane);
            }
#pragma unroll
            for (int f = 0; f < TN; ++f)
#pragma unroll
                for (int g = 0; g < TM; ++g) {
                    if constexpr (ALL) sum[f][g] += acc[f][g];
                    else store_four(a, static_cast<char*>(a.C) + share * a.part_stride * 4, m0 + g * 16 + r, n0 + f * 16 + 4 * kg, acc[f][g]);
                }
            do ++share; while (share < share1 && share_end(blocks, share) <= b);
        }
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // the last copies, which nobody reads, must not land in another's LDS
    }
    if constexpr (ALL) {
#pragma unroll
        for (int f = 0; f < TN; ++f)
#pragma unroll
            for (int g = 0; g < TM; ++g) store_four(a, static_cast<char*>(a.C), m0 + g * 16 + r, n0 + f * 16 + 4 * kg, sum[f][g]);
    }
}

template <int TM, bool ALL>
void launch_tile(SplitArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + 16 * TM - 1) / (16 * TM);
    a.tiles_n = (a.N + TILE_N - 1) / TILE_N;
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(a.tiles_m) * a.tiles_n * (ALL ? 1 : a.groups) + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_split_tile_kernel<TM, ALL>), dim3(grid), dim3(TILE_WAVES * PULSE_WAVE), 0, stream, a);
}

// Up to some hundreds of rows, without anything made of X before: a workgroup has 16 * BM rows of X and 16 * BN weight rows, its
// WAVES wavefronts a share or two of K each.  A wavefront copies its own blocks (128 bytes of eight rows an instruction: read
// straight into registers, the lanes that are served together touch sixteen rows) into two stages of its own, reads the next block
// while this one is multiplied, and takes both operands apart; no barrier until the shares meet.
template <int BM, int BN, int WAVES>
__global__ __launch_bounds__(WAVES* PULSE_WAVE) void gemm_split_staged_kernel(SplitArgs a) {
    constexpr int S = 2, T = BM + BN, TILES = BM * BN, STAGE = T * 2048, PER = SHARES / WAVES;
    constexpr int RING = WAVES * S * STAGE, MEET = SHARES * TILES * PULSE_WAVE * 16;
    __shared__ __attribute__((aligned(1024))) char lds[RING > MEET ? RING : MEET];

    // (the workgroups of a die, every eighth, take neighbouring tiles: those of one span of weight rows)
    const int total = a.tiles_m * a.tiles_n;
    const int per_die = (total + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || tile >= total) return;
    const int m0 = tile % a.tiles_m * (16 * BM), n0 = tile / a.tiles_m * (16 * BN);

    const int lane = threadIdx.x % PULSE_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int r = lane % 16, kg = lane / 16;
    const int blocks = (a.K + KB - 1) / KB, s0 = wave * PER;
    const int first = s0 > 0 ? share_end(blocks, s0 - 1) : 0, last = share_end(blocks, s0 + PER - 1);

    // Copies: half h of tile t is its rows 8 h .. 8 h + 7, 128 bytes each; piece c of row q sits at place c ^ (q % 8).  (Rows past
    // the end are the last row again, their results are not written; a piece behind K is the row's last, and zeros once read.)
    const int crow = lane / 8, cpiece = (lane % 8) ^ crow;
    const float* from[T][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < BN; ++j) from[j][h] = a.W + static_cast<int64_t>(min(n0 + 16 * j + 8 * h + crow, a.N - 1)) * a.ldw;
#pragma unroll
        for (int i = 0; i < BM; ++i) from[BN + i][h] = a.A + static_cast<int64_t>(min(m0 + 16 * i + 8 * h + crow, a.M - 1)) * a.lda;
    }
    char* const mine = lds + wave * S * STAGE;
    const uint32_t mine_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((void __attribute__((address_space(3)))*)(mine)));
    auto copy = [&](int block, int stage) __attribute__((always_inline)) {
        const int at = min(min(block, last - 1) * KB + 4 * cpiece, a.K - 4);
        const uint32_t to = __builtin_amdgcn_readfirstlane(mine_at + stage * STAGE);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) load_to_lds(from[t][h] + at, to + t * 2048 + h * 1024);
    };
    f32x4 raw[T][2];             // values 8 kg .. of a block
    auto read = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                raw[t][q] = *reinterpret_cast<const f32x4*>(mine + stage * STAGE + t * 2048 + r * 128 + ((2 * kg + q) ^ (r % 8)) * 16);
    };

    f32x4 acc[PER][BN][BM];
#pragma unroll
    for (int p = 0; p < PER; ++p)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
            for (int i = 0; i < BM; ++i) acc[p][j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    int stage = 0;               // of block b
    if (first < last) {
#pragma unroll
        for (int s = 0; s < S; ++s) copy(first + s, s);
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"((S - 1) * T * 2) : "memory");
        read(0);
    }
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int b0 = s0 + p > 0 ? share_end(blocks, s0 + p - 1) : 0, b_end = share_end(blocks, s0 + p);
        uint32_t most[T];
#pragma unroll
        for (int t = 0; t < T; ++t) most[t] = 0;
        for (int b = b0; b < b_end; ++b) {
            if ((b + 1) * KB > a.K) {                                // behind K: zeros
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if (b * KB + 8 * kg + 4 * q >= a.K) {
#pragma unroll
                        for (int t = 0; t < T; ++t) raw[t][q] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
            tile_bf16x8 parts[T][3];
#pragma unroll
            for (int t = 0; t < T; ++t) {
                uint32_t v[3][4];
                each<SPLIT_STEPS>([&](auto n) __attribute__((always_inline)) { split_step<decltype(n)::value>(raw[t], v, most[t]); });
#pragma unroll
                for (int x = 0; x < 3; ++x) parts[t][x] = __builtin_bit_cast(tile_bf16x8, uint4{v[x][0], v[x][1], v[x][2], v[x][3]});
            }
            // this block's values are in registers, so its stage is free; the next block's copies have landed
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
            copy(b + S, stage);
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"((S - 1) * T * 2) : "memory");
            stage = stage == S - 1 ? 0 : stage + 1;
            read(stage);
#pragma unroll
            for (int i = 0; i < BM; ++i)
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int j = 0; j < BN; ++j)
                        acc[p][j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(parts[j][w_part(q)], parts[BN + i][x_part(q)], acc[p][j][i], 0, 0, 0);
        }
        uint32_t bad[T], any = 0;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            uint32_t top = max(most[t] & 0xffffu, most[t] >> 16);
            top = max(top, static_cast<uint32_t>(__shfl_xor(top, 16)));
            top = max(top, static_cast<uint32_t>(__shfl_xor(top, 32)));
            any |= bad[t] = static_cast<uint32_t>(__ballot(outside(top))) & 0xffffu;
        }
        if (any != 0) {
#pragma unroll
            for (int j = 0; j < BN; ++j)
#pragma unroll
                for (int i = 0; i < BM; ++i)
                    if ((bad[j] | bad[BN + i]) != 0)
                        replace_flagged(acc[p][j][i], bad[j], bad[BN + i], a.A + static_cast<int64_t>(min(m0 + 16 * i + r, a.M - 1)) * a.lda,
                                        a.W + static_cast<int64_t>(min(n0 + 16 * j + r, a.N - 1)) * a.ldw, b0 * KB, min(b_end * KB, a.K), lane);
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory");   // the last copies, which nobody reads, must not land in what follows
    __syncthreads();

    f32x4* const meet = reinterpret_cast<f32x4*>(lds);              // [SHARES][TILES][64]
#pragma unroll
    for (int p = 0; p < PER; ++p)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
            for (int i = 0; i < BM; ++i) meet[((s0 + p) * TILES + j * BM + i) * PULSE_WAVE + lane] = acc[p][j][i];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        if (t % WAVES != wave) continue;
        f32x4 v = meet[t * PULSE_WAVE + lane];
#pragma unroll
        for (int s = 1; s < SHARES; ++s) v += meet[(s * TILES + t) * PULSE_WAVE + lane];
        store_four(a, static_cast<char*>(a.C), m0 + 16 * (t % BM) + r, n0 + 16 * (t / BM) + 4 * kg, v);
    }
}

// The shares' results added up in their order, four a thread.
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(const float* parts, int64_t part_stride, SplitArgs a) {
    const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (at >= part_stride) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(parts + at);
#pragma unroll
    for (int s = 1; s < SHARES; ++s) v += *reinterpret_cast<const f32x4*>(parts + s * part_stride + at);
    store_four(a, static_cast<char*>(a.C), static_cast<int>(at / a.N), static_cast<int>(at % a.N), v);
}

template <int BM, int BN, int WAVES>
void launch_staged(SplitArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + 16 * BM - 1) / (16 * BM);
    a.tiles_n = (a.N + 16 * BN - 1) / (16 * BN);
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(a.tiles_m) * a.tiles_n + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_split_staged_kernel<BM, BN, WAVES>), dim3(grid), dim3(WAVES * PULSE_WAVE), 0, stream, a);
}

constexpr int CHUNK = 2016;                          // rows whose parts are in scratch at a time
constexpr int64_t RESULTS_AT_MOST = 128ll << 20;     // bytes of the shares' results

int64_t parts_bytes(int M, int K) { return static_cast<int64_t>((M + 15) / 16) * ((K + KB - 1) / KB) * 3072; }
int64_t flags_bytes(int M) { return (static_cast<int64_t>((M + 15) / 16) * 16 * SHARES + 255) / 256 * 256; }

// The ways, of the least estimated time.  All give the same bits, so the choice is free; its figures are fitted to 6,900 times of 14 weights
// (128 to 12,288 long, 2,048 to 151,936 of them) at 1 to 1,024 rows, weights from memory: the way it takes is 1 % slower than
// the best one on average, 19 % at most, and 0.80 times the float32 instruction's time on average (slower by more than 3 % at 12 of
// 425 sizes, most at 49,152 x 128; 2,048 x 8,192 at one row 20.8 -> 23.3 us, 6,144 x 1,024 at 17 to 64 rows by 5 %).
// A block of k takes a lone workgroup `alone` us and a unit that is full of its kind `full` us for each SIMD's wavefront; `rate`:
// bytes a ps from memory.
struct Staged { int bm, bn, waves; double alone, full, rate; };
constexpr Staged STAGED[] = {{1, 1, 8, 0.40, 0.30, 5.82}, {1, 2, 4, 0.42, 0.47, 5.75}, {1, 2, 8, 0.49, 0.44, 5.24}, {2, 1, 8, 0.44, 0.44, 4.51},
                             {2, 2, 8, 0.62, 0.60, 4.70}, {2, 2, 4, 0.50, 0.60, 5.09}, {2, 4, 4, 0.75, 0.89, 5.20}, {3, 2, 4, 0.59, 0.78, 4.63},
                             {3, 4, 4, 0.95, 1.09, 4.99}, {4, 4, 4, 1.16, 1.27, 4.67}};
constexpr int STAGED_WAYS = sizeof(STAGED) / sizeof(STAGED[0]);
// Tiles of 96 or 64 rows by 256 weight rows, `groups` workgroups that share K.
struct Tiled { int tiles, groups; double block; };
constexpr Tiled TILED[] = {{6, 1, 1.29}, {4, 1, 1.06}, {6, 8, 1.29}, {4, 8, 1.06}, {6, 4, 1.29}, {4, 4, 1.06}};
constexpr int TILED_WAYS = sizeof(TILED) / sizeof(TILED[0]);

double larger_of(double a, double b, double c) {     // (a little more than the largest where others come near)
    a *= a; b *= b; c *= c;
    return std::sqrt(std::sqrt(a * a + b * b + c * c));
}

double staged_us(const Staged& w, int M, int N, int K, double bytes, int units) {
    const int64_t wgs = static_cast<int64_t>((M + 16 * w.bm - 1) / (16 * w.bm)) * ((N + 16 * w.bn - 1) / (16 * w.bn));
    const int64_t a_unit = (wgs + units - 1) / units;
    const int lds = std::max(w.waves * 2 * (w.bm + w.bn) * 2048, SHARES * w.bm * w.bn * 1024);
    const int together = std::min(160 * 1024 / lds, 16 / w.waves);
    const double walk = (K + KB - 1) / KB / static_cast<double>(w.waves);
    return 2.1 + larger_of(a_unit * walk * w.waves / 4 * w.full, (a_unit + together - 1) / together * (walk + 7.6) * w.alone, bytes / (w.rate * 1e6));
}

double tiled_us(const Tiled& w, int M, int N, int K, double bytes, int units) {
    const int64_t blocks = (K + KB - 1) / KB;
    const int64_t wgs = static_cast<int64_t>((M + 16 * w.tiles - 1) / (16 * w.tiles)) * ((N + TILE_N - 1) / TILE_N) * w.groups;
    double us = larger_of((wgs + units - 1) / units * ((blocks + w.groups - 1) / w.groups + 4.0) * w.block, bytes / 4.05e6, 0.);
    if (w.groups > 1) us += 2. * M * N * SHARES * 4 / 6.07e6;
    return us + 8.7 + M * (K * 4.) / 1.28e6;
}

// The number of a staged way, or STAGED_WAYS + that of tiles (`scratch`: they may be chosen; `results`: so may shares over workgroups).
int way_for(int M, int N, int K, bool scratch, bool results) {
    const double bytes = 4. * (static_cast<double>(N) * K + static_cast<double>(M) * K + static_cast<double>(M) * N);
    const int units = pulse_compute_units();
    int best = 0;
    double least = 0.;
    for (int i = 0; i < STAGED_WAYS; ++i) {
        if (i > 0 && STAGED[i].bm > std::max(1, (M + 15) / 16)) continue;
        const double us = staged_us(STAGED[i], M, N, K, bytes, units);
        if (i == 0 || us < least) { best = i; least = us; }
    }
    if (!scratch || M <= 16 || parts_bytes(M, K) >= (1ll << 32)) return best;
    for (int i = 0; i < TILED_WAYS; ++i) {
        if (TILED[i].groups > 1 && (!results || (K + KB - 1) / KB < 2 * SHARES || N % 4 != 0 ||
                                    static_cast<int64_t>(M) * N * SHARES * 4 > RESULTS_AT_MOST)) continue;
        const double us = tiled_us(TILED[i], M, N, K, bytes, units);
        if (us < least) { best = STAGED_WAYS + i; least = us; }
    }
    return best;
}

void launch_staged_way(int way, const SplitArgs& a, hipStream_t stream) {
    switch (way) {
        case 0: launch_staged<1, 1, 8>(a, stream); break;
        case 1: launch_staged<1, 2, 4>(a, stream); break;
        case 2: launch_staged<1, 2, 8>(a, stream); break;
        case 3: launch_staged<2, 1, 8>(a, stream); break;
        case 4: launch_staged<2, 2, 8>(a, stream); break;
        case 5: launch_staged<2, 2, 4>(a, stream); break;
        case 6: launch_staged<2, 4, 4>(a, stream); break;
        case 7: launch_staged<3, 2, 4>(a, stream); break;
        case 8: launch_staged<3, 4, 4>(a, stream); break;
        default: launch_staged<4, 4, 4>(a, stream); break;
    }
}

}  // namespace

// A rule of the weight alone, so that a row's sums do not depend on the batch.  Smaller products than this stay with the float32
// instruction: those of a few hundred thousand values gain nothing (1,024 x 512 at 512 / 1,024 rows 8.3 / 13.0 us there, 9.3 / 13.6
// here), and between them and this line little (2,048 x 2,048 at 12 / 97 / 200 / 333 rows 9.9 / 14.0 / 22.1 / 30.2 and 8.4 / 14.1 / 21.5 /
// 26.5), so that the line has stayed where tiles alone begin to pay (3,072 x 2,048 at 333 rows 58 and 42).
bool pulse_split_takes(int N, int K) { return static_cast<int64_t>(N) * K >= 6ll << 20; }

int64_t pulse_split_scratch(int M, int N, int K) {
    if (!pulse_split_takes(N, K)) return 0;
    M = M < CHUNK ? M : CHUNK;
    const int way = way_for(M, N, K, true, true) - STAGED_WAYS;
    if (way < 0) return 0;
    return parts_bytes(M, K) + flags_bytes(M) + (TILED[way].groups > 1 ? static_cast<int64_t>(SHARES) * M * N * 4 : 0);
}

void pulse_split_launch(const float* A, const float* W, void* C, bool c_bf16, bool c_wide, int M, int N, int K, int64_t lda, int64_t ldw,
                        int64_t ldc, void* scratch, hipStream_t stream) {
    SplitArgs a{A, W, C, c_bf16 ? 1 : 0, c_wide ? 1 : 0, M, N, K, lda, ldw, ldc, 0, 0, 1, 0, nullptr, nullptr};
    const int whole = way_for(M < CHUNK ? M : CHUNK, N, K, scratch != nullptr, true);
    if (whole < STAGED_WAYS) {
        launch_staged_way(M <= CHUNK ? whole : way_for(M, N, K, false, false), a, stream);
        return;
    }
    // (the scratch is that of the largest chunk: a way whose results it holds)
    const bool results = TILED[whole - STAGED_WAYS].groups > 1;
    for (int m = 0; m < M; m += CHUNK) {
        SplitArgs c = a;
        c.M = M - m < CHUNK ? M - m : CHUNK;
        c.A = A + static_cast<int64_t>(m) * lda;
        c.C = static_cast<char*>(C) + static_cast<int64_t>(m) * ldc * (c_bf16 ? 2 : 4);
        const int way = m == 0 ? whole : way_for(c.M, N, K, true, results);
        if (way < STAGED_WAYS) {
            launch_staged_way(way, c, stream);
            continue;
        }
        const Tiled& w = TILED[way - STAGED_WAYS];
        char* parts = static_cast<char*>(scratch);
        uint8_t* flags = reinterpret_cast<uint8_t*>(parts + parts_bytes(c.M, K));
        float* shares = reinterpret_cast<float*>(parts + parts_bytes(c.M, K) + flags_bytes(c.M));
        hipLaunchKernelGGL(gemm_split_prepare_kernel, dim3((c.M + 15) / 16, SHARES), dim3(PREPARE_WAVES * PULSE_WAVE), 0, stream, c, parts, flags);
        c.xparts = parts;
        c.xflags = flags;
        if (w.groups == 1) {
            if (w.tiles == 6) launch_tile<6, true>(c, stream);
            else launch_tile<4, true>(c, stream);
            continue;
        }
        SplitArgs p = c;
        p.C = shares;
        p.c_bf16 = 0;
        p.c_wide = 1;
        p.ldc = N;
        p.groups = w.groups;
        p.part_stride = static_cast<int64_t>(c.M) * N;
        if (w.tiles == 6) launch_tile<6, false>(p, stream);
        else launch_tile<4, false>(p, stream);
        hipLaunchKernelGGL(gemm_split_sum_kernel, dim3(static_cast<unsigned>((p.part_stride / 4 + 255) / 256)), dim3(256), 0, stream,
                           shares, p.part_stride, c);
    }
}
