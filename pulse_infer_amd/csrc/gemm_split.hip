// C[M, N] = A[M, K] * W[N, K]^T of float32 operands on the bfloat16 matrix instruction, no less exact than on the float32 one.
// (reference: cublasSgemm, src/ops/kernels/cuda/matmul_kernel.cu:70-88)
//
// A float32 value is the sum of three bfloat16 parts, exactly: the value rounded, what that leaves rounded, the rest (8 + 8 + 8
// bits).  Of the nine products of two values' parts the six largest are made (second x second and third x third and the like
// below: at most 2^-26 of the product are left out, a quarter of a float32 rounding), each exact, on v_mfma_f32_16x16x32_bf16
// with float32 sums.  That instruction does sixteen times the arithmetic of v_mfma_f32_16x16x4_f32, so six of it take 3/8 of the
// time.  Error against 64 bits, relative, normal operands, K of 2,048 / 8,192: 2.4e-7 / 5.1e-7, the float32 instruction with
// four shares of K 4.1e-7 / 8.1e-7; largest difference over the result's root mean square 1.7e-6 / 3.1e-6 against 3.3e-6 /
// 6e-6; positive operands, and operands whose sizes spread over e^3, likewise smaller.
//
// The order: K is cut into blocks of 32 and the blocks into eight shares.  A share is added up block after block, in a block
// product after product as `w_part` and `x_part` say, and the shares in their order.  The cut depends on K alone and every way
// below does the same, so a row's result does not depend on what else is in the batch, bit for bit.
//
// Range: parts are as exact as said for rows (of a share) whose largest value is at least 2^-100 and below 2^60, or that are
// zeros.  Any other row, one with an infinity or NaN among them, is flagged, and results of flagged rows are made anew on the
// float32 instruction (`replace_flagged`): products of parts would overflow, or make a NaN of an infinity times zero.
//
// Ways: few rows straight from memory into registers (gemm_split_rows_kernel); from there on X is taken apart once
// (gemm_split_prepare_kernel) and multiplied in tiles of up to 96 x 256, whose wavefronts take the weights apart as they go
// (gemm_split_tile_kernel), K in one go or its shares over workgroups, added up by gemm_split_sum_kernel.
// What bounds the tiles: 333 x 16,384 x 2,048 takes 125 us, its matrix instructions alone 91 (the power limit: 1.47 PFLOP/s);
// the difference is the issue of the weights' arithmetic, 104 instructions a wavefront and block beside 72 products.  Two
// wavefronts a SIMD are what hides it: with one, 160 us.  Taking X apart in the tiles, as its weights, 146 to 160.
// Measured, weight rows x K, us, float32 instruction -> parts:
//                        12 rows       32           64           97           200           333           1,024
//   16,384 x 2,048       54 -> 50      56 -> 56     62 -> 71     84 -> 81     155 -> 100    237 -> 123    602 -> 340
//   3,072 x 2,048        13 -> 14      18 -> 17     19 -> 22     26 -> 29     35 -> 41      60 -> 48
//   2,048 x 8,192        38 -> 37      64 -> 40     62 -> 43     55 -> 48     83 -> 65      110 -> 79     264 -> 205
// (At 40 to 200 rows the smallest of these lose by the two kernels beside the tiles what the others of a layer gain; a choice by
// the rows would make a row's sums depend on the batch.)
#include "gemm_split.h"
#include "tile_loop.h"
#include <algorithm>

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

// Few rows, where the weights' way from memory is the time: a workgroup has 16 * BM rows of X and 16 * BN weight rows, its
// wavefronts a share of K each, straight from memory into registers, U blocks a set, the next set on its way.
template <int BM, int BN, int U>
__global__ __launch_bounds__(SHARES* PULSE_WAVE) void gemm_split_rows_kernel(SplitArgs a) {
    constexpr int T = BM + BN;
    __shared__ f32x4 meet[SHARES][BN * BM][PULSE_WAVE];
    const int n0 = blockIdx.x * (16 * BN), m0 = blockIdx.y * (16 * BM);
    const int lane = threadIdx.x % PULSE_WAVE;
    const int share = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int r = lane % 16, kg = lane / 16;
    const int blocks = (a.K + KB - 1) / KB;
    const int b0 = share > 0 ? share_end(blocks, share - 1) : 0, b_end = share_end(blocks, share);

    // (rows past the end are the last row again: their results are not written)
    const float* row[T];
#pragma unroll
    for (int j = 0; j < BN; ++j) row[j] = a.W + static_cast<int64_t>(min(n0 + 16 * j + r, a.N - 1)) * a.ldw;
#pragma unroll
    for (int i = 0; i < BM; ++i) row[BN + i] = a.A + static_cast<int64_t>(min(m0 + 16 * i + r, a.M - 1)) * a.lda;

    f32x4 acc[BN][BM];
    uint32_t most[T];
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
        for (int i = 0; i < BM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < T; ++j) most[j] = 0;

    f32x4 raw[2][U][T][2];       // values 8 kg .. of a block
    auto fetch = [&](int set, int block) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < T; ++j) raw[set][u][j][q] = load4(row[j], (block + u) * KB + 8 * kg + 4 * q, a.K);
        __builtin_amdgcn_sched_barrier(0);   // (the loads stay ahead of the products that they hide behind)
    };
    auto multiply = [&](int set, int block) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (block + u >= b_end) continue;
            if ((block + u + 1) * KB > a.K) {                    // behind K: zeros
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if ((block + u) * KB + 8 * kg + 4 * q >= a.K) {
#pragma unroll
                        for (int j = 0; j < T; ++j) raw[set][u][j][q] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
            tile_bf16x8 parts[T][3];
#pragma unroll
            for (int j = 0; j < T; ++j) {
                uint32_t v[3][4];
                each<SPLIT_STEPS>([&](auto n) __attribute__((always_inline)) { split_step<decltype(n)::value>(raw[set][u][j], v, most[j]); });
#pragma unroll
                for (int p = 0; p < 3; ++p) parts[j][p] = __builtin_bit_cast(tile_bf16x8, uint4{v[p][0], v[p][1], v[p][2], v[p][3]});
            }
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < BN; ++j)
#pragma unroll
                    for (int i = 0; i < BM; ++i)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(parts[j][w_part(q)], parts[BN + i][x_part(q)], acc[j][i], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch(0, b0);
    for (int b = b0; b < b_end; b += 2 * U) {
        fetch(1, b + U);
        multiply(0, b);
        fetch(0, b + 2 * U);
        multiply(1, b + U);
    }

    uint32_t bad[T];
#pragma unroll
    for (int j = 0; j < T; ++j) {
        u16x2 top = __builtin_bit_cast(u16x2, most[j]);
#pragma unroll
        for (int x = 16; x <= 32; x *= 2) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, __shfl_xor(__builtin_bit_cast(uint32_t, top), x)));
        bad[j] = static_cast<uint32_t>(__ballot(outside(__builtin_bit_cast(uint32_t, top)))) & 0xffffu;
    }
#pragma unroll
    for (int j = 0; j < BN; ++j)
#pragma unroll
        for (int i = 0; i < BM; ++i) {
            if ((bad[j] | bad[BN + i]) != 0) replace_flagged(acc[j][i], bad[j], bad[BN + i], row[BN + i], row[j], b0 * KB, min(b_end * KB, a.K), lane);
            meet[share][j * BM + i][lane] = acc[j][i];
        }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < BN * BM; ++t) {
        if (t % SHARES != share) continue;
        f32x4 v = meet[0][t][lane];
#pragma unroll
        for (int s = 1; s < SHARES; ++s) v += meet[s][t][lane];
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

template <int BM, int BN, int U>
void launch_rows(const SplitArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL((gemm_split_rows_kernel<BM, BN, U>), dim3((a.N + 16 * BN - 1) / (16 * BN), (a.M + 16 * BM - 1) / (16 * BM)),
                       dim3(SHARES * PULSE_WAVE), 0, stream, a);
}

struct Way { int tiles, groups; double block; };    // tiles of 16 rows a workgroup, workgroups that share K, ns a block of k
constexpr Way WAYS[] = {{6, 1, 1900.}, {4, 1, 1450.}, {2, 1, 1050.}, {6, 8, 1900.}, {4, 8, 1450.}, {2, 8, 1050.},
                        {6, 4, 1900.}, {4, 4, 1450.}, {2, 4, 1050.}};
constexpr int CHUNK = 2016;                          // rows whose parts are in scratch at a time
constexpr int64_t RESULTS_AT_MOST = 128ll << 20;     // bytes of the shares' results

int64_t parts_bytes(int M, int K) { return static_cast<int64_t>((M + 15) / 16) * ((K + KB - 1) / KB) * 3072; }
int64_t flags_bytes(int M) { return (static_cast<int64_t>((M + 15) / 16) * 16 * SHARES + 255) / 256 * 256; }

// The tiles of the least estimated time: rounds of workgroups x blocks of k (three more for a workgroup's start) x the time of
// one, as measured with the chip full; shares over workgroups cost the second kernel and their results' way to memory and back.
int way_for(int M, int N, int K) {
    const int64_t units = pulse_compute_units(), blocks = (K + KB - 1) / KB;
    int best = 0;
    double least = 0.0;
    for (int i = 0; i < 9; ++i) {
        const Way& w = WAYS[i];
        const int64_t results = static_cast<int64_t>(M) * N * SHARES * 4;
        if (w.groups > 1 && (blocks < 2 * SHARES || N % 4 != 0 || results > RESULTS_AT_MOST)) continue;
        const int64_t wgs = static_cast<int64_t>((M + 16 * w.tiles - 1) / (16 * w.tiles)) * ((N + TILE_N - 1) / TILE_N) * w.groups;
        double cost = ((wgs + units - 1) / units) * ((blocks + w.groups - 1) / w.groups + 3) * w.block;
        if (w.groups > 1) cost += 3000. + 2 * results / 4500.;
        if (i == 0 || cost < least) { best = i; least = cost; }
    }
    return best;
}

// Few rows, whose weights go straight into registers: always up to 16; up to 32 of a weight of many rows (16,384 x 2,048 at 32
// rows 56 us, tiles 65); more where the workgroups of 32 rows by 16 or 32 weight rows find a compute unit each and K is short
// (3,072 x 2,048 at 64 rows 22 us, tiles 25; but 2,048 x 8,192 52 us, tiles 43).
// Weight rows a workgroup (in sixteens) of this way, or 0: tiles.
int rows_way_for(int M, int N, int K) {
    const int64_t units = pulse_compute_units();
    if (M <= 16) return N >= 64 * units ? 4 : 1;
    if (M <= 32 && N >= 64 * units) return 4;
    if (K >= 4096) return 0;
    for (int bn = 1; bn <= 2; ++bn)
        if (static_cast<int64_t>((M + 31) / 32) * ((N + 16 * bn - 1) / (16 * bn)) <= units) return bn;
    return 0;
}

}  // namespace

// A rule of the weight alone, so that a row's sums do not depend on the batch.  Smaller products than this stay with the float32
// instruction: the kernels beside the tiles cost what the tiles gain (2,048 x 2,048 at 97 / 333 rows 18 / 33 us there, 22 / 35
// here; 1,024 x 512 at 300 rows 11 against 14; 3,072 x 2,048, the first that is made here, 26 against 29 and 60 against 48).
bool pulse_split_takes(int N, int K) { return static_cast<int64_t>(N) * K >= 6ll << 20; }

int64_t pulse_split_scratch(int M, int N, int K) {
    if (!pulse_split_takes(N, K)) return 0;
    M = M < CHUNK ? M : CHUNK;
    if (rows_way_for(M, N, K) != 0 || parts_bytes(M, K) >= (1ll << 32)) return 0;
    return parts_bytes(M, K) + flags_bytes(M) + (WAYS[way_for(M, N, K)].groups > 1 ? static_cast<int64_t>(SHARES) * M * N * 4 : 0);
}

void pulse_split_launch(const float* A, const float* W, void* C, bool c_bf16, bool c_wide, int M, int N, int K, int64_t lda, int64_t ldw,
                        int64_t ldc, void* scratch, int way, hipStream_t stream) {
    SplitArgs a{A, W, C, c_bf16 ? 1 : 0, c_wide ? 1 : 0, M, N, K, lda, ldw, ldc, 0, 0, 1, 0, nullptr, nullptr};
    if (scratch == nullptr || (way < 0 && pulse_split_scratch(M, N, K) == 0)) {
        const int bn = rows_way_for(M, N, K);
        if (M <= 16) {
            if (bn == 4) launch_rows<1, 4, 1>(a, stream);
            else if (K >= 4096) launch_rows<1, 1, 4>(a, stream);    // (2,048 x 8,192 at 12 rows 37 us against 40 with two blocks a set,
            else launch_rows<1, 1, 2>(a, stream);                   //  3,072 x 2,048 14.7 against 13.6)
        } else if (bn == 4) {
            launch_rows<2, 4, 1>(a, stream);
        } else if (bn == 2) {
            launch_rows<2, 2, 1>(a, stream);
        } else if (bn == 1) {
            launch_rows<2, 1, 1>(a, stream);
        } else {
            launch_rows<4, 2, 1>(a, stream);                        // (no scratch was given)
        }
        return;
    }
    for (int m = 0; m < M; m += CHUNK) {
        SplitArgs c = a;
        c.M = M - m < CHUNK ? M - m : CHUNK;
        c.A = A + static_cast<int64_t>(m) * lda;
        c.C = static_cast<char*>(C) + static_cast<int64_t>(m) * ldc * (c_bf16 ? 2 : 4);
        // (the scratch is that of the largest chunk: a way whose results it holds)
        const int which = way >= 0 ? way : m == 0 ? way_for(c.M, N, K) : WAYS[way_for(CHUNK, N, K)].groups > 1 ? way_for(c.M, N, K) : way_for(CHUNK, N, K);
        char* parts = static_cast<char*>(scratch);
        uint8_t* flags = reinterpret_cast<uint8_t*>(parts + parts_bytes(c.M, K));
        float* results = reinterpret_cast<float*>(parts + parts_bytes(c.M, K) + flags_bytes(c.M));
        hipLaunchKernelGGL(gemm_split_prepare_kernel, dim3((c.M + 15) / 16, SHARES), dim3(PREPARE_WAVES * PULSE_WAVE), 0, stream, c, parts, flags);
        c.xparts = parts;
        c.xflags = flags;
        SplitArgs p = c;
        p.C = results;
        p.c_bf16 = 0;
        p.c_wide = 1;
        p.ldc = N;
        p.groups = WAYS[which].groups;
        p.part_stride = static_cast<int64_t>(c.M) * N;
        if (which == 0) launch_tile<6, true>(c, stream);
        else if (which == 1) launch_tile<4, true>(c, stream);
        else if (which == 2) launch_tile<2, true>(c, stream);
        else if (WAYS[which].tiles == 6) launch_tile<6, false>(p, stream);
        else if (WAYS[which].tiles == 4) launch_tile<4, false>(p, stream);
        else launch_tile<2, false>(p, stream);
        if (WAYS[which].groups > 1)
            hipLaunchKernelGGL(gemm_split_sum_kernel, dim3(static_cast<unsigned>((p.part_stride / 4 + 255) / 256)), dim3(256), 0, stream,
                               results, p.part_stride, c);
    }
}
