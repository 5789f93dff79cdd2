// The loop of a matrix product on an output tile of WR weight rows x XR rows of X, bfloat16 operands, float32 sums:
// WN wavefronts along the weight rows by WM along the rows of X, on v_mfma_f32_32x32x16_bf16.
//
// K goes in steps of 64 through S stages of LDS for the tile's rows of W and SX for those of X (128 bytes a row), filled
// straight from memory; S - 1 steps are on their way while one is multiplied, and there is one barrier a step, before its
// last products: behind it, the next step's stages are whole, and this step's, whose operands everyone then holds, are free
// for the copies that go out between these products and the next step's.  Many stages are for what bounds a product of few
// rows, the weights' way from memory: a compute unit must have some tens of kilobytes on their way all the time (6 TB/s x
// 2 us over 256 units: 48 KB).  X comes from L2 and may have one stage less: it goes out first.
//
// The tile of the matrix instruction is D[n][m] = W . X^T: lane l holds column m = l % 32 and rows n = 8 (i / 4) +
// 4 (l / 32) + i % 4, i = 0 .. 15, of a 32 x 32 piece.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 tile_bf16x4;
typedef __attribute__((ext_vector_type(16))) float tile_f32x16;

// Where along K (of so many steps) the tiles of a block of TILE_BLOCK weight rows start.  Rows of a power of two bytes, at the
// same place in all of a launch's workgroups at a time, fall on few of the memory's channels; blocks that start elsewhere, in
// turns of five steps, spread over them.  A function of the weight's row alone, and every tile lies inside a block: a result's
// sums have one order, whatever the tile.  (All at the start -> this: 22,016 x 4,096 with SwiGLU at 70 / 97 / 128 / 256 rows 39.6 /
// 41.5 / 43.9 / 57.7 us -> 34.1 / 36.9 / 39.4 / 54.5; 64 experts of 1,024 x 2,048, 8 chosen a token, 32 / 211 tokens 150 / 168 -> 137 /
// 152.  Rows of other lengths lie on channels of their own as it is, and their blocks start together: 34,816 x 5,120 at 70 / 128
// rows 69.9 / 73.6 so, 71.0 / 75.0 in turns; 19,456 x 2,560 26.1 / 31.1 and 26.8 / 31.7.)
constexpr int TILE_BLOCK = 768;
__device__ __forceinline__ int tile_first_step(int block, int steps) { return (steps & (steps - 1)) == 0 ? (block * 5) & (steps - 1) : 0; }

template <int WR, int XR, int WN, int WM, int S, bool NT = false, int SX = S>
struct TileLoop {
    static constexpr int BK = 64;
    static constexpr int ROW_BYTES = BK * 2;
    static constexpr int STAGE_W = WR * ROW_BYTES, STAGE_X = XR * ROW_BYTES, X0 = S * STAGE_W;
    static constexpr int NW = WN * WM;
    static constexpr int TN = WR / 32 / WN, TM = XR / 32 / WM;       // 32-row pieces a wavefront
    static constexpr int PER_W = WR / 8 / NW, PER_X = XR / 8 / NW;   // chunks of 1 KB (8 rows) a wavefront copies
    static constexpr int PER = PER_W + PER_X;
    static constexpr int KK = BK / 16;                               // products of the matrix instruction's depth a step
    static constexpr int LDS = X0 + SX * STAGE_X;
    // The next products' operand reads go out between these, over the first READS of them, so that the last is here in time: a
    // lone wavefront a SIMD issues no product while it issues reads.  (All of them ahead of the products, 24,576 x 4,096 with
    // SwiGLU alone: 357 rows in tiles of 192 x 192 74 us, so 70; 509 rows in 192 x 256 91 and 86.  Inside a step, at the power
    // limit, a prompt of 509 gains 0.6 %.)  Where a step has few products the reads go ahead of them (0): behind the first they
    // are late (experts of 8 tokens in 64 x 32, a step 1 % slower).
    static constexpr int READS = TN * TM < 6 ? 0 : TN * TM == 6 ? 4 : TN * TM - 3;
    static_assert(WR % (8 * NW) == 0 && XR % (8 * NW) == 0 && TN >= 1 && TM >= 1 && SX >= 2 && S >= SX,
                  "whole chunks and pieces a wavefront");
    static_assert(TILE_BLOCK % WR == 0, "a tile lies inside a block of weight rows");

    // Piece c (16 bytes) of row r of a stage sits at place c ^ swz(r): the rows that neighbouring lanes read together then
    // lie in different places of what LDS serves at once.
    static __device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

    tile_f32x16 acc[TN][TM];

    // Row (of the tile's W for j < PER_W, else of its X) and piece that this lane brings with the wavefront's j-th chunk.
    static __device__ __forceinline__ int row_of(int j, int wave, int lane) {
        return (j < PER_W ? wave * PER_W + j : wave * PER_X + j - PER_W) * 8 + lane / 8;
    }
    static __device__ __forceinline__ int piece_of(int row, int lane) { return (lane % 8) ^ swz(row); }

    // from[j]: where that piece lies in memory at k = 0.  The walk along K starts at step `first` and goes round its end.
    __device__ __forceinline__ void run(const bf16_t* const (&from)[PER], char* lds, int wave, int lane, int K, int first = 0) {
        const int wave_n = wave % WN, wave_m = wave / WN;
        const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
            (void __attribute__((address_space(3)))*)(lds)));
        const int steps = K / BK;
        auto place = [&](int step) __attribute__((always_inline)) {      // (steps past the last: copies that nobody reads)
            const int at = min(step, steps - 1) + first;
            return (at >= steps ? at - steps : at) * BK;
        };
        // The j-th copy of a batch, X first; a batch: W of one step into its slot, X of another into its.
        auto copy = [&](int step_w, int slot_w, int step_x, int slot_x, int j) __attribute__((always_inline)) {
            if (j < PER_X) {
                load_to_lds(from[PER_W + j] + place(step_x), lds0 + X0 + slot_x * STAGE_X + (wave * PER_X + j) * 1024);
            } else {
                const bf16_t* at = from[j - PER_X] + place(step_w);
                const uint32_t to = lds0 + slot_w * STAGE_W + (wave * PER_W + j - PER_X) * 1024;
                if constexpr (NT) stream_to_lds(at, to);
                else load_to_lds(at, to);
            }
        };
        const int h = lane / 32, e = h ^ swz(lane % 32);
        int w_at[KK], x_at[KK];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int place = (e ^ (kk << 1)) * 16;
            w_at[kk] = (wave_n * TN * 32 + lane % 32) * ROW_BYTES + place;
            x_at[kk] = X0 + (wave_m * TM * 32 + lane % 32) * ROW_BYTES + place;
        }
#pragma unroll
        for (int f = 0; f < TN; ++f)
#pragma unroll
            for (int g = 0; g < TM; ++g)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[f][g][i] = 0.f;

        // The batch of step s, W of step s + S and X of step s + SX, goes out behind that step's barrier: FIRST copies of it
        // between the step's last products, the others between the next step's.
        constexpr int ALL = KK * TN * TM, FIRST = TN * TM * PER / ALL;
        constexpr int LATER = (SX - 2) * PER + (S > SX ? PER_W : 0);   // copies behind the last that the next step needs
#pragma unroll
        for (int s = -S; s < -1; ++s)
#pragma unroll
            for (int j = s + SX >= 0 ? 0 : PER_X; j < PER; ++j) copy(s + S, s + S, s + SX, s + SX, j);
#pragma unroll
        for (int j = 0; j < FIRST; ++j) copy(S - 1, S - 1, SX - 1, SX - 1, j);
        tile_bf16x8 wf[2][TN], xf[2][TM];
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(LATER + FIRST) : "memory");
#pragma unroll
        for (int g = 0; g < TM; ++g) xf[0][g] = *reinterpret_cast<const tile_bf16x8*>(lds + x_at[0] + g * 32 * ROW_BYTES);
#pragma unroll
        for (int f = 0; f < TN; ++f) wf[0][f] = *reinterpret_cast<const tile_bf16x8*>(lds + w_at[0] + f * 32 * ROW_BYTES);
        int sw = 0, sx = 0;
        for (int s = 0; s < steps; ++s) {
            const int next_w = sw == S - 1 ? 0 : sw + 1, before_w = sw == 0 ? S - 1 : sw - 1;
            const int next_x = sx == SX - 1 ? 0 : sx + 1, before_x = sx == 0 ? SX - 1 : sx - 1;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const int buf = kk & 1, then = kk == KK - 1 ? 0 : kk + 1;
                const char* const lds_w = lds + (kk == KK - 1 ? next_w : sw) * STAGE_W + w_at[then];
                const char* const lds_x = lds + (kk == KK - 1 ? next_x : sx) * STAGE_X + x_at[then];
                __builtin_amdgcn_sched_barrier(0);
                // before a step's last products: this wavefront's copies of the next step have landed and its operands are
                // here; behind the barrier that holds for everyone
                if (kk == KK - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LATER) : "memory");
                // (the operands of the products behind these, in the order in which those ask for them)
                auto read = [&](int i) __attribute__((always_inline)) {
                    if (i < TM) xf[buf ^ 1][i] = *reinterpret_cast<const tile_bf16x8*>(lds_x + i * 32 * ROW_BYTES);
                    else wf[buf ^ 1][i - TM] = *reinterpret_cast<const tile_bf16x8*>(lds_w + (i - TM) * 32 * ROW_BYTES);
                };
                if constexpr (READS == 0) {
#pragma unroll
                    for (int i = 0; i < TN + TM; ++i) read(i);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int p = 0; p < TN * TM; ++p) {
                    acc[p / TM][p % TM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[buf][p / TM], xf[buf][p % TM],
                                                                                  acc[p / TM][p % TM], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (READS > 0) {
#pragma unroll
                        for (int i = min(p, READS) * (TN + TM) / READS; i < min(p + 1, READS) * (TN + TM) / READS; ++i) read(i);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // the copies, spread evenly over the products
                    const int q = (kk == KK - 1 ? 0 : kk + 1) * TN * TM + p;
#pragma unroll
                    for (int j = q * PER / ALL; j < (q + 1) * PER / ALL; ++j) {
                        if (kk == KK - 1) copy(s + S, sw, s + SX, sx, j);
                        else copy(s + S - 1, before_w, s + SX - 1, before_x, j);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            sw = next_w, sx = next_x;
        }
        // the last copies, which nobody reads, must not land in what follows
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
    }
};

// A wavefront's own order of what it writes to and reads from LDS.
__device__ __forceinline__ void tile_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
