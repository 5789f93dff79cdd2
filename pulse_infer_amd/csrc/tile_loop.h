// The loop of a matrix product on an output tile of WR weight rows x XR rows of X, bfloat16 operands, float32 sums:
// WN wavefronts along the weight rows by WM along the rows of X, on v_mfma_f32_16x16x32_bf16.
//
// K goes in steps of 64 through S stages of LDS for the tile's rows of W and SX for those of X (128 bytes a row), filled
// straight from memory; S - 1 steps are on their way while one is multiplied, and there is one barrier a step, before its
// last products: behind it, the next step's stages are whole, and this step's, whose operands everyone then holds, are free
// for the copies that go out between these products and the next step's.  Many stages are for what bounds a product of few
// rows, the weights' way from memory: a compute unit must have some tens of kilobytes on their way all the time (6 TB/s x
// 2 us over 256 units: 48 KB).  X comes from L2 and may have one stage less: it goes out first.
//
// The tile of the matrix instruction is D[n][m] = W . X^T: lane l holds column m = l % 16 and rows n = 4 (l / 16) + i, i = 0 .. 3, of
// a 16 x 16 piece.
//
// The instruction: from some 300 rows on a product takes what the card's power allows, and v_mfma_f32_16x16x32_bf16 reads and writes half
// as many sums a product as v_mfma_f32_32x32x16_bf16, on which this loop ran before: 2,048 rows of 24,576 x 4,096 with SwiGLU in tiles
// of 256 x 256 314 -> 282 us (with operands of zeros, which cost little power, 227 and 224), 509 rows in 192 x 256 84 -> 81.
// Neighbouring products share an operand (two rows of X's pieces in turns): 285 -> 281 us against one row after the other.
//
// The copies: a base in scalar registers, which moves along K, and a lane's byte offset from it, which does not; a wavefront's eight
// chunks of 1 KB lie in a row in LDS and are told apart by the instruction's own offset, so a copy is one instruction in the loop (with a
// pointer a lane and M0 set for each, six: 324 -> 306 us at 2,048 rows, 85 -> 81 at 357 in 192 x 256, before the other instruction).
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 tile_bf16x4;
typedef __attribute__((ext_vector_type(4))) float tile_f32x4;

// Where along K (of so many steps) the tiles of a block of TILE_BLOCK weight rows start.  Rows of a power of two bytes, at the
// same place in all of a launch's workgroups at a time, fall on few of the memory's channels; blocks that start elsewhere, in
// turns of five steps, spread over them.  A function of the weight's row alone, and every tile lies inside a block: a result's
// sums have one order, whatever the tile.  (All at the start -> this: 22,016 x 4,096 with SwiGLU at 70 / 97 / 128 / 256 rows 39.6 /
// 41.5 / 43.9 / 57.7 us -> 34.1 / 36.9 / 39.4 / 54.5; 64 experts of 1,024 x 2,048, 8 chosen a token, 32 / 211 tokens 150 / 168 -> 137 /
// 152.  Rows of other lengths lie on channels of their own as it is, and their blocks start together: 34,816 x 5,120 at 70 / 128
// rows 69.9 / 73.6 so, 71.0 / 75.0 in turns; 19,456 x 2,560 26.1 / 31.1 and 26.8 / 31.7.)
constexpr int TILE_BLOCK = 768;
__device__ __forceinline__ int tile_first_step(int block, int steps) { return (steps & (steps - 1)) == 0 ? (block * 5) & (steps - 1) : 0; }

// FAR: rows further than 4 GB from their base (a pointer a lane, as slow as that is).
template <int WR, int XR, int WN, int WM, int S, bool NT = false, int SX = S, bool FAR = false>
struct TileLoop {
    static constexpr int BK = 64;
    static constexpr int ROW_BYTES = BK * 2;
    static constexpr int STAGE_W = WR * ROW_BYTES, STAGE_X = XR * ROW_BYTES, X0 = S * STAGE_W;
    static constexpr int NW = WN * WM;
    static constexpr int TN = WR / 16 / WN, TM = XR / 16 / WM;       // 16-row pieces a wavefront
    static constexpr int PER_W = WR / 8 / NW, PER_X = XR / 8 / NW;   // chunks of 1 KB (8 rows) a wavefront copies
    static constexpr int PER = PER_W + PER_X;
    static constexpr int KK = BK / 32;                               // products of the matrix instruction's depth a step
    static constexpr int P = TN * TM, ALL = KK * P;                  // products a depth, and a step
    static constexpr int LDS = X0 + SX * STAGE_X;
    // The next products' operand reads go out between these, over the first READS of them, so that the last is here in time: a
    // lone wavefront a SIMD issues no product while it issues reads.  (Ahead of the products, o of 4,096 x 4,096 in shares in tiles of
    // 128 x 128: 14.3 -> 15.7 us at 192 rows, 20.4 -> 22.5 at 400; 128 x 64 at 150 rows 18.5 -> 18.9.)  Where a step has four products a
    // wavefront the reads go ahead of them (0): behind the first they are late (experts of 8 tokens in 64 x 32, a step 1 % slower).
    static constexpr int READS = P < 8 ? 0 : P * 3 / 4;
    static_assert(WR % (8 * NW) == 0 && XR % (8 * NW) == 0 && TN >= 1 && TM % 2 == 0 && SX >= 2 && S >= SX,
                  "whole chunks and pieces a wavefront");
    static_assert(TILE_BLOCK % WR == 0, "a tile lies inside a block of weight rows");

    // Piece c (16 bytes) of row r of a stage sits at place c ^ swz(r): the rows that neighbouring lanes read together then
    // lie in different places of what LDS serves at once.
    static __device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

    tile_f32x4 acc[TN][TM];

    // Row (of the tile's W for j < PER_W, else of its X) and piece that this lane brings with the wavefront's j-th chunk.
    static __device__ __forceinline__ int row_of(int j, int wave, int lane) {
        return (j < PER_W ? wave * PER_W + j : wave * PER_X + j - PER_W) * 8 + lane / 8;
    }
    static __device__ __forceinline__ int piece_of(int row, int lane) { return (lane % 8) ^ swz(row); }

    // A lane's offset for its j-th chunk from that piece's place in memory at k = 0, in values from the chunk's base.  (Less what the
    // copy's instruction adds, which moves both the place in LDS and the one in memory; BACK keeps it from below zero.)
    typedef std::conditional_t<FAR, uint64_t, uint32_t> Offset;
    static constexpr int BACK = FAR ? 0 : 3072;
    static constexpr int inside(int j) { return FAR ? 0 : ((j < PER_W ? j : j - PER_W) % 8 - 4) * 1024; }
    static __device__ __forceinline__ Offset offset_of(int j, int64_t values) { return static_cast<Offset>(values * 2 + BACK - inside(j)); }

    // base(j): where the wavefront's j-th chunk counts its offsets from, the same for all lanes.  The walk along K starts at step
    // `first` and goes round its end.
    template <typename Base>
    __device__ __forceinline__ void run(Base&& base, const Offset (&from)[PER], char* lds, int wave, int lane, int K, int first = 0) {
        const int wave_n = wave % WN, wave_m = wave / WN;
        const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
            (void __attribute__((address_space(3)))*)(lds)));
        const int steps = K / BK;
        auto place = [&](int step) __attribute__((always_inline)) {      // (steps past the last: copies that nobody reads)
            const int at = min(step, steps - 1) + first;
            return (at >= steps ? at - steps : at) * ROW_BYTES;
        };
        // The batch of step s, W of step s + S and X of step s + SX, goes out behind that step's barrier: FIRST copies of it
        // between the step's last products, the others between the next step's.
        constexpr int FIRST = P * PER / ALL;
        constexpr int LATER = (SX - 2) * PER + (S > SX ? PER_W : 0);   // copies behind the last that the next step needs
        // The j-th copy of a batch, X first; a batch: W of one step into its slot, X of another into its.
        auto copy = [&](int step_w, int slot_w, int step_x, int slot_x, auto jc) __attribute__((always_inline)) {
            constexpr int j = jc;
            constexpr bool is_x = j < PER_X;
            constexpr int i = is_x ? j : j - PER_X, c = is_x ? PER_W + j : j - PER_X;
            const Offset off = from[c];
            const char* at = reinterpret_cast<const char*>(base(c)) - BACK + place(is_x ? step_x : step_w);
            const uint32_t to = lds0 + (is_x ? X0 + slot_x * STAGE_X + wave * PER_X * 1024 : slot_w * STAGE_W + wave * PER_W * 1024);
            if constexpr (FAR) {
                if constexpr (NT && !is_x) stream_to_lds(at + off, to + i * 1024);
                else load_to_lds(at + off, to + i * 1024);
            } else {
                if constexpr (i % 8 == 0 || j == FIRST) lds_place(to + (i / 8 * 8 + 4) * 1024);
                copy_to_place<inside(c), NT && !is_x>(at, off);
            }
        };
        const int h = lane / 16, e = h ^ swz(lane % 16);
        int w_at[KK], x_at[KK];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int piece = (e ^ (kk << 2)) * 16;
            w_at[kk] = (wave_n * TN * 16 + lane % 16) * ROW_BYTES + piece;
            x_at[kk] = X0 + (wave_m * TM * 16 + lane % 16) * ROW_BYTES + piece;
        }
#pragma unroll
        for (int f = 0; f < TN; ++f)
#pragma unroll
            for (int g = 0; g < TM; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[f][g][i] = 0.f;

        each<S - 1>([&](auto sc) __attribute__((always_inline)) {
            constexpr int s = sc - S;
            each<PER>([&](auto j) __attribute__((always_inline)) {
                if constexpr (s + SX >= 0 || j >= PER_X) copy(s + S, s + S, s + SX, s + SX, j);
            });
        });
        each<FIRST>([&](auto j) __attribute__((always_inline)) { copy(S - 1, S - 1, SX - 1, SX - 1, j); });
        tile_bf16x8 wf[2][TN], xf[2][TM];
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(LATER + FIRST) : "memory");
#pragma unroll
        for (int g = 0; g < TM; ++g) xf[0][g] = *reinterpret_cast<const tile_bf16x8*>(lds + x_at[0] + g * 16 * ROW_BYTES);
#pragma unroll
        for (int f = 0; f < TN; ++f) wf[0][f] = *reinterpret_cast<const tile_bf16x8*>(lds + w_at[0] + f * 16 * ROW_BYTES);
        int sw = 0, sx = 0;
        for (int s = 0; s < steps; ++s) {
            const int next_w = sw == S - 1 ? 0 : sw + 1, before_w = sw == 0 ? S - 1 : sw - 1;
            const int next_x = sx == SX - 1 ? 0 : sx + 1, before_x = sx == 0 ? SX - 1 : sx - 1;
            each<KK>([&](auto kc) __attribute__((always_inline)) {
                constexpr int kk = kc, buf = kk & 1, then = kk == KK - 1 ? 0 : kk + 1;
                const char* const lds_w = lds + (kk == KK - 1 ? next_w : sw) * STAGE_W + w_at[then];
                const char* const lds_x = lds + (kk == KK - 1 ? next_x : sx) * STAGE_X + x_at[then];
                __builtin_amdgcn_sched_barrier(0);
                // before a step's last products: this wavefront's copies of the next step have landed and its operands are
                // here; behind the barrier that holds for everyone
                if constexpr (kk == KK - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LATER) : "memory");
                // (the operands of the products behind these)
                auto read = [&](int i) __attribute__((always_inline)) {
                    if (i < TM) xf[buf ^ 1][i] = *reinterpret_cast<const tile_bf16x8*>(lds_x + i * 16 * ROW_BYTES);
                    else wf[buf ^ 1][i - TM] = *reinterpret_cast<const tile_bf16x8*>(lds_w + (i - TM) * 16 * ROW_BYTES);
                };
                if constexpr (READS == 0) {
#pragma unroll
                    for (int i = 0; i < TN + TM; ++i) read(i);
                }
                __builtin_amdgcn_sched_barrier(0);
                each<P>([&](auto pc) __attribute__((always_inline)) {
                    // two pieces of X in turns along the pieces of W, and back with the next two
                    constexpr int p = pc, pair = p / (2 * TN), f = p % (2 * TN) / 2, g = 2 * pair + (p % 2 ^ f % 2), n = pair % 2 ? TN - 1 - f : f;
                    acc[n][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[buf][n], xf[buf][g], acc[n][g], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (READS > 0) {
                        constexpr int from_i = (p < READS ? p : READS) * (TN + TM) / READS, to_i = (p + 1 < READS ? p + 1 : READS) * (TN + TM) / READS;
#pragma unroll
                        for (int i = from_i; i < to_i; ++i) read(i);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // the copies, spread evenly over the products
                    constexpr int q = (kk == KK - 1 ? 0 : kk + 1) * P + p;
                    each<(q + 1) * PER / ALL - q * PER / ALL>([&](auto jc) __attribute__((always_inline)) {
                        constexpr std::integral_constant<int, q * PER / ALL + jc> j{};
                        if constexpr (kk == KK - 1) copy(s + S, sw, s + SX, sx, j);
                        else copy(s + S - 1, before_w, s + SX - 1, before_x, j);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            sw = next_w, sx = next_x;
        }
        // the sums stay in the registers they are made in up to here (where their stores want them elsewhere, the compiler moved them in the loop)
#pragma unroll
        for (int f = 0; f < TN; ++f)
#pragma unroll
            for (int g = 0; g < TM; ++g) {
                if constexpr (P >= 12) asm volatile("" : "+a"(acc[f][g]));
                else asm volatile("" : "+v"(acc[f][g]));
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
