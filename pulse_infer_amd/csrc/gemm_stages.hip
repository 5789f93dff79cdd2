// C[M, N] = X[M, K] W[N, K]^T for some tens to some hundreds of rows (short prompts, portions beside decoded tokens):
// bfloat16 operands, float32 sums on the matrix cores, on the loop of tile_loop.h.
// (reference: cuBLAS for every product, src/ops/kernels/cuda/matmul_kernel.cu:132-154)
//
// What bounds it: the bytes that the fullest compute unit copies into LDS.  A unit takes in 29 to 55 bytes a nanosecond over a
// launch, least where they are weights that come from memory, and the matrix cores are busy for 13 to 50 % of it, LDS waits
// make 3 to 7 % (counters at 97, 357 and 509 rows; from 300 rows on the power limit comes near: 357 rows of gate + up take 58 us with
// operands of zeros, 62 to 65 with others, 2,048 rows 224 and 284), so the shape and the shares of K are chosen for the least bytes
// (`plan_for`).  Measured alone with weights from memory, us, against the vendor library's product (gate and up: with its
// pass for SwiGLU behind it) and this package's shared-out product for up to 192 rows; in brackets behind a figure, what it
// takes inside a step, between other kernels and with the chip warm:
//                                   97 rows              192                  357                 509
//   gate + up, 24,576 x 4,096       38 [38]              53                   66 [68]             84 [88]
//     library                       54                   64                   84                  96
//   qkv, 6,144 x 4,096              19 [20]              26                   32 [33]             35 [35]
//     library                       25                   36                   41                  42
//   o, 4,096 x 4,096, shares        12 [14]              14                   21 [24]             24 [26]
//     library / shared out          25 / 16              37 / 21              29                  32
//   down, 4,096 x 12,288, shares    24 [25]              31                   39 [43]             52 [55]
//     library / shared out          44 / 34              92 / 47              52, shared [46]     59, shared [60]
// (2,048 rows, inside a step, against the library's: gate + up 284 to 316 for 278 + 30, down in two shares 142 to 158, o 61 to 66, qkv 77 to
// 84 for its 84; 8,192 rows of gate + up 1,095 to 1,130, 1.46 to 1.51 PFLOP/s.  Cards differ by a tenth.)
// From some 260 rows on tiles of 192 or 256 rows of X (their weights through three stages, X, which comes from L2, through
// two where LDS holds no third) take the place of the library's: 357 rows of gate + up ran 96 us in tiles of 192 x 128.
// Steps of 32 of K in twice the stages, the other way to fit such tiles, bring 64 bytes of a row at a time, which a unit
// takes in at half the rate (192 x 256: 107 us).
// Weights are read past the caches (nontemporal) by tiles of up to 128 rows of X: 5 % where they are the time; the larger
// tiles, whose weights are read by several, lose 2 % by it.
#include "common.h"
#include "tile_loop.h"
#include <algorithm>

namespace {

enum { OUT_BF16 = 0, OUT_SWIGLU = 1, OUT_F32 = 2 };

struct StageArgs {
    const bf16_t* X;
    int64_t ldx;
    const bf16_t* W;
    int64_t ldw;
    void* C;
    int64_t ldc;
    int M, N, K;          // K: of one share
    int tiles_m, tiles_n;
    int splits;           // shares of K, each with a float32 result of its own
    int64_t part_stride;  // elements between the shares' results
};

constexpr int PANEL = 8;  // tiles of rows a panel of the tile order

template <int MODE, int WR, int XR, int WN, int WM, int S, int SX, bool NT, bool FAR>
__global__ __launch_bounds__(256) void gemm_stages_kernel(StageArgs a) {
    using Loop = TileLoop<WR, XR, WN, WM, S, NT, SX, FAR>;
    __shared__ __attribute__((aligned(1024))) char lds[Loop::LDS];

    // The workgroups of a die (every eighth) take neighbouring tiles, in panels of eight tiles of rows, which share
    // their operands in that die's L2; a share of K is a whole set of tiles.
    const int tiles = a.tiles_m * a.tiles_n, total = tiles * a.splits;
    const int per_die = (total + 7) / 8;
    const int t_all = (blockIdx.x % 8) * per_die + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per_die || t_all >= total) return;
    const int split = t_all / tiles, t = t_all - split * tiles;
    const int panel = t / (PANEL * a.tiles_n);
    const int panel_m = min(PANEL, a.tiles_m - panel * PANEL);
    const int in_panel = t - panel * PANEL * a.tiles_n;
    const int m0 = (panel * PANEL + in_panel % panel_m) * XR, n0 = in_panel / panel_m * WR;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int lane = threadIdx.x % PULSE_WAVE;
    const int64_t k0 = static_cast<int64_t>(split) * a.K;
    typename Loop::Offset from[Loop::PER];       // (rows past an operand's end are its last row: their results are not written)
#pragma unroll
    for (int j = 0; j < Loop::PER; ++j) {
        const int row = Loop::row_of(j, wave, lane);
        const int64_t at = j < Loop::PER_W ? min(row, a.N - 1 - n0) * a.ldw : min(row, a.M - 1 - m0) * a.ldx;
        from[j] = Loop::offset_of(j, at + Loop::piece_of(row, lane) * 8);
    }
    const bf16_t* const w_rows = a.W + n0 * a.ldw + k0;
    const bf16_t* const x_rows = a.X + m0 * a.ldx + k0;
    Loop loop;
    loop.run([&](int j) __attribute__((always_inline)) { return j < Loop::PER_W ? w_rows : x_rows; }, from, lds, wave, lane, a.K,
             MODE == OUT_SWIGLU ? tile_first_step(n0 / TILE_BLOCK, a.K / Loop::BK) : 0);

    // Results leave through LDS, a wavefront's 32 rows at a time, in whole 16-byte pieces of rows.
    constexpr int TN = Loop::TN, TM = Loop::TM;
    constexpr int SIZE = MODE == OUT_F32 ? 4 : 2;
    constexpr int COLS = TN * (MODE == OUT_SWIGLU ? 8 : 16), PITCH = COLS * SIZE + 16, PCS = COLS * SIZE / 16;
    constexpr int WAVE_LDS = Loop::LDS / 4;
    static_assert(32 * PITCH <= WAVE_LDS && TN % 2 == 0, "a wavefront's piece of LDS holds 32 rows of its part of the tile");
    char* mine = lds + wave * WAVE_LDS;
    const int wave_n = wave % WN, wave_m = wave / WN, h = lane / 16;
    const int n_wave = (n0 + wave_n * TN * 16) / (MODE == OUT_SWIGLU ? 2 : 1);
    const int n_end = MODE == OUT_SWIGLU ? a.N / 2 : a.N;
    char* out = static_cast<char*>(a.C) + (MODE == OUT_F32 ? split * a.part_stride * 4 : 0);
#pragma unroll
    for (int g0 = 0; g0 < TM; g0 += 2) {
        const int m_base = m0 + (wave_m * TM + g0) * 16;
        if (m_base >= a.M) break;
#pragma unroll
        for (int g = g0; g < g0 + 2; ++g) {
            char* at = mine + ((g - g0) * 16 + lane % 16) * PITCH + h * 4 * SIZE;
#pragma unroll
            for (int f = 0; f < TN; f += MODE == OUT_SWIGLU ? 2 : 1) {
                const tile_f32x4& acc = loop.acc[f][g];
                if constexpr (MODE == OUT_F32) {
                    *reinterpret_cast<float4*>(at + f * 64) = float4{acc[0], acc[1], acc[2], acc[3]};
                } else {
                    tile_bf16x4 v;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (MODE == OUT_BF16) {
                            v[i] = (__bf16)acc[i];
                        } else {     // weight rows alternate in slabs of 16: the gate rows of 16 outputs, their up rows behind
                            const float gate = acc[i], up = loop.acc[f + 1][g][i];
                            // (a quarter of 1 + exp(-gate): its reciprocal is a normal number as long as the exponential is
                            // finite.  expf and a division, no nearer to 64 bits behind the rounding to bfloat16, cost 2 to 16 %.)
                            v[i] = (__bf16)(0.25f * gate * __builtin_amdgcn_rcpf(fmaf(0.25f, __expf(-gate), 0.25f)) * up);
                        }
                    }
                    *reinterpret_cast<tile_bf16x4*>(at + f * (MODE == OUT_SWIGLU ? 16 : 32)) = v;
                }
            }
        }
        tile_wave_sync();
#pragma unroll
        for (int it = 0; it < PCS / 2; ++it) {
            const int row = (it * PULSE_WAVE + lane) / PCS, pc = (it * PULSE_WAVE + lane) % PCS;
            const uint4 v = *reinterpret_cast<const uint4*>(mine + row * PITCH + pc * 16);
            const int m = m_base + row, n = n_wave + pc * (16 / SIZE);
            if (m < a.M && n < n_end) *reinterpret_cast<uint4*>(out + (m * a.ldc + n) * SIZE) = v;
        }
        tile_wave_sync();
    }
}

template <int MODE, int WR, int XR, int WN, int WM, int S, int SX = S, bool NT = true, bool FAR = false>
void launch(StageArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + XR - 1) / XR;
    a.tiles_n = (a.N + WR - 1) / WR;
    const int64_t grid = (static_cast<int64_t>(a.tiles_m) * a.tiles_n * a.splits + 7) / 8 * 8;
    hipLaunchKernelGGL((gemm_stages_kernel<MODE, WR, XR, WN, WM, S, SX, NT, FAR>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, a);
}

// weight rows and rows of X a tile (the kernels below, in this order)
constexpr int SHAPES[][2] = {{64, 64}, {64, 128}, {96, 128}, {128, 64}, {128, 128}, {192, 128}, {256, 128},
                               {192, 192}, {192, 256}, {256, 192}, {256, 256}};
constexpr int64_t FAR_ROWS = 1 << 22;   // values between rows that pulse_gemm_tile refuses
// Whether a tile's last row lies as near its first as a lane's 32-bit offset reaches (with the pieces and BACK and `inside` of TileLoop).
bool reaches(int rows, int64_t ld) { return (rows - 1) * ld * 2 + 8192 < (int64_t{1} << 32); }
constexpr int NUM_SHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

template <int MODE>
void launch_shape(int shape, const StageArgs& a, hipStream_t s) {
    // (what does not goes by pointers, in the smallest tiles: rows from 16 MB apart on in the largest ones, 68 MB in these)
    if (!reaches(SHAPES[shape][0], a.ldw) || !reaches(SHAPES[shape][1], a.ldx)) return launch<MODE, 64, 64, 2, 2, 6, 6, true, true>(a, s);
    switch (shape) {
        case 0: return launch<MODE, 64, 64, 2, 2, 6>(a, s);
        case 1: return launch<MODE, 64, 128, 2, 2, 6>(a, s);
        case 2: return launch<MODE, 96, 128, 1, 4, 5>(a, s);
        case 3: return launch<MODE, 128, 64, 4, 1, 3>(a, s);
        case 4: return launch<MODE, 128, 128, 2, 2, 4>(a, s);
        case 5: return launch<MODE, 192, 128, 2, 2, 3>(a, s);
        case 6: return launch<MODE, 256, 128, 2, 2, 3>(a, s);
        case 7: return launch<MODE, 192, 192, 2, 2, 3, 3, false>(a, s);
        case 8: return launch<MODE, 192, 256, 2, 2, 3, 2, false>(a, s);
        case 9: return launch<MODE, 256, 192, 2, 2, 3, 2, false>(a, s);
        default: return launch<MODE, 256, 256, 2, 2, 3, 2, false>(a, s);
    }
}

struct Plan { int shape, splits; double ns; };

// The shape (and, for float32 results in shares, their number: `shares` 0 leaves it open) of the least estimated time.  A
// row of a stage (128 bytes) takes a compute unit 3.1 ns.  Tiles of more than 128 rows of X hold weights long enough for
// their further rounds to find them near: 2 ns a row then, or what its products take on the matrix cores (1.13 x their
// time at the rate of a large product, 5.5 flops a picosecond a unit), and 0.75 of that for a last round that leaves half
// the units idle.  Beyond 512 rows, where several tiles read a weight's rows, large tiles take 2.6 ns a row from the first round on, or
// 0.94 x their products' time, and small ones 3.5.  Every share adds its results' way to memory and back to whoever adds them up (8
// bytes a value at 4 TB/s).  Estimated / measured, 24,576 x 4,096 with SwiGLU, us: 97 rows 96 x 128 44 / 38, 128 x 128 51 / 41; 357 rows
// 192 x 192 76 / 62, 192 x 256 89 / 78; 512 rows 192 x 256 89 / 80, 256 x 256 111 / 85; 1,024 rows 192 x 256 149 / 157; 2,048 rows 256 x 256
// 269 / 284.  (Which shape is best follows from it: over the 288 sizes measured from 257 rows on, of 18 weights, its choices take
// 0.3 % longer than the best shape's; without the figures for 512 rows and more 0.6 %, and shares of K that pay were not seen.)
Plan plan_for(int M, int N, int K, int shares) {
    const int64_t units = pulse_compute_units();
    Plan best{0, 1, 0.0};
    bool any = false;
    for (int splits = shares > 0 ? shares : 1; splits <= (shares > 0 ? shares : 16); ++splits) {
        if (K % (64 * splits)) continue;
        for (int i = 0; i < NUM_SHAPES; ++i) {
            const int wr = SHAPES[i][0], xr = SHAPES[i][1];
            const int64_t tiles = static_cast<int64_t>((M + xr - 1) / xr) * ((N + wr - 1) / wr) * splits;
            const int64_t rounds = (tiles + units - 1) / units, last = tiles - (rounds - 1) * units;
            const bool many = M > 512;
            double row = rounds * (many ? 3.5 : 3.1);
            if (xr > 128) {
                const double later = std::max(many ? 2.6 : 2.0, (many ? 0.94 : 1.13) * wr * xr * 128.0 / (wr + xr) / 5500.0);
                row = std::max(many ? 2.6 : 3.1, later) + (rounds - 1) * later;
                if (rounds > 1 && 2 * last <= units) row -= (many ? 0.2 : 0.25) * later;
            }
            const double ns = row * (wr + xr) * (K / splits / 64) + (shares == 1 ? 0.0 : splits * 8.0 / 4000.0 * M * N);
            if (!any || ns < best.ns) { best = {i, splits, ns}; any = true; }
        }
    }
    return best;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

// Whether the product takes these sizes: an inner dimension whose shares are multiples of 64, weight rows in multiples of
// 8 (of 32 with SwiGLU inside, of 4 for float32 results), shares only with float32 results.
extern "C" int pulse_gemm_stages_takes(int M, int N, int K, int mode, int splits) {
    if (M <= 0 || N <= 0 || K <= 0 || splits < 1 || mode < OUT_BF16 || mode > OUT_F32) return 0;
    if (splits > 1 && mode != OUT_F32) return 0;
    if (K % (64 * splits)) return 0;
    const int n_step = mode == OUT_SWIGLU ? 32 : (mode == OUT_BF16 ? 8 : 4);
    if (N % n_step) return 0;
    return static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64) * splits <= (1 << 27);
}

// How many shares of K float32 results are best made in (0: a shape that the product does not take).
extern "C" int pulse_gemm_stages_shares(int M, int N, int K) {
    if (!pulse_gemm_stages_takes(M, N, K, OUT_F32, 1)) return 0;
    return plan_for(M, N, K, 0).splits;
}

// The tile of a product in so many shares: weight rows * 1,024 + rows of X (0: a shape that the product does not take).
extern "C" int pulse_gemm_stages_tile(int M, int N, int K, int splits) {
    if (!pulse_gemm_stages_takes(M, N, K, OUT_F32, splits) && !(splits == 1 && pulse_gemm_stages_takes(M, N, K, OUT_BF16, 1))) return 0;
    const int shape = plan_for(M, N, K, splits).shape;
    return SHAPES[shape][0] * 1024 + SHAPES[shape][1];
}

// The estimated time of bfloat16 results in nanoseconds, at most 2 s (0: a shape that the product
// does not take).
extern "C" int pulse_gemm_stages_time(int M, int N, int K) {
    return pulse_gemm_stages_takes(M, N, K, OUT_BF16, 1) ? static_cast<int>(std::min(plan_for(M, N, K, 1).ns, 2e9)) : 0;
}

// What both products check before they launch: operands there and aligned, rows that hold K values, results that hold N.
static int check_operands(const char* name, const void* X, int64_t ldx, const void* W, int64_t ldw, const void* C, int64_t ldc, int M, int N,
                          int K, int mode, int splits, int64_t part_stride) {
    PULSE_REQUIRE(pulse_gemm_stages_takes(M, N, K, mode, splits),
                  "%s: %d rows x %d weight rows x inner dimension %d, mode %d, %d shares: the inner dimension must "
                  "be a multiple of 64 a share, the weight rows a multiple of 8 (32 with SwiGLU, 4 for float32 results), "
                  "shares need float32 results", name, M, N, K, mode, splits);
    PULSE_REQUIRE(X && W && C && aligned16(X) && aligned16(W) && aligned16(C), "%s: operands must be aligned to 16 bytes", name);
    PULSE_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0, "%s: rows of X and W must be K long at "
                  "least and start at multiples of 16 bytes (strides %lld, %lld)", name, (long long)ldx, (long long)ldw);
    const int out_cols = mode == OUT_SWIGLU ? N / 2 : N;
    PULSE_REQUIRE(ldc >= out_cols && ldc % (mode == OUT_F32 ? 4 : 8) == 0, "%s: rows of the result must be %d long "
                  "at least and start at multiples of 16 bytes (stride %lld)", name, out_cols, (long long)ldc);
    PULSE_REQUIRE(splits == 1 || (part_stride >= static_cast<int64_t>(M - 1) * ldc + N && part_stride % 4 == 0),
                  "%s: the shares' results overlap (stride %lld)", name, (long long)part_stride);
    return 0;
}

static void launch_mode(int mode, int shape, const StageArgs& a, hipStream_t stream) {
    if (mode == OUT_BF16) launch_shape<OUT_BF16>(shape, a, stream);
    else if (mode == OUT_SWIGLU) launch_shape<OUT_SWIGLU>(shape, a, stream);
    else launch_shape<OUT_F32>(shape, a, stream);
}

// mode 0: C [M, N] bfloat16.  mode 1: the rows of W alternate in slabs of 16 gate rows and their 16 up rows;
// C [M, N / 2] bfloat16 = silu(gate) * up.  mode 2: float32, one result [M, N] for every share of K, `part_stride`
// elements apart (the shares are added up by whoever reads them, in order).
extern "C" int pulse_gemm_stages(const void* X, int64_t ldx, const void* W, int64_t ldw, void* C, int64_t ldc, int M, int N,
                                 int K, int mode, int splits, int64_t part_stride, hipStream_t stream) {
    if (const int bad = check_operands("gemm_stages", X, ldx, W, ldw, C, ldc, M, N, K, mode, splits, part_stride)) return bad;
    launch_mode(mode, plan_for(M, N, K, splits).shape,
                {static_cast<const bf16_t*>(X), ldx, static_cast<const bf16_t*>(W), ldw, C, ldc, M, N, K / splits, 0, 0, splits,
                 splits > 1 ? part_stride : 0}, stream);
    PULSE_LAUNCH_CHECK("gemm_stages");
    return 0;
}

// The same in tiles of 256 x 256 whatever the rows (fewer sizes: at most 2^24 tiles, rows less than 4M values apart).
extern "C" int pulse_gemm_tile_takes(int M, int N, int K, int mode, int splits) {
    if (!pulse_gemm_stages_takes(M, N, K, mode, splits)) return 0;
    return static_cast<int64_t>((M + 255) / 256) * ((N + 255) / 256) * splits <= (1 << 24);
}

extern "C" int pulse_gemm_tile(const void* X, int64_t ldx, const void* W, int64_t ldw, void* C, int64_t ldc, int M, int N,
                               int K, int mode, int splits, int64_t part_stride, void* stream) {
    if (const int bad = check_operands("gemm_tile", X, ldx, W, ldw, C, ldc, M, N, K, mode, splits, part_stride)) return bad;
    PULSE_REQUIRE(pulse_gemm_tile_takes(M, N, K, mode, splits) && ldx < FAR_ROWS && ldw < FAR_ROWS,
                  "gemm_tile: at most 2^24 tiles, and rows of X and W less than 4M elements apart (strides %lld, %lld)",
                  (long long)ldx, (long long)ldw);
    launch_mode(mode, NUM_SHAPES - 1,
                {static_cast<const bf16_t*>(X), ldx, static_cast<const bf16_t*>(W), ldw, C, ldc, M, N, K / splits, 0, 0, splits,
                 splits > 1 ? part_stride : 0}, static_cast<hipStream_t>(stream));
    PULSE_LAUNCH_CHECK("gemm_tile");
    return 0;
}
