// Paged attention on the matrix cores over latent rows of up to 576 channels, which every query head shares as keys and, up to 512
// channels of them, as values.  bfloat16 operands, float32 everything else, float32 results.
//
// An item is 32 rows: `hp` query heads (all of them, up to 32) for 32 / hp consecutive tokens of one request.  A workgroup takes an
// item and a share of its keys in blocks of 64, and brings every key and every value of them in once:
//
//   S^T = K Q^T      eight wavefronts: wavefront w takes keys 16 (w % 4) .. + 15 of the block over half w / 4 of the channels, for both
//                    row tiles (the rows' queries lie in LDS); the two with the same keys meet in LDS and go on with a row tile each.
//                    A lane holds, for its row (lane % 16), the scores of keys 4 (lane / 16) + i;
//   softmax          the maxima of the keys meet in LDS, then every wavefront puts its weights there, row by row;
//   O^T += V^T P^T   wavefront w takes value channels 64 w .. of all 64 keys: the weights from LDS, the values straight from the
//                    pages (channel by channel there, so eight keys of a channel are one piece of 16 bytes).
//
// What bounds it: trips to memory (list and block table, then queries, keys and values together), then what a compute unit takes
// in, 139 KB a block at 576 + 512 channels; with few tokens also the merge behind.  So a block's values are asked for with its keys,
// the next block's keys as soon as this block's scores are there, and the keys are cut as finely as the launch has room for.  The
// kernel for wide values, which took this work before, gives a workgroup 16 rows and 256 value channels: at 32 heads it brought every
// key in four times and every value twice.  One wavefront more a SIMD (128 registers) does not hold the keys and values in flight.
// us with the merge, 32 heads, rows of 576 channels from memory, before -> this: one request of 600 tokens 16.8 -> 12.8, of 5,000
// 36 -> 22; 8 of 300 18 -> 12.8, of 1,500 28.5 -> 17.7, of 4,000 50 -> 27; 32 of 1,000 49 -> 27; 64 of 500 50 -> 27; prompts of 3 x 51
// 24.8 -> 11.5.  A block takes 4 us when everything is found in L2: the wavefronts' instructions and LDS, three barriers among them.
#include "common.h"

#include <math.h>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;

constexpr int ROWS = 32;             // of an item, two tiles of 16
constexpr int KEYS = 64;             // of a block
constexpr int PAGES = 4;             // tiles of 16 keys, each within a page
static_assert(KEYS == 16 * PAGES, "four tiles a block");
constexpr int WAVES = 2 * PAGES;
constexpr int CT = 4;                // tiles of 16 value channels a wavefront has at most
constexpr int P_STRIDE = KEYS + 8;   // of a row of weights: 16 bytes more, so that sixteen rows' pieces lie in different banks

struct LatentArgs {
    int nq, d, wv, hp;
    int64_t q_stride, o_stride;
    int page_size, num_pages, bt_width;
    float scale, cap;
    int window;
    int n_splits;         // > 1: an item's blocks are shared out over gridDim.y workgroups, whose sums go to `part`
    float* part;          // [items, ROWS, n_splits, wv] sums not yet divided
    float* part_ml;       // [items, ROWS, n_splits, 2] maximum and sum of weights
};

// Integers that are only read.  AGAIN: by scalar loads also behind stores (where there are none the compiler sees that by itself, and
// asks for the queries first).
template <bool AGAIN>
__device__ __forceinline__ auto scalars(const int* p) {
    if constexpr (AGAIN) return (const __attribute__((address_space(4))) int*)reinterpret_cast<uintptr_t>(p);
    else return p;
}

// A row's result is its sums times this: 1 / sum of weights; a sink is one more term of that sum, exp(sink), with no key and no value.
__device__ __forceinline__ float whole_share(float m, float l, const float* sink, int head) {
    float scale_out = 1.f;
    if (sink) {
        const float sk = sink[head];
        if (m == -INFINITY) l = 1.f;
        else if (sk > m) { scale_out = expf(m - sk); l = l * scale_out + 1.f; }
        else l += expf(sk - m);
    }
    return l > 0.f ? scale_out / l : 0.f;
}

// CHUNKS: of 192 channels, as many as hold the head's; USUAL: exactly as many, every wavefront's value channels, and pages of 16 keys.
//
// SEVERAL: items may hold several tokens.  A value that is not finite and that not all of them see would reach the others too (zero
// times it).  So the blocks that not all see in full are looked through; where one is found, nothing is stored and the tokens come one
// at a time, with every value that the token does not see cleared.  (A kernel of its own: short portions wait for it, us without /
// with: 8 x 16 tokens on 1,000 keys at 16 heads 37.2 / 38.1, 3 x 51 10.1 / 11.2; a decoded token, which needs none of it, would take
// 11.9 / 12.4 on 600 keys.)
template <int CHUNKS, bool USUAL, bool SEVERAL>
__global__ __launch_bounds__(WAVES* PULSE_WAVE, 2) void attn_latent_kernel(const bf16_t* __restrict__ q, float* __restrict__ out,
                                                                           const bf16_t* __restrict__ kcache,
                                                                           const bf16_t* __restrict__ vcache,
                                                                           const int* __restrict__ positions,
                                                                           const int* __restrict__ token_entry,
                                                                           const int* __restrict__ block_table,
                                                                           const int* __restrict__ items,
                                                                           const float* __restrict__ sink, LatentArgs a) {
    constexpr int THREADS = WAVES * PULSE_WAVE;
    constexpr int PIECES = 3 * CHUNKS;                     // of 32 channels, of half of a head
    constexpr int WIDTH = 64 * PIECES;
    constexpr int Q_STRIDE = WIDTH + 8;                    // (16 bytes more, as P_STRIDE)
    __shared__ __attribute__((aligned(16))) bf16_t q_s[ROWS * Q_STRIDE];
    __shared__ __attribute__((aligned(16))) bf16_t p_s[ROWS * P_STRIDE];
    __shared__ f32x4 half_s[WAVES][PULSE_WAVE];
    __shared__ float max_s[PAGES][ROWS], sum_s[PAGES][ROWS];
    const int* it = items + 4 * blockIdx.x;
    const int t0 = it[0], nt = it[1], head0 = it[2], nh = it[3];
    for (int from = 0, to = nt;;) {      // (all tokens at once, or one after the other)
        int thread = threadIdx.x;
        if constexpr (SEVERAL) asm volatile("" : "+v"(thread));      // (nothing made of it is kept in registers for another pass)
        const int lane = thread % PULSE_WAVE, wave = __builtin_amdgcn_readfirstlane(thread / PULSE_WAVE);
        const int kt = wave % PAGES, half = wave / PAGES;
        const int r = lane % 16, g = lane / 16;
        const int d = USUAL ? WIDTH : a.d, page_size = USUAL ? 16 : a.page_size;

        // the rows' queries (rows that nobody has repeat the first token's first head; channels behind the head's are zeros)
        constexpr int Q_PIECES = ROWS * WIDTH / 8, Q_EACH = (Q_PIECES + THREADS - 1) / THREADS;     // of 16 bytes; those of a thread
        u32x4 qv[Q_EACH];
#pragma unroll
        for (int i = 0; i < Q_EACH; ++i) {
            const int at = min(thread + i * THREADS, Q_PIECES - 1), row = at / (WIDTH / 8), e = at % (WIDTH / 8) * 8;
            const int ti = row / a.hp, hi = row % a.hp;
            const bool there = ti < nt && hi < nh;
            qv[i] = *reinterpret_cast<const u32x4*>(q + static_cast<int64_t>(t0 + (there ? ti : 0)) * a.q_stride +
                                                    static_cast<int64_t>(head0 + (there ? hi : 0)) * d + min(e, d - 8));
        }
        __builtin_amdgcn_sched_barrier(0);      // (the queries are asked for before the trips to the lists)
        const auto bt = scalars<SEVERAL>(block_table) + static_cast<int64_t>(scalars<SEVERAL>(token_entry)[t0]) * a.bt_width;
        const int pos_first = scalars<SEVERAL>(positions)[t0], pos_last = scalars<SEVERAL>(positions)[t0 + nt - 1];
        const int lo = (a.window > 0 && pos_first - a.window + 1 > 0) ? pos_first - a.window + 1 : 0;
        const int lo16 = lo & ~15;
        const int blocks = (pos_last + 1 - lo16 + KEYS - 1) / KEYS;
        const int per = (blocks + a.n_splits - 1) / a.n_splits;
        const int block0 = static_cast<int>(blockIdx.y) * per, block1 = min(blocks, block0 + per);

        // the page of a block's tile of 16 keys, -1 where there is none
        pulse_i32x4 page, found;      // (vectors: of arrays that a lane or a wavefront chooses from, the compiler makes memory)
        auto look_up = [&](int block) __attribute__((always_inline)) {      // (a block ahead, so that the table's trip lies behind another)
#pragma unroll
            for (int t = 0; t < PAGES; ++t) found[t] = bt[min((lo16 + block * KEYS + 16 * t) / page_size, a.bt_width - 1)];
        };
        auto take_pages = [&](int block) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < PAGES; ++t) {
                const int j = lo16 + block * KEYS + 16 * t, pi = j / page_size;
                const int p = __builtin_amdgcn_readfirstlane(found[t]);
                page[t] = (j <= pos_last) & (pi < a.bt_width) & (p >= 0) & (p < a.num_pages) ? p : -1;
            }
        };
        auto own_page = [&]() __attribute__((always_inline)) {
            int mine = page[0];
#pragma unroll
            for (int t = 1; t < PAGES; ++t) mine = kt == t ? page[t] : mine;
            return mine;
        };
        bf16x8 ka[PIECES];
        auto ask_keys = [&](int block) __attribute__((always_inline)) {      // (addresses that always hold keys; masked behind)
            const int off = (lo16 + block * KEYS + 16 * kt) % page_size;
            const int e0 = 32 * PIECES * half + 8 * g;
            const bf16_t* krow = kcache + (static_cast<int64_t>(max(own_page(), 0)) * page_size + off + r) * d + (USUAL ? e0 : 0);
#pragma unroll
            for (int u = 0; u < PIECES; ++u) ka[u] = *reinterpret_cast<const bf16x8*>(krow + (USUAL ? 32 * u : min(e0 + 32 * u, d - 8)));
        };
        const int tiles = USUAL ? CT : max(0, min(CT, a.wv / 16 - CT * wave));   // of value channels, this wavefront's
        u32x4 values[2][CT][2];                                              // of this block and the next, in turn
        const bool idle = !USUAL && tiles == 0;      // no value channels: nothing to bring in and nothing to add up
        auto ask_values = [&](int block, u32x4 (&va)[CT][2]) __attribute__((always_inline)) {
            if (idle) return;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int p = g / 2 ? page[2 * u + 1] : page[2 * u];
                const int off = (lo16 + block * KEYS + 32 * u + 16 * (g / 2)) % page_size + 8 * (g % 2);
                const bf16_t* base = vcache + (static_cast<int64_t>(max(p, 0)) * d + 16 * CT * wave + r) * page_size + off;
#pragma unroll
                for (int c = 0; c < CT; ++c) va[c][u] = *reinterpret_cast<const u32x4*>(base + (USUAL ? c : min(c, tiles - 1)) * (16 * page_size));
            }
        };

        int pos[2], token[2], head[2];
        bool valid[2];
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            const int row = 16 * rr + r, ti = row / a.hp, hi = row % a.hp;
            valid[rr] = ti >= from && ti < to && hi < nh;
            token[rr] = t0 + (valid[rr] ? ti : 0);
            head[rr] = head0 + (valid[rr] ? hi : 0);
            pos[rr] = positions[token[rr]];
        }
        const int seen_last = SEVERAL ? scalars<SEVERAL>(positions)[t0 + to - 1] : pos_last;       // the keys that any of the pass's tokens sees
        const int seen_first = from == 0 ? lo : a.window > 0 ? max(0, seen_last - a.window + 1) : 0;
        u16x2 odd = {0, 0};      // the largest of the values that not all of them see, without their signs
        const bool own_valid = half ? valid[1] : valid[0];
        const int own_pos = half ? pos[1] : pos[0];
        float m_run[2] = {-INFINITY, -INFINITY}, l_run = 0.f;
        f32x4 acc[2][CT];
#pragma unroll
        for (int rr = 0; rr < 2; ++rr)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[rr][c] = f32x4{0.f, 0.f, 0.f, 0.f};

        look_up(block0);
        take_pages(block0);
        look_up(block0 + 1);
        ask_keys(block0);          // (a workgroup without blocks asks for the first page's, for nobody)
        ask_values(block0, values[0]);
#pragma unroll
        for (int i = 0; i < Q_EACH; ++i) {
            const int at = min(thread + i * THREADS, Q_PIECES - 1), e = at % (WIDTH / 8) * 8;   // (the last piece several times)
            *reinterpret_cast<u32x4*>(&q_s[at / (WIDTH / 8) * Q_STRIDE + e]) = e < d ? qv[i] : u32x4{0u, 0u, 0u, 0u};
        }
        __syncthreads();

        auto step = [&](int block, u32x4 (&va)[CT][2], u32x4 (&va_next)[CT][2]) __attribute__((always_inline)) {
            const int j0 = lo16 + block * KEYS;
            if constexpr (!USUAL) {
#pragma unroll
                for (int u = 0; u < PIECES; ++u)
                    if (32 * (PIECES * half + u) + 8 * g >= d) ka[u] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
            }
            f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
            // (a piece's queries ahead of its products, no more: the keys and values in flight take the registers)
            bf16x8 qb[2][2];
            const bf16_t* q_at = &q_s[r * Q_STRIDE + 32 * PIECES * half + 8 * g];
            auto read_queries = [&](int u) __attribute__((always_inline)) {
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) qb[u % 2][rr] = *reinterpret_cast<const bf16x8*>(q_at + 16 * rr * Q_STRIDE + 32 * u);
            };
            read_queries(0);
#pragma unroll
            for (int u = 0; u < PIECES; ++u) {
                if (u + 1 < PIECES) read_queries(u + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) s[rr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[u], qb[u % 2][rr], s[rr], 0, 0, 0);
            }
            const f32x4 s0 = s[0], s1 = s[1];
            half_s[wave][lane] = half ? s0 : s1;
            __syncthreads();
            f32x4 own = half ? s1 : s0;
            own += half_s[(wave + PAGES) % WAVES][lane];
            // what of this block's values nobody sees, or has never been stored, is cleared (a weight of zero times whatever lies there
            // must stay zero)
            const bool there = own_page() >= 0;
            const bool whole = j0 >= seen_first && j0 + KEYS - 1 <= seen_last && page[0] >= 0 && page[1] >= 0 && page[2] >= 0 && page[3] >= 0;
            if (!whole && !idle) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int p = g / 2 ? page[2 * u + 1] : page[2 * u];
                    const int gone = seen_first - (j0 + 32 * u + 8 * g);
                    const uint32_t seen = p >= 0 ? seen_last + 1 - seen_first : 0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t keep = (static_cast<uint32_t>(2 * k - gone) < seen ? 0x0000FFFFu : 0u) |
                                              (static_cast<uint32_t>(2 * k + 1 - gone) < seen ? 0xFFFF0000u : 0u);
#pragma unroll
                        for (int c = 0; c < CT; ++c) va[c][u][k] &= keep;
                    }
                }
            }
            if (SEVERAL && !idle && to - from > 1 && (j0 + KEYS - 1 > pos_first || (a.window > 0 && j0 <= pos_last - a.window))) {
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int c = 0; c < CT; ++c)
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            odd = __builtin_elementwise_max(odd, __builtin_bit_cast(u16x2, va[c][u][k] & 0x7FFF7FFFu));
            }
            if (block + 1 < block1) {
                take_pages(block + 1);
                look_up(block + 2);
                ask_keys(block + 1);
                ask_values(block + 1, va_next);
            }
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = j0 + 16 * kt + 4 * g + i;
                float x = own[i] * a.scale;
                if (a.cap > 0.f) x = a.cap * tanhf(x / a.cap);
                own[i] = own_valid && there && j <= own_pos && (a.window == 0 || own_pos - j < a.window) ? x : -INFINITY;
                mx = fmaxf(mx, own[i]);
            }
            mx = across_rows(mx, LaneMax());
            if (g == 0) max_s[kt][16 * half + r] = mx;
            __syncthreads();
            float alpha[2];
#pragma unroll
            for (int rr = 0; rr < 2; ++rr) {
                float m_new = m_run[rr];
#pragma unroll
                for (int w = 0; w < PAGES; ++w) m_new = fmaxf(m_new, max_s[w][16 * rr + r]);
                alpha[rr] = m_new == -INFINITY ? 1.f : expf(m_run[rr] - m_new);
                m_run[rr] = m_new;
            }
            const float m_own = half ? m_run[1] : m_run[0];
            float sum = 0.f;
            bf16x4 p4;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = own[i] == -INFINITY ? 0.f : expf(own[i] - m_own);
                sum += p;
                p4[i] = static_cast<__bf16>(p);
            }
            *reinterpret_cast<bf16x4*>(&p_s[(16 * half + r) * P_STRIDE + 16 * kt + 4 * g]) = p4;
            l_run = l_run * (half ? alpha[1] : alpha[0]) + sum;
            __syncthreads();
            if (idle) return;
#pragma unroll
            for (int rr = 0; rr < 2; ++rr)
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[rr][c] *= alpha[rr];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bf16x8 pb[2];
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) pb[rr] = *reinterpret_cast<const bf16x8*>(&p_s[(16 * rr + r) * P_STRIDE + 32 * u + 8 * g]);
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int rr = 0; rr < 2; ++rr)
                        acc[rr][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, va[c][u]), pb[rr], acc[rr][c], 0, 0, 0);
            }
            // (the next block's weights are written behind two more barriers, its halves and maxima behind one, after all have been read)
        };
        for (int block = block0; block < block1; block += 2) {
            step(block, values[0], values[1]);
            if (block + 1 < block1) step(block + 1, values[1], values[0]);
        }
        if constexpr (SEVERAL) {
            if (to - from > 1 && __syncthreads_or(max(odd[0], odd[1]) >= 0x7F80)) {
                to = 1;
                continue;
            }
        }
        // a row's sum over the lanes and the wavefronts that share it
        l_run = across_rows(l_run, LaneSum());
        if (g == 0) sum_s[kt][16 * half + r] = l_run;
        __syncthreads();
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
            float l = 0.f;
#pragma unroll
            for (int w = 0; w < PAGES; ++w) l += sum_s[w][16 * rr + r];
            float* row;
            float share = 1.f;
            if (a.n_splits > 1) {       // one of several workgroups over these keys: the sums as they are, for the merge
                const int64_t at = (static_cast<int64_t>(blockIdx.x) * ROWS + 16 * rr + r) * a.n_splits + blockIdx.y;
                if (valid[rr] && wave == 0 && g == 0) { a.part_ml[2 * at] = m_run[rr]; a.part_ml[2 * at + 1] = l; }
                row = a.part + at * a.wv;
            } else {
                share = whole_share(m_run[rr], l, sink, head[rr]);
                row = out + static_cast<int64_t>(token[rr]) * a.o_stride + static_cast<int64_t>(head[rr]) * d;
            }
            if (valid[rr]) {
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    if (c < tiles) *reinterpret_cast<f32x4*>(row + 16 * (CT * wave + c) + 4 * g) = acc[rr][c] * share;
            }
        }
        if (!SEVERAL || to == nt) break;
        from = to++;
        __syncthreads();
    }
}

// The sums of the workgroups that shared an item's keys, brought together: a workgroup a row of an item.
__global__ __launch_bounds__(256) void attn_latent_merge_kernel(const float* __restrict__ part, const float* __restrict__ part_ml,
                                                                float* __restrict__ out, const int* __restrict__ items,
                                                                const float* __restrict__ sink, LatentArgs a) {
    __shared__ float factor[PULSE_WAVE];
    const int* it = items + 4 * blockIdx.x;
    const int ti = blockIdx.y / a.hp, hi = blockIdx.y % a.hp;
    if (ti >= it[1] || hi >= it[3]) return;
    const int token = it[0] + ti, head = it[2] + hi;
    const int64_t at = (static_cast<int64_t>(blockIdx.x) * ROWS + blockIdx.y) * a.n_splits;
    const int lane = threadIdx.x % PULSE_WAVE;         // (at most 64 splits: a lane a split, every wavefront for itself)
    const float m = lane < a.n_splits ? part_ml[2 * (at + lane)] : -INFINITY;
    const float l = lane < a.n_splits ? part_ml[2 * (at + lane) + 1] : 0.f;
    const float m_all = wave_max(m);
    const float f = m == -INFINITY ? 0.f : expf(m - m_all);
    const float l_all = wave_sum(m == -INFINITY ? 0.f : l * f);
    if (threadIdx.x < PULSE_WAVE) factor[lane] = f;
    __syncthreads();
    const float share = whole_share(m_all, l_all, sink, head);
    float* row = out + static_cast<int64_t>(token) * a.o_stride + static_cast<int64_t>(head) * a.d;
    // (two groups of threads take the splits in turn, four channels a thread, and meet in LDS: a split's values by themselves are a
    // trip to memory)
    __shared__ f32x4 half[128];
    const int part_of = threadIdx.x / 128, ch = threadIdx.x % 128 * 4;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (ch < a.wv) {
        const float* from = part + at * a.wv + ch;
        constexpr int AHEAD = 8;
        for (int s0 = part_of; s0 < a.n_splits; s0 += 2 * AHEAD) {
            f32x4 v[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                v[u] = *reinterpret_cast<const f32x4*>(from + static_cast<int64_t>(min(s0 + 2 * u, a.n_splits - 1)) * a.wv);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (s0 + 2 * u < a.n_splits) sum += v[u] * factor[s0 + 2 * u];
        }
    }
    if (part_of == 1) half[threadIdx.x - 128] = sum;
    __syncthreads();
    if (part_of == 0 && ch < a.wv) *reinterpret_cast<f32x4*>(row + ch) = (sum + half[threadIdx.x]) * share;
}

}  // namespace

// q [tokens, q_stride] bfloat16: head h's query at h * d.  out float32 [tokens, o_stride]: of head h's d channels at h * d the first
// wv are written.  items int32 [n_items, 4]: first token, tokens, first head, heads; row r (of 32) of an item is token r / hp, head
// r % hp; rows that no item holds are left as they are.  several: whether an item may hold several tokens.  n_splits > 1: the keys
// of every item are shared out over that many workgroups, whose sums (part float32 [n_items, 32, n_splits, wv], part_ml [n_items, 32,
// n_splits, 2]) a second kernel brings together.  kcache [pages, 1, page, d], vcache [pages, 1, d, page] bfloat16.
extern "C" int pulse_attn_latent(const void* q, int64_t q_stride, float* out, int64_t o_stride, const void* kcache,
                                 const void* vcache, const int* positions, const int* token_entry, const int* block_table,
                                 int bt_width, const int* items, int n_items, int hp, int several, int nq, int d, int wv,
                                 int page_size, int num_pages, float scale, int window, const float* sink, float softcap, int n_splits,
                                 float* part, float* part_ml, hipStream_t stream) {
    PULSE_REQUIRE(nq > 0 && d >= 16 && d % 16 == 0 && d <= 576, "attn_latent: %d heads of %d channels", nq, d);
    PULSE_REQUIRE(wv > 0 && wv % 16 == 0 && wv <= d && wv <= 16 * CT * WAVES, "attn_latent: %d of %d value channels", wv, d);
    PULSE_REQUIRE(page_size > 0 && page_size % 16 == 0 && num_pages > 0 && bt_width > 0, "attn_latent: pages must hold a multiple of 16 keys");
    PULSE_REQUIRE(hp >= 1 && hp <= ROWS && n_items >= 0, "attn_latent: bad items");
    PULSE_REQUIRE(window >= 0 && softcap >= 0.f, "attn_latent: bad window or score cap");
    PULSE_REQUIRE(n_splits >= 1 && n_splits <= 64 && (n_splits == 1 || (part && part_ml)), "attn_latent: %d splits need their scratch", n_splits);
    PULSE_REQUIRE(q_stride >= static_cast<int64_t>(nq) * d && o_stride >= static_cast<int64_t>(nq) * d && o_stride % 4 == 0 &&
                  q_stride % 8 == 0, "attn_latent: row strides too small or unaligned");
    PULSE_REQUIRE(q && out && kcache && vcache && positions && token_entry && block_table && items, "attn_latent: null pointer");
    PULSE_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(kcache) % 16 == 0 && reinterpret_cast<uintptr_t>(vcache) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(part) % 16 == 0, "attn_latent: operands must be 16-byte aligned");
    if (n_items == 0) return 0;
    LatentArgs a;
    a.nq = nq; a.d = d; a.wv = wv; a.hp = hp;
    a.q_stride = q_stride; a.o_stride = o_stride; a.page_size = page_size; a.num_pages = num_pages; a.bt_width = bt_width;
    a.scale = scale; a.cap = softcap; a.window = window;
    a.n_splits = n_splits; a.part = part; a.part_ml = part_ml;
    auto launch = [&](auto chunks, auto usual) {
        auto run = [&](auto several_v) {
            hipLaunchKernelGGL((attn_latent_kernel<decltype(chunks)::value, decltype(usual)::value, decltype(several_v)::value>),
                               dim3(n_items, n_splits), dim3(WAVES * PULSE_WAVE), 0, stream, static_cast<const bf16_t*>(q), out,
                               static_cast<const bf16_t*>(kcache), static_cast<const bf16_t*>(vcache), positions, token_entry,
                               block_table, items, sink, a);
        };
        if (several && hp <= ROWS / 2) run(std::true_type());      // (with more heads an item holds one token)
        else run(std::false_type());
    };
    if (d == 576 && wv == 16 * CT * WAVES && page_size == 16) launch(std::integral_constant<int, 3>(), std::true_type());
    else if (d > 384) launch(std::integral_constant<int, 3>(), std::false_type());
    else launch(std::integral_constant<int, 2>(), std::false_type());
    PULSE_LAUNCH_CHECK("attn_latent");
    if (n_splits > 1) {
        hipLaunchKernelGGL(attn_latent_merge_kernel, dim3(n_items, ROWS), dim3(256), 0, stream, part, part_ml, out, items, sink, a);
        PULSE_LAUNCH_CHECK("attn_latent_merge");
    }
    return 0;
}
