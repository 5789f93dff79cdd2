// Paged causal attention for any head size, page size and storage type: one
// wavefront per (token, query head), float32 arithmetic throughout.
//
// A token at position p sees keys lo..p of its own request through the block
// table, lo = max(0, p - window + 1) when a window is set, p - p mod chunk when chunks are, else 0.  Keys are
// taken 64 at a time (one per lane); the softmax is the running-maximum form
// (reference: src/ops/kernels/cuda/paged_attention.cu:88-137), the scale is a
// parameter (the reference fixes rsqrt(head_size), paged_attention.cu:108), and
// query head h reads kv head h / (nq / nkv) (paged_attention.cu:61-70).
//
// With `gate` every head's output is multiplied by sigmoid(gate[token, head]) before it is stored (an output gate
// whose logits another product left, one a token and head, `gate_stride` elements from row to row); with
// `gate_width` > 0 there is a logit for each of the first `gate_width` channels of every head instead
// (gate[token, head * gate_width + channel]).  `softcap` > 0 bounds the scaled scores, s <- cap * tanh(s / cap).
// `sink` (float32, one a query head) adds exp(sink[h]) to the softmax's denominator: a term without key or value.
//
// `keep_first` > 0 (with a window): the first keep_first keys of the request stay visible whatever the window, at their
// true positions.  `all_values`: a query head's weights are applied to the values of EVERY kv head, not only its own:
// the output row of (token, head) is nkv * d wide (value head c at columns c * d ..), in float32, for a caller that
// mixes the heads' weights afterwards (a weighted sum over query heads of these rows is the same as mixing the weights
// before they meet the values).
//
// This is the kernel of the true 32-bit path and the fallback for sizes that the
// matrix-core kernels refuse.  Float32 heads of 32, 64, 128 or 256 channels in pages of a multiple of 16 keys take
// `attn_rows_f32_kernel` below, which walks the same keys on the float32 matrix instruction.
#include "common.h"

#include <math.h>

namespace {


struct AttnArgs {
    int nq, nkv, d;
    int64_t q_stride, o_stride;
    int page_size, num_pages, bt_width;
    float scale;
    int window;  // 0: all keys
    int chunk;   // > 0 (without a window): the keys of the token's own chunk of this many positions
    float cap;   // > 0: a score s becomes cap * tanh(s / cap); 0: scores as they are
    int gate_per_channel;   // 0: one gate logit a head; 1: one a channel (gate [T, nq * gate_width])
    int gate_width;         // channels of a head that have a gate logit (the others are stored ungated)
    int keep_first;         // with a window: keys 0 .. keep_first - 1 stay visible
    int all_values;         // 1: the values of all kv heads side by side (nkv * d accumulators a query head)
};

template <typename TX, typename TC, typename TO, int MAX_ACC>
__global__ __launch_bounds__(64) void attn_generic_kernel(const TX* __restrict__ q, TO* __restrict__ out,
                                                          const TC* __restrict__ kcache,
                                                          const TC* __restrict__ vcache,
                                                          const int* __restrict__ positions,
                                                          const int* __restrict__ token_entry,
                                                          const int* __restrict__ block_table,
                                                          const TX* __restrict__ gate, int64_t gate_stride,
                                                          const float* __restrict__ sink, AttnArgs a) {
    extern __shared__ long long lds[];
    long long* v_s = lds;                                         // [64] value offsets of a tile's keys
    float* p_s = reinterpret_cast<float*>(lds + PULSE_WAVE);      // [64] a tile's probabilities
    float* q_s = p_s + PULSE_WAVE;                                // [d]  the scaled query

    const int t = blockIdx.x;
    const int h = blockIdx.y;
    const int lane = threadIdx.x;
    const int d = a.d;
    const int group = a.nq / a.nkv;
    const int kvh = h / group;
    const int pos = positions[t];
    const int* bt = block_table + static_cast<int64_t>(token_entry[t]) * a.bt_width;
    const int lo = a.chunk > 0 ? pos - pos % a.chunk : (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
    const int n_first = min(a.keep_first, lo);        // kept keys below the window
    const int total = n_first + pos - lo + 1;         // keys this token sees
    const int width = a.all_values ? a.nkv * d : d;   // values accumulated for this query head

    const TX* qrow = q + static_cast<int64_t>(t) * a.q_stride + static_cast<int64_t>(h) * d;
    for (int e = lane; e < d; e += PULSE_WAVE) q_s[e] = to_f32<TX>(qrow[e]) * a.scale;
    __syncthreads();

    float m = -INFINITY, l = 0.f;
    float acc[MAX_ACC];
#pragma unroll
    for (int r = 0; r < MAX_ACC; ++r) acc[r] = 0.f;

    for (int u0 = 0; u0 < total; u0 += PULSE_WAVE) {
        const int u = u0 + lane;
        const int j = u < n_first ? u : lo + u - n_first;
        float s = -INFINITY;
        long long vbase = -1;
        if (u < total) {
            const int pi = j / a.page_size;
            const int page = pi < a.bt_width ? bt[pi] : -1;
            if (page >= 0 && page < a.num_pages) {
                const int slot = j % a.page_size;
                const int64_t pg = static_cast<int64_t>(page) * a.nkv + kvh;
                const TC* krow = kcache + (pg * a.page_size + slot) * d;
                float dot = 0.f;
                for (int e = 0; e < d; ++e) dot = fmaf(q_s[e], to_f32<TC>(krow[e]), dot);
                s = a.cap > 0.f ? a.cap * tanhf(dot / a.cap) : dot;
                vbase = (a.all_values ? static_cast<int64_t>(page) * a.nkv : pg) * d * a.page_size + slot;
            }
        }
        const float tile_max = wave_max(s);
        const float m_new = fmaxf(m, tile_max);
        // every tile holds at least one visible key; were its page missing, m_new could still be -inf
        const float alpha = (m_new == -INFINITY) ? 1.f : expf(m - m_new);
        const float p = (s == -INFINITY) ? 0.f : expf(s - m_new);
        l = l * alpha + wave_sum(p);
        m = m_new;
        p_s[lane] = p;
        v_s[lane] = vbase;
        __syncthreads();
        const int nkeys = min(PULSE_WAVE, total - u0);
#pragma unroll
        for (int r = 0; r < MAX_ACC; ++r) {
            const int e = lane + r * PULSE_WAVE;
            if (e < width) {
                float sum = 0.f;
                for (int jj = 0; jj < nkeys; ++jj) {
                    const long long vb = v_s[jj];
                    if (vb >= 0) sum = fmaf(p_s[jj], to_f32<TC>(vcache[vb + static_cast<int64_t>(e) * a.page_size]), sum);
                }
                acc[r] = acc[r] * alpha + sum;
            }
        }
        __syncthreads();
    }

    TO* orow = out + static_cast<int64_t>(t) * a.o_stride + static_cast<int64_t>(h) * width;
    // a sink is one more term of the softmax's denominator, exp(sink[h]), with no key and no value
    if (sink) {
        const float sk = sink[h];
        if (m == -INFINITY) { l = 1.f; }
        else if (sk > m) { l = l * expf(m - sk) + 1.f; const float f = expf(m - sk);
#pragma unroll
            for (int r = 0; r < MAX_ACC; ++r) acc[r] *= f; }
        else l += expf(sk - m);
    }
    float inv_l = l > 0.f ? 1.0f / l : 0.f;
    const TX* grow = gate ? gate + static_cast<int64_t>(t) * gate_stride : nullptr;
    if (grow && !a.gate_per_channel) inv_l *= 1.0f / (1.0f + expf(-to_f32<TX>(grow[h])));
#pragma unroll
    for (int r = 0; r < MAX_ACC; ++r) {
        const int e = lane + r * PULSE_WAVE;
        if (e < width) {
            float v = acc[r] * inv_l;
            if (grow && a.gate_per_channel && e < a.gate_width)
                v *= 1.0f / (1.0f + expf(-to_f32<TX>(grow[static_cast<int64_t>(h) * a.gate_width + e])));
            orow[e] = from_f32<TO>(v);
        }
    }
}

// ------------------------------------------------------------------ float32 rows on the matrix cores
// Attention of float32 queries to float32 pages: a workgroup of four wavefronts owns 16 rows of one kv head, `tp`
// consecutive tokens of `hp` heads each.  Keys go in blocks of 16 that start at multiples of 16, block b to wavefront
// b % 4, each of which keeps a running softmax of its own for every row; the four meet in LDS in their order.  Blocks and
// shares are counted from key 0, and a block that a row sees nothing of leaves its sums as they are, so a row's result
// does not depend on the rows beside it.
//
// S[key][row] = K Q^T comes out of v_mfma_f32_16x16x4_f32 with keys 4 g + e (g = lane / 16) of row lane % 16 in a lane,
// which is how the next product, out[channel][row] += V^T P, wants its column operand: the e-th instruction takes keys
// 4 g + e, and a value row of the cache (the slots of a page side by side a channel) is read four keys a lane.
//
// What bounds it: trips to memory (a block's keys and values are asked for together, 16 KB a wavefront for 128 channels).
// 333 tokens, 16 heads over 4 kv heads of 128: 279 us with a wavefront a (token, head), which fetches every key for every
// row, 28 us with this.
typedef __attribute__((ext_vector_type(4))) float f32x4;

// f over the values of the first sixteen lanes.
template <typename F>
__device__ __forceinline__ int of_sixteen(int v, F f) {
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false));    // (row_ror:8, then 4, 2, 1)
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x124, 0xf, 0xf, false));
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x122, 0xf, 0xf, false));
    v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x121, 0xf, 0xf, false));
    return __builtin_amdgcn_readfirstlane(v);
}

template <int DB>
__global__ __launch_bounds__(256, DB == 2 ? 5 : DB == 4 ? 4 : 1) void attn_rows_f32_kernel(const float* __restrict__ q, float* __restrict__ out,
                                                            const float* __restrict__ kcache,
                                                            const float* __restrict__ vcache,
                                                            const int* __restrict__ positions,
                                                            const int* __restrict__ token_entry,
                                                            const int* __restrict__ block_table,
                                                            const float* __restrict__ gate, int64_t gate_stride,
                                                            const float* __restrict__ sink, AttnArgs a, int tokens, int tp,
                                                            int hp, int takers) {
    constexpr int D = 16 * DB;
    __shared__ f32x4 acc_s[4][DB][PULSE_WAVE];
    __shared__ float m_s[4][16], l_s[4][16];

    const int group = a.nq / a.nkv;
    const int t0 = blockIdx.x * tp;
    const int kvh = blockIdx.y, parts = (group + hp - 1) / hp, turn = blockIdx.z / parts, first_head = blockIdx.z % parts * hp, h0 = kvh * group + first_head;
    const int lane = threadIdx.x % PULSE_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PULSE_WAVE);
    const int r = lane % 16, kg = lane / 16;
    const int t_end = min(t0 + tp, tokens);

    // A tile may hold tokens of several entries: every one's rows are a walk of their own, which begin where `begins` has a
    // bit, and the workgroups of the tile take them in turn.  (Lane i looks at the tile's i-th token.)
    const int n = t_end - t0, own = t0 + min(lane, n - 1);
    const int own_entry = token_entry[own], own_pos = positions[own];
    const int entry_before = __shfl_up(own_entry, 1, PULSE_WAVE);
    unsigned long long begins = __ballot(lane < n && (lane == 0 || own_entry != entry_before));
    if (turn > 0 && __popcll(begins) <= turn) return;       // (the first has a walk for sure and need not wait to know it)

    // this lane's row (a row past the end is row 0 of the tile, sees nothing and is not written)
    bool live = r / hp < tp && t0 + r / hp < t_end && first_head + r % hp < group;
    const int t = live ? t0 + r / hp : t0;
    const int h = live ? h0 + r % hp : h0;
    const int pos = live ? positions[t] : -1;
    int lo = a.chunk > 0 ? pos - pos % a.chunk : (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
    lo = live ? lo : 0;
    const int n_first = live ? min(a.keep_first, lo) : 0;
    const float* qrow = q + static_cast<int64_t>(t) * a.q_stride + static_cast<int64_t>(h) * D;
    f32x4 qf[DB], acc[DB];
#pragma unroll
    for (int c = 0; c < DB; ++c) {
        qf[c] = *reinterpret_cast<const f32x4*>(qrow + 16 * c + 4 * kg) * a.scale;
        acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float m = -INFINITY, l = 0.f;    // l: of this lane's keys

    auto block = [&](int b, const int* bt, bool in_entry) __attribute__((always_inline)) {
        const int key0 = 16 * b, pi = key0 / a.page_size;
        const int page = pi < a.bt_width ? bt[pi] : -1;
        if (page < 0 || page >= a.num_pages) return;
        const int slot = key0 % a.page_size;
        const int64_t pg = (static_cast<int64_t>(page) * a.nkv + kvh) * D * a.page_size;
        const float* krow = kcache + pg + static_cast<int64_t>(slot + r) * D + 4 * kg;
        const float* vrow = vcache + pg + static_cast<int64_t>(r) * a.page_size + slot + 4 * kg;
        f32x4 kf[DB], vf[DB];
#pragma unroll
        for (int c = 0; c < DB; ++c) kf[c] = *reinterpret_cast<const f32x4*>(krow + 16 * c);
#pragma unroll
        for (int c = 0; c < DB; ++c) vf[c] = *reinterpret_cast<const f32x4*>(vrow + static_cast<int64_t>(16 * c) * a.page_size);
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DB; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][e], qf[c][e], s, 0, 0, 0);
        bool seen[4], all = true;
        float top = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = key0 + 4 * kg + e;
            seen[e] = in_entry && j <= pos && (j >= lo || j < n_first);
            all = all && seen[e];
            if (a.cap > 0.f) s[e] = a.cap * tanhf(s[e] / a.cap);
            s[e] = seen[e] ? s[e] : -INFINITY;
            top = fmaxf(top, s[e]);
        }
        top = across_rows(top, LaneMax());
        const float m_new = fmaxf(m, top);
        const float alpha = m_new == -INFINITY ? 1.f : expf(m - m_new);
        f32x4 p;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[e] = s[e] == -INFINITY ? 0.f : expf(s[e] - m_new);
            sum += p[e];
        }
        l = l * alpha + sum;
        m = m_new;
#pragma unroll
        for (int c = 0; c < DB; ++c) acc[c] *= alpha;
        // A weight of 0 keeps an unseen key out of a row only while the key's value is finite.  Where rows differ in
        // what they see of the block (or its slots were never written), values that are not go row by row instead.
        const bool partly = __ballot(!all) != 0;
        bool odd = false;
        if (partly) {
#pragma unroll
            for (int c = 0; c < DB; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) odd = odd || !(fabsf(vf[c][e]) < INFINITY);
        }
        if (partly && __ballot(odd) != 0) {
            for (int row = 0; row < 16; ++row) {
                // what row `row` sees of this lane's four keys (lane 16 g + row holds it for keys 4 g + e)
                bool sees[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) sees[e] = (__ballot(seen[e]) >> (16 * kg + row)) & 1ull;
#pragma unroll
                for (int c = 0; c < DB; ++c) {
                    f32x4 one = acc[c];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        one = __builtin_amdgcn_mfma_f32_16x16x4f32(sees[e] ? vf[c][e] : 0.f, p[e], one, 0, 0, 0);
                    if (r == row) acc[c] = one;
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < DB; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[c][e], p[e], acc[c], 0, 0, 0);
        }
    };

    const int own_lo = a.chunk > 0 ? own_pos - own_pos % a.chunk : (a.window > 0 && own_pos - a.window + 1 > 0) ? own_pos - a.window + 1 : 0;
    bool took = false;
    for (int run = 0; begins != 0; ++run) {
        const int ia = __builtin_ctzll(begins);
        begins &= begins - 1;
        const int ib = begins != 0 ? __builtin_ctzll(begins) : n;
        if (run % takers != turn) continue;
        const bool in_walk = lane >= ia && lane < ib;
        int hi = in_walk ? own_pos : -1, low = in_walk ? own_lo : 0x7fffffff, kept = in_walk ? min(a.keep_first, own_lo) : 0;
        hi = of_sixteen(hi, [](int x, int y) { return max(x, y); });
        low = of_sixteen(low, [](int x, int y) { return min(x, y); });
        kept = of_sixteen(kept, [](int x, int y) { return max(x, y); });
        const int* bt = block_table + static_cast<int64_t>(__builtin_amdgcn_readlane(own_entry, ia)) * a.bt_width;
        const bool in_entry = t >= t0 + ia && t < t0 + ib;
        const int first = (kept + 15) / 16, from = max(low / 16, first), to = hi / 16;
        for (int b = wave; b < first && b <= to; b += 4) block(b, bt, in_entry);
        for (int b = from + ((wave - from) & 3); b <= to; b += 4) block(b, bt, in_entry);
        took = took || in_entry;
    }
    live = live && took;

    l = across_rows(l, LaneSum());
    if (kg == 0) {
        m_s[wave][r] = m;
        l_s[wave][r] = l;
    }
#pragma unroll
    for (int c = 0; c < DB; ++c) acc_s[wave][c][lane] = acc[c];
    __syncthreads();
    if (!live) return;
    float top = m_s[0][r];
#pragma unroll
    for (int w = 1; w < 4; ++w) top = fmaxf(top, m_s[w][r]);
    float factor[4], den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        factor[w] = m_s[w][r] == -INFINITY ? 0.f : expf(m_s[w][r] - top);
        den += l_s[w][r] * factor[w];
    }
    float rescale = 1.f;
    if (sink) {      // one more term of the denominator, exp(sink[h]), with no key and no value
        const float sk = sink[h];
        if (top == -INFINITY) { den = 1.f; }
        else if (sk > top) { rescale = expf(top - sk); den = den * rescale + 1.f; }
        else den += expf(sk - top);
    }
    float inv = den > 0.f ? 1.0f / den : 0.f;
    const float* grow = gate ? gate + static_cast<int64_t>(t) * gate_stride : nullptr;
    if (grow && !a.gate_per_channel) inv *= 1.0f / (1.0f + expf(-grow[h]));
    float* orow = out + static_cast<int64_t>(t) * a.o_stride + static_cast<int64_t>(h) * D;
#pragma unroll
    for (int c = 0; c < DB; ++c) {
        if (c % 4 != wave) continue;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < 4; ++w) v += acc_s[w][c][lane] * factor[w];     // (NaN stays NaN whatever its share weighs)
        v *= rescale * inv;
        const int ch = 16 * c + 4 * kg;
        if (grow && a.gate_per_channel) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ch + e < a.gate_width) v[e] *= 1.0f / (1.0f + expf(-grow[static_cast<int64_t>(h) * a.gate_width + ch + e]));
        }
        *reinterpret_cast<f32x4*>(orow + ch) = v;
    }
}

// Whether the kernel above takes a call (everything float32, own values): what its 16-byte accesses ask for.
bool rows_f32_takes(const AttnArgs& a, const void* q, const void* out, const void* kcache, const void* vcache) {
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return (a.d == 32 || a.d == 64 || a.d == 128 || a.d == 256) && a.page_size % 16 == 0 && !a.all_values && a.nkv < 65536 &&
           a.q_stride % 4 == 0 && a.o_stride % 4 == 0 && aligned(q) && aligned(out) && aligned(kcache) && aligned(vcache);
}

int launch_rows_f32(const void* q, void* out, const void* kcache, const void* vcache, const int* positions,
                    const int* token_entry, const int* block_table, const void* gate, int64_t gate_stride, const float* sink,
                    const AttnArgs& a, int tokens, hipStream_t stream) {
    const int group = a.nq / a.nkv;
    const int hp = group < 16 ? group : 16;
    // Few tokens (decoding) get a tile each: their keys are those of one request or another, and more tiles fill the chip.
    const int tp = tokens <= 64 ? 1 : 16 / hp;
    // More tokens may still be as many requests, whose walks one workgroup would do one behind the other (80 requests of 1,000
    // keys, 8 heads of 256 with keys of their own: 1,870 us): as many workgroups a tile as the chip has room for take them in
    // turn (398 us), and in a prompt, where a tile is one walk, all but the first of them leave at once.
    const int tiles = (tokens + tp - 1) / tp, z = (group + hp - 1) / hp;
    const int64_t walks = static_cast<int64_t>(tiles) * a.nkv * z, room = 8 * static_cast<int64_t>(pulse_compute_units());
    const int takers = static_cast<int>(walks * tp <= room ? tp : walks < room ? room / walks : 1);
    const dim3 grid(tiles, a.nkv, z * takers);     // (those that leave at once come last)
#define PULSE_ROWS_LAUNCH(DB)                                                                                            \
    hipLaunchKernelGGL((attn_rows_f32_kernel<DB>), grid, dim3(256), 0, stream, static_cast<const float*>(q),             \
                       static_cast<float*>(out), static_cast<const float*>(kcache), static_cast<const float*>(vcache),  \
                       positions, token_entry, block_table, static_cast<const float*>(gate), gate_stride, sink, a, tokens, \
                       tp, hp, takers)
    if (a.d == 32) PULSE_ROWS_LAUNCH(2);
    else if (a.d == 64) PULSE_ROWS_LAUNCH(4);
    else if (a.d == 128) PULSE_ROWS_LAUNCH(8);
    else PULSE_ROWS_LAUNCH(16);
#undef PULSE_ROWS_LAUNCH
    return 0;
}

template <typename TX, typename TC, typename TO>
int launch_generic(int acc, const void* q, void* out, const void* kcache, const void* vcache, const int* positions,
                   const int* token_entry, const int* block_table, const void* gate, int64_t gate_stride,
                   const float* sink, const AttnArgs& a, int tokens, size_t lds, hipStream_t stream) {
#define PULSE_GENERIC_LAUNCH(N)                                                                                      \
    hipLaunchKernelGGL((attn_generic_kernel<TX, TC, TO, N>), dim3(tokens, a.nq), dim3(64), lds, stream,              \
                       static_cast<const TX*>(q), static_cast<TO*>(out), static_cast<const TC*>(kcache),            \
                       static_cast<const TC*>(vcache), positions, token_entry, block_table,                         \
                       static_cast<const TX*>(gate), gate_stride, sink, a)
    if (acc <= 2) PULSE_GENERIC_LAUNCH(2);
    else if (acc <= 8) PULSE_GENERIC_LAUNCH(8);
    else PULSE_GENERIC_LAUNCH(32);
#undef PULSE_GENERIC_LAUNCH
    return 0;
}

}  // namespace

// `out_f32`: out is float32 whatever the storage type of q (required with `all_values`, whose rows are nkv * d wide).
extern "C" int pulse_attn_generic_ex(const void* q, int64_t q_stride, void* out, int64_t o_stride, int x_dtype,
                                     const void* kcache, const void* vcache, int c_dtype, const int* positions,
                                     const int* token_entry, const int* block_table, int bt_width, int tokens, int nq,
                                     int nkv, int d, int page_size, int num_pages, float scale, int window,
                                     const void* gate, int64_t gate_stride, int gate_width, const float* sink,
                                     float softcap, int keep_first, int all_values, int out_f32, int chunk,
                                     hipStream_t stream) {
    const int width = all_values ? nkv * d : d;
    PULSE_REQUIRE(tokens >= 0 && nq > 0 && nkv > 0 && d > 0, "attn_generic: bad sizes");
    PULSE_REQUIRE(nq % nkv == 0, "attn_generic: %d query heads are not a multiple of %d kv heads", nq, nkv);
    PULSE_REQUIRE(width <= PULSE_WAVE * 32, "attn_generic: head_dim %d gives %d value channels a query head, more than %d", d,
                  width, PULSE_WAVE * 32);
    PULSE_REQUIRE(nq < 65536, "attn_generic: at most 65535 query heads, got %d", nq);
    PULSE_REQUIRE(page_size > 0 && num_pages > 0 && bt_width > 0, "attn_generic: bad cache geometry");
    PULSE_REQUIRE(window >= 0 && keep_first >= 0, "attn_generic: negative window or kept keys");
    PULSE_REQUIRE(chunk >= 0 && (chunk == 0 || window == 0), "attn_generic: a window and chunks at once");
    PULSE_REQUIRE(!all_values || (out_f32 && !gate), "attn_generic: all values side by side come out in float32, ungated");
    PULSE_REQUIRE(q_stride >= static_cast<int64_t>(nq) * d && o_stride >= static_cast<int64_t>(nq) * width,
                  "attn_generic: row strides too small");
    PULSE_REQUIRE(pulse_dtype_ok(x_dtype) && pulse_dtype_ok(c_dtype), "attn_generic: bad dtype tag");
    PULSE_REQUIRE(q && out && kcache && vcache && positions && token_entry && block_table, "attn_generic: null pointer");
    PULSE_REQUIRE(gate_width >= 0 && gate_width <= d, "attn_generic: %d gated channels of a head of %d", gate_width, d);
    PULSE_REQUIRE(!gate || gate_stride >= static_cast<int64_t>(nq) * (gate_width ? gate_width : 1),
                  "attn_generic: the gate's rows are too short");
    PULSE_REQUIRE(softcap >= 0.f, "attn_generic: a negative score cap");
    if (tokens == 0) return 0;
    AttnArgs a;
    a.nq = nq; a.nkv = nkv; a.d = d; a.q_stride = q_stride; a.o_stride = o_stride;
    a.page_size = page_size; a.num_pages = num_pages; a.bt_width = bt_width; a.scale = scale; a.window = window; a.chunk = chunk;
    a.cap = softcap; a.gate_per_channel = gate_width > 0 ? 1 : 0; a.gate_width = gate_width;
    a.keep_first = window > 0 ? keep_first : 0; a.all_values = all_values ? 1 : 0;
    if (x_dtype == PULSE_F32 && c_dtype == PULSE_F32 && rows_f32_takes(a, q, out, kcache, vcache)) {
        launch_rows_f32(q, out, kcache, vcache, positions, token_entry, block_table, gate, gate_stride, sink, a, tokens, stream);
        PULSE_LAUNCH_CHECK("attn_generic");
        return 0;
    }
    const size_t lds = static_cast<size_t>(d) * sizeof(float) + PULSE_WAVE * sizeof(float) + PULSE_WAVE * sizeof(long long);
    const int acc = (width + PULSE_WAVE - 1) / PULSE_WAVE;
    PULSE_DISPATCH_DTYPE(x_dtype, TX, PULSE_DISPATCH_DTYPE(c_dtype, TC,
        if (out_f32) launch_generic<TX, TC, float>(acc, q, out, kcache, vcache, positions, token_entry, block_table, gate,
                                                   gate_stride, sink, a, tokens, lds, stream);
        else launch_generic<TX, TC, TX>(acc, q, out, kcache, vcache, positions, token_entry, block_table, gate,
                                        gate_stride, sink, a, tokens, lds, stream)));
    PULSE_LAUNCH_CHECK("attn_generic");
    return 0;
}

extern "C" int pulse_attn_generic(const void* q, int64_t q_stride, void* out, int64_t o_stride, int x_dtype,
                                  const void* kcache, const void* vcache, int c_dtype, const int* positions,
                                  const int* token_entry, const int* block_table, int bt_width, int tokens, int nq,
                                  int nkv, int d, int page_size, int num_pages, float scale, int window,
                                  const void* gate, int64_t gate_stride, int gate_width, const float* sink,
                                  float softcap, hipStream_t stream) {
    return pulse_attn_generic_ex(q, q_stride, out, o_stride, x_dtype, kcache, vcache, c_dtype, positions, token_entry,
                                 block_table, bt_width, tokens, nq, nkv, d, page_size, num_pages, scale, window, gate,
                                 gate_stride, gate_width, sink, softcap, 0, 0, 0, 0, stream);
}
