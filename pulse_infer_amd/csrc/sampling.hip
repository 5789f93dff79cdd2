// Choosing the next token from float32 logits, one workgroup per row.
//
// The steps and their order are the reference sampler's
// (reference: demo/qwen3_infer.cpp:230-423):
//   1. presence penalty: subtract it from every token the request has seen;
//   2. banned ids are removed;
//   3. temperature <= 0: the largest logit wins, the lowest index among equals
//      (reference: src/scheduler/continuous_batch_engine.cpp:20-62);
//   4. top-k: keep the k largest;
//   5. weights exp((l - max) / temperature);
//   6. top-p in (0, 1): keep the most likely tokens whose mass first reaches
//      top_p of the total;
//   7. draw: u * (kept mass), walked along the cumulative sum.
// With top-k (or top-p alone on a peaked row) the row is read three times: the maximum, a histogram of the values
// that locates the k-th largest, and the collection of what lies at or above its bin; the rest happens on that
// short list in LDS.  Rows that do not fit (many equal values, a flat row under top-p alone) take passes over the
// whole vocabulary for their threshold, with the same result.
// Differences, both of measure zero or none in distribution: the kept sets are
// found as thresholds (tokens equal to the threshold are all kept), and the
// cumulative walk runs in vocabulary order rather than sorted order.  The
// uniform number u comes from the host's per-request counter-based generator,
// so a row's result does not depend on the other rows.
#include "common.h"
#include "no_alloc.h"

#include <math.h>

#include <mutex>

namespace {

constexpr int SAMPLE_THREADS = 1024;
constexpr int SAMPLE_WAVES = SAMPLE_THREADS / PULSE_WAVE;

__device__ __forceinline__ uint32_t order_key(float f) {
    if (f != f) return 0u;  // NaN sorts lowest
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

struct RowView {
    const float* logits;
    const uint32_t* seen;    // bit per token, or null
    const uint32_t* banned;  // bit per token, or null
    float penalty;
    int vocab;
    __device__ __forceinline__ bool masked() const { return seen != nullptr || banned != nullptr; }
    // The value of entry i; MASKED is masked(), asked once before a loop: a branch on either pointer beside every load would
    // have each load waited for before the next is issued.  (A row that has one of the masks reads it in both's place.)
    template <bool MASKED>
    __device__ __forceinline__ float at(int i) const {
        const float x = logits[i];
        if constexpr (!MASKED) return x != x ? -INFINITY : x;
        const uint32_t bit = 1u << (i & 31);
        const uint32_t b = (banned ? banned : seen)[i >> 5], s = (seen ? seen : banned)[i >> 5];
        const bool out = banned != nullptr && (b & bit) != 0u, was = seen != nullptr && (s & bit) != 0u;
        return (out || x != x) ? -INFINITY : (was ? x - penalty : x);
    }
};

template <bool V>
struct Is { static constexpr bool value = V; };
template <int V>
struct Int { static constexpr int value = V; };

// f(Is<row.masked()>)
template <typename F>
__device__ __forceinline__ void by_mask(const RowView& row, F f) {
    if (row.masked()) f(Is<true>());
    else f(Is<false>());
}

// f(i, value) for i = first, first + step, .. below end, in that order; the values of AHEAD entries are asked for
// before the first is used (a workgroup alone on its row otherwise waits out a trip to memory for every entry).  32 rows of
// 151,936 with all options among them: 565 us with the masks' branches beside every load, 503 without.  MOST: entries ahead
// in a row without masks, no more than a thread has.
template <int MOST = 16, typename F>
__device__ __forceinline__ void sweep(const RowView& row, int first, int end, int step, F f) {
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        constexpr int AHEAD = MASKED ? 8 : MOST;
        int i = first;
        for (; i + (AHEAD - 1) * step < end; i += AHEAD * step) {
            float x[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) x[u] = row.at<MASKED>(i + u * step);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) f(i + u * step, x[u]);
        }
        if (i < end) {        // what is left, asked for together too (past the end: the last entry again, for nobody)
            float x[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) x[u] = row.at<MASKED>(min(i + u * step, end - 1));
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (i + u * step < end) f(i + u * step, x[u]);
        }
    });
}

__device__ float block_sum_f(float v, float* scratch) { return block_sum(v, scratch); }

__device__ float block_max_f(float v, float* scratch) {
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float m = scratch[0];
    for (int w = 1; w < SAMPLE_WAVES; ++w) m = fmaxf(m, scratch[w]);
    return m;
}

__device__ int block_sum_i(int v, int* scratch) {
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    int total = 0;
    for (int w = 0; w < SAMPLE_WAVES; ++w) total += scratch[w];
    return total;
}

// (value, index) maximum with the lowest index among equal values
__device__ void block_argmax(float& v, int& idx, float* sv, int* si) {
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    wave_argmax(v, idx);
    __syncthreads();
    if (lane == 0) { sv[wave] = v; si[wave] = idx; }
    __syncthreads();
    v = sv[0]; idx = si[0];
    for (int w = 1; w < SAMPLE_WAVES; ++w)
        if (sv[w] > v || (sv[w] == v && si[w] < idx)) { v = sv[w]; idx = si[w]; }
}

// ---- the walk along the cumulative sum, a wavefront over 64 consecutive entries at a time ---------------------
// `weight(i)` is the weight of entry i of [begin, end) (0 for what is not kept), entries in vocabulary order.  The
// wavefront finds the first entry at which the running sum exceeds `rest` and returns its number, or -1 if the sum
// never gets there (rounding); `last` is the last entry with a weight.  Every lane returns the same.
template <typename Weight>
__device__ int wave_walk(int begin, int end, float rest, Weight weight, int& last) {
    const int lane = threadIdx.x % PULSE_WAVE;
    constexpr int AHEAD = 16;  // steps of 64 entries whose weights are asked for together (a step's trip to memory
                               // would otherwise be waited for before the next one starts)
    float run = 0.f;
    last = -1;
    for (int first = begin; first < end; first += AHEAD * PULSE_WAVE) {
        float ws[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int i = first + u * PULSE_WAVE + lane;
            ws[u] = i < end ? weight(i) : 0.f;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int base = first + u * PULSE_WAVE;
            const float w = ws[u];
            const unsigned long long has = __ballot(w > 0.f);
            if (has == 0ull) continue;
            last = base + (63 - __builtin_clzll(has));
            // inclusive prefix over the lanes, in lane order
            float pre = w;
#pragma unroll
            for (int off = 1; off < PULSE_WAVE; off <<= 1) {
                const float up = __shfl_up(pre, off, PULSE_WAVE);
                if (lane >= off) pre += up;
            }
            const unsigned long long hit = __ballot(w > 0.f && rest < run + pre);
            if (hit != 0ull) return base + __builtin_ctzll(hit);
            run += __shfl(pre, PULSE_WAVE - 1, PULSE_WAVE);
        }
    }
    return -1;
}

constexpr int HIST_BINS = 2048;                         // bins of the value histogram that locates the k-th largest
constexpr int WAVE_CAP = 128;                           // candidates a wavefront may collect
constexpr int LIST_CAP = SAMPLE_WAVES * WAVE_CAP;       // candidates of a row
constexpr int LIST_PER_LANE = LIST_CAP / PULSE_WAVE;

// The end of the choice on a short list in LDS, by one wavefront: `n` candidates in vocabulary order (`list_i`, their
// values `list_x`, which are overwritten), among them every token that top-k keeps.  The k-th largest value by a
// search bit by bit, then top-p on what that kept (relative to its mass; without top-k relative to `whole`, the mass
// of the whole row, and only if the list holds that much: else false and nothing is chosen), then the walk along the
// cumulative sum.  Every lane returns the same.  PER: entries a lane takes (n <= PER * 64).
template <int PER>
__device__ bool finish_on_list(const int* list_i, float* list_x, int n, bool by_k, int k, bool use_p, float p, float whole,
                               float best, float inv_t, float u, int best_i, int& token) {
    const int lane = threadIdx.x % PULSE_WAVE;
    uint32_t keys[PER];
    float wts[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = lane + j * PULSE_WAVE;
        keys[j] = e < n ? order_key(list_x[e]) : 0u;
        wts[j] = e < n ? expf((list_x[e] - best) * inv_t) : 0.f;
    }
    // the k-th largest key, bit by bit
    uint32_t keep = 0u;
    if (by_k) {
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = keep | (1u << bit);
            int c = 0;
#pragma unroll
            for (int j = 0; j < PER; ++j) c += (lane + j * PULSE_WAVE < n && keys[j] >= cand) ? 1 : 0;
            if (wave_sum(c) >= k) keep = cand;
        }
    }
    if (use_p) {
        float mass = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) mass += keys[j] >= keep ? wts[j] : 0.f;
        mass = wave_sum(mass);
        const float want = p * (by_k ? mass : whole);
        if (!by_k && !(mass >= want)) return false;   // without top-k the list must hold all of the top_p set
        uint32_t thr = 0u;
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = thr | (1u << bit);
            const uint32_t lim = cand > keep ? cand : keep;
            float part_mass = 0.f;
#pragma unroll
            for (int j = 0; j < PER; ++j) part_mass += keys[j] >= lim ? wts[j] : 0.f;
            if (wave_sum(part_mass) >= want) thr = cand;
        }
        if (thr > keep) keep = thr;
    }
    // what is kept, as weights in the list's place of x, then the walk
    float kept = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = lane + j * PULSE_WAVE;
        const float w = (e < n && keys[j] >= keep) ? wts[j] : 0.f;
        if (e < n) list_x[e] = w;
        kept += w;
    }
    kept = wave_sum(kept);
    int last;
    const int e = wave_walk(0, n, u * kept, [&](int q) { return list_x[q]; }, last);
    token = e >= 0 ? list_i[e] : (last >= 0 ? list_i[last] : best_i);
    return true;
}

// What the kernels in front of sample_kernel leave of a row that the chunks could not choose for: the histogram's counts and
// masses, then the mass of each of sample_kernel's wavefronts (as it would sum it) and the smallest number of each.
constexpr int REST_MASS = 2 * HIST_BINS, REST_LOWEST = REST_MASS + SAMPLE_WAVES;
constexpr int REST_WORDS = REST_LOWEST + SAMPLE_WAVES;

__device__ __forceinline__ void add_in_group(float* p, float v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

constexpr int CANDIDATES = 15;   // most thresholds whose masses are summed side by side in a pass

// The largest threshold t with M(t) >= want (see sample_kernel), from the histogram of a row under top-p alone; false where
// the bracket does not hold it (or too many tokens share the bins), and then nothing is said.  Called by a whole workgroup.
__device__ bool nucleus_edge(const RowView& row, float want, float best, float inv_t, float scale, const int* hist,
                             const float* hist_w, float* sf, int* si, int* list_i, float* list_x, uint32_t* cand,
                             unsigned long long* nearest, uint32_t& thr) {
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    // the first bin at which the masses from the top reach `want`: thread t sums bins 2 t and 2 t + 1
    constexpr int PER = HIST_BINS / SAMPLE_THREADS;
    static_assert(PER == 2, "two bins a thread");
    const float w0 = hist_w[2 * threadIdx.x], w1 = hist_w[2 * threadIdx.x + 1];
    float pre = w0 + w1;
#pragma unroll
    for (int off = 1; off < PULSE_WAVE; off <<= 1) {
        const float up = __shfl_up(pre, off, PULSE_WAVE);
        if (lane >= off) pre += up;
    }
    __syncthreads();
    if (lane == PULSE_WAVE - 1) sf[wave] = pre;
    if (threadIdx.x == 0) { si[0] = HIST_BINS; si[1] = 0; *nearest = ~0ull; }
    __syncthreads();
    float before = 0.f;
    for (int w = 0; w < wave; ++w) before += sf[w];
    const float through1 = before + pre, through0 = through1 - w1;     // masses through this thread's bins
    if (through0 >= want) atomicMin(&si[0], 2 * static_cast<int>(threadIdx.x));
    else if (through1 >= want) atomicMin(&si[0], 2 * static_cast<int>(threadIdx.x) + 1);
    __syncthreads();
    const int at = si[0];
    if (at >= HIST_BINS) return false;
    const int b0 = max(0, at - 1), b1 = min(HIST_BINS - 1, at + 1);
    int count = 0;
    for (int b = b0; b <= b1; ++b) count += hist[b];
    if (count > LIST_CAP) return false;
    float mine = 0.f;
    for (int b = threadIdx.x; b < b0; b += SAMPLE_THREADS) mine += hist_w[b];
    const float base = block_sum_f(mine, sf);       // the mass above the three bins
    // their tokens, in any order: keys and weights
    sweep(row, threadIdx.x, row.vocab, SAMPLE_THREADS, [&](int, float x) {
        if (x == -INFINITY) return;
        const int b = min(HIST_BINS - 1, static_cast<int>((best - x) * scale));
        if (b < b0 || b > b1) return;
        const int e = atomicAdd(&si[1], 1);
        if (e < LIST_CAP) {
            list_i[e] = static_cast<int>(order_key(x));
            list_x[e] = expf((x - best) * inv_t);
        }
    });
    __syncthreads();
    const int n = si[1];
    if (n > LIST_CAP || n == 0) return false;
    // every token's place among them and the mass through it; of those that reach `want`, the one placed first
    int place[LIST_CAP / SAMPLE_THREADS];
    uint32_t keys[LIST_CAP / SAMPLE_THREADS];
#pragma unroll
    for (int u = 0; u < LIST_CAP / SAMPLE_THREADS; ++u) {
        const int e = threadIdx.x + u * SAMPLE_THREADS;
        place[u] = -1;
        keys[u] = 0u;
        if (e >= n) continue;
        const uint32_t key = static_cast<uint32_t>(list_i[e]);
        float through = base;
        int higher = 0;
        for (int j = 0; j < n; ++j) {
            const uint32_t other = static_cast<uint32_t>(list_i[j]);
            through += other >= key ? list_x[j] : 0.f;
            higher += other > key ? 1 : 0;
        }
        place[u] = higher;
        keys[u] = key;
        if (through >= want) atomicMin(nearest, static_cast<unsigned long long>(higher));
    }
    __syncthreads();
    if (*nearest == ~0ull) return false;
    // M at the places round that one.  The histogram's masses are good to a few units in the last place of the whole, which is
    // less than a token there unless the row is very flat: two places to either side first, seven where those do not hold it.
    auto try_round = [&](auto count) __attribute__((always_inline)) {
        constexpr int C = decltype(count)::value;
        const int first = static_cast<int>(*nearest) - C / 2;
        __syncthreads();
        if (threadIdx.x < C) cand[threadIdx.x] = 0u;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < LIST_CAP / SAMPLE_THREADS; ++u)
            if (place[u] >= first && place[u] >= 0 && place[u] < first + C) cand[place[u] - first] = keys[u];
        __syncthreads();
        // (equal tokens share a place, and the places behind it stay empty: 0)
        uint32_t t[C], least = 0xffffffffu;
        float above[C];
#pragma unroll
        for (int j = 0; j < C; ++j) {
            t[j] = cand[j];
            above[j] = 0.f;
            if (t[j] != 0u && t[j] < least) least = t[j];
        }
        sweep(row, threadIdx.x, row.vocab, SAMPLE_THREADS, [&](int, float x) {
            if (x == -INFINITY) return;
            const uint32_t key = order_key(x);
            if (key < least) return;
            const float w = expf((x - best) * inv_t);
#pragma unroll
            for (int j = 0; j < C; ++j)
                if (key >= t[j]) above[j] += w;
        });
        bool below = false, found = false, open = true;      // a larger candidate's mass falls short; the first that does not is known
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const float m = block_sum_f(above[j], sf);
            if (t[j] == 0u || found || !open) continue;
            if (m < want) below = true;
            else if (below) { found = true; thr = t[j]; }
            else open = false;                               // (the same for every thread)
        }
        return found;
    };
    return try_round(Int<5>()) || try_round(Int<CANDIDATES>());
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, int* __restrict__ out, const int* __restrict__ done,
    const float* __restrict__ part_max, const int* __restrict__ part_idx, int chunks, const int* __restrict__ rest) {
    __shared__ float sf[SAMPLE_WAVES];
    __shared__ int si[SAMPLE_WAVES];
    __shared__ int hist[HIST_BINS];
    __shared__ float hist_w[HIST_BINS];     // top-p alone: the bins' masses (in the order of arrival: good for a bracket)
    if (done && done[blockIdx.x]) return;   // the kernels that work in chunks have chosen this row's token already
    __shared__ int wave_bins[SAMPLE_WAVES];
    __shared__ int region_i[SAMPLE_WAVES][WAVE_CAP];
    __shared__ float region_x[SAMPLE_WAVES][WAVE_CAP];
    __shared__ int region_n[SAMPLE_WAVES];
    __shared__ int list_i[LIST_CAP];
    __shared__ float list_x[LIST_CAP];
    __shared__ float part_sum[SAMPLE_WAVES];
    __shared__ int list_done;
    __shared__ uint32_t cand[CANDIDATES];
    __shared__ unsigned long long nearest;

    const int r = blockIdx.x;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    RowView row;
    row.logits = logits + r * row_stride;
    row.vocab = vocab;
    row.banned = banned;
    row.penalty = penalty ? penalty[r] : 0.f;
    row.seen = (seen_masks && seen_row && seen_row[r] >= 0 && row.penalty > 0.f)
                   ? seen_masks + static_cast<int64_t>(seen_row[r]) * mask_words : nullptr;

    // largest logit, lowest index among equals (from the chunks' where the kernels before left them); the smallest number
    // too (the histogram's range), here or with the mass below
    float best = -INFINITY, lowest = INFINITY;
    int best_i = 0x7fffffff;
    if (part_max) {
        for (int c = threadIdx.x; c < chunks; c += SAMPLE_THREADS) {
            const float v = part_max[static_cast<int64_t>(r) * chunks + c];
            const int i = part_idx[static_cast<int64_t>(r) * chunks + c];
            if (v > best || (v == best && i < best_i)) { best = v; best_i = i; }
        }
    } else {
        sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int i, float x) {
            if (x > best) { best = x; best_i = i; }
        });
    }
    block_argmax(best, best_i, sf, si);
    if (best_i == 0x7fffffff) {  // everything banned or NaN
        if (threadIdx.x == 0) out[r] = -1;
        return;
    }
    const float temp = temperature ? temperature[r] : 0.f;
    if (!(temp > 0.f)) {
        if (threadIdx.x == 0) out[r] = best_i;
        return;
    }
    const float inv_t = 1.0f / temp;
    const int k = top_k ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 0.f;
    const bool use_p = p > 0.f && p < 1.f;
    // each wavefront owns a contiguous part of the vocabulary, walked 64 entries at a time
    const int part = ((vocab + SAMPLE_WAVES - 1) / SAMPLE_WAVES + PULSE_WAVE - 1) / PULSE_WAVE * PULSE_WAVE;
    const int part_begin = min(vocab, wave * part), part_end = min(vocab, wave * part + part);

    // ---- with top-k: locate the k-th largest with a histogram over [lowest, best], collect what lies at or above
    // its bin (in vocabulary order), and finish on that short list in LDS.  Falls through to the passes over the
    // whole vocabulary when the list would not fit (many equal values) or the range is empty.
    // Top-p alone takes the same way with the LIST_TRY largest values, if their mass reaches top_p of the whole.
    constexpr int LIST_TRY = 1024;
    const bool by_k = k > 0 && k < vocab;
    const int k_list = by_k ? k : min(vocab - 1, LIST_TRY);
    float whole = 0.f;   // without top-k: the mass of the whole vocabulary, which top_p refers to
    float bin_scale = 0.f;
    if (by_k || (use_p && k_list > 0)) {
        if (rest) {      // (the kernels before have been over the row for both, and for the histogram)
            rest += static_cast<int64_t>(r) * REST_WORDS;
            for (int w = 0; w < SAMPLE_WAVES; ++w) whole += __int_as_float(rest[REST_MASS + w]);
            lowest = __int_as_float(rest[REST_LOWEST + threadIdx.x % SAMPLE_WAVES]);
        } else if (!by_k) {
            float mass = 0.f;
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                if (x != -INFINITY) { mass += expf((x - best) * inv_t); lowest = fminf(lowest, x); }
            });
            whole = block_sum_f(mass, sf);
        } else {
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                if (x != -INFINITY) lowest = fminf(lowest, x);
            });
        }
        lowest = -block_max_f(-lowest, sf);
        const float scale = static_cast<float>(HIST_BINS) / (best - lowest);
        const bool ranged = best > lowest && scale < INFINITY;
        auto bin_of = [&](float x) { return min(HIST_BINS - 1, static_cast<int>((best - x) * scale)); };  // 0: the largest values
        int edge = -1, listed = 0;
        if (ranged) {
            for (int b = threadIdx.x; b < HIST_BINS; b += SAMPLE_THREADS) {
                hist[b] = rest ? rest[b] : 0;
                if (!by_k) hist_w[b] = rest ? __int_as_float(rest[HIST_BINS + b]) : 0.f;
            }
            __syncthreads();
            if (!rest) {
                sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    if (x != -INFINITY) atomicAdd(&hist[bin_of(x)], 1);
                });
                __syncthreads();
            }
            if (!by_k) bin_scale = scale;
            // the bin in which the count from the top reaches k: first by wavefronts' shares of the bins, then by bins
            constexpr int SHARE = HIST_BINS / SAMPLE_WAVES;
            int mine = 0;
            for (int b = wave * SHARE + lane; b < (wave + 1) * SHARE; b += PULSE_WAVE) mine += hist[b];
            mine = wave_sum(mine);
            if (lane == 0) wave_bins[wave] = mine;
            __syncthreads();
            int w = 0;
            while (w < SAMPLE_WAVES && listed + wave_bins[w] < k_list) listed += wave_bins[w++];
            if (w < SAMPLE_WAVES) {
                int b = w * SHARE;
                while (listed + hist[b] < k_list) listed += hist[b++];
                listed += hist[b];
                edge = b;
            }
        }
        bool may_hold = true;    // whether the list can hold top_p of the row (its mass is known to a thousandth at least)
        if (rest && !by_k && edge >= 0) {
            float above = 0.f;
            for (int b = threadIdx.x; b <= edge; b += SAMPLE_THREADS) above += hist_w[b];
            may_hold = block_sum_f(above, sf) >= 0.999f * p * whole;
        }
        if (edge >= 0 && listed <= LIST_CAP && may_hold) {
            int count = 0;
            by_mask(row, [&](auto masked) __attribute__((always_inline)) {
            constexpr int AHEAD = 8;   // steps of 64 entries whose values are asked for together
            for (int base = part_begin; base < part_end; base += AHEAD * PULSE_WAVE) {
                float xs[AHEAD];
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const int i = base + u * PULSE_WAVE + lane;
                    xs[u] = i < part_end ? row.at<decltype(masked)::value>(i) : -INFINITY;
                }
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const int i = base + u * PULSE_WAVE + lane;
                    const float x = xs[u];
                    const bool in = x != -INFINITY && bin_of(x) <= edge;
                    const unsigned long long mask = __ballot(in);
                    const int at = count + __builtin_popcountll(mask & ((1ull << lane) - 1ull));
                    if (in && at < WAVE_CAP) { region_i[wave][at] = i; region_x[wave][at] = x; }
                    count += __builtin_popcountll(mask);
                }
            }
            });
            if (lane == 0) region_n[wave] = count;
            __syncthreads();
            bool fits = true;
            for (int w = 0; w < SAMPLE_WAVES; ++w) fits = fits && region_n[w] <= WAVE_CAP;
            if (fits) {
                // one list, in vocabulary order
                int n = 0;
                for (int w = 0; w < SAMPLE_WAVES; ++w) {
                    for (int e = threadIdx.x; e < region_n[w]; e += SAMPLE_THREADS) {
                        list_i[n + e] = region_i[w][e];
                        list_x[n + e] = region_x[w][e];
                    }
                    n += region_n[w];
                }
                __syncthreads();
                // the first wavefront finishes alone (lane l holds entries l, l + 64, ..); the others wait for its word
                if (wave == 0) {
                    int token;
                    const bool enough = n <= 8 * PULSE_WAVE
                        ? finish_on_list<8>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, uniform[r], best_i, token)
                        : finish_on_list<LIST_PER_LANE>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, uniform[r],
                                                        best_i, token);
                    if (lane == 0) {
                        if (enough) out[r] = token;   // else (only without top-k) the list is too short: the passes
                        list_done = enough ? 1 : 0;   // over the whole vocabulary
                    }
                }
                __syncthreads();
                if (list_done) return;
            }
        }
    }

    // ---- passes over the whole vocabulary
    // top-k threshold: the k-th largest key, found bit by bit
    uint32_t keep = 0u;
    if (k > 0 && k < vocab) {
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = keep | (1u << bit);
            int count = 0;
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) { count += order_key(x) >= cand; });
            if (block_sum_i(count, si) >= k) keep = cand;
        }
    }
    auto weight_of = [&](float x) { return (x != -INFINITY && order_key(x) >= keep) ? expf((x - best) * inv_t) : 0.f; };
    if (use_p) {
        // M(t), the mass at or above a threshold t as this kernel sums it (every thread its entries in their order, then the
        // threads): no larger for a larger t, so the largest t with M(t) >= want is one value however it is looked for.
        uint32_t thr = 0u;
        bool found = false;
        float want;
        if (!by_k && bin_scale > 0.f) {
            // Top-p alone: the histogram's masses say near which token the sum reaches `want`; the tokens of that bin and
            // its neighbours are ranked, and M is summed, in its own order, for the five (or fifteen) round that place side by side.
            // (A search for the threshold's bits, four a pass, takes eight such passes.  32 rows of 151,936, this kernel:
            // 661 us with the search, 377 with this, 141 with the mass and the histogram made by the kernels in front.  The masses
            // are summed for the rows that come here alone: every row's cost those whose list holds top_p 1.7 to 2.5 times.)
            want = p * whole;
            if (!rest) {
                sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    if (x != -INFINITY)
                        add_in_group(&hist_w[min(HIST_BINS - 1, static_cast<int>((best - x) * bin_scale))], expf((x - best) * inv_t));
                });
                __syncthreads();
            }
            found = nucleus_edge(row, want, best, inv_t, bin_scale, hist, hist_w, sf, si, list_i, list_x, cand, &nearest, thr);
        } else {
            float mass = 0.f;
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) { mass += weight_of(x); });
            want = p * block_sum_f(mass, sf);
        }
        // Else the largest threshold whose kept mass still reaches `want`, four bits of it a pass over the row: the masses
        // above the fifteen candidates of a digit are summed side by side (each in the order in which a pass for it
        // alone would sum it, so the choice is that of a search bit by bit, in an eighth of the passes).
        if (!found) thr = 0u;
        for (int shift = 28; shift >= 0 && !found; shift -= 4) {
            float above[15];
#pragma unroll
            for (int j = 0; j < 15; ++j) above[j] = 0.f;
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                if (x == -INFINITY) return;
                const uint32_t key = order_key(x);
                if (key < keep || key < (thr | (1u << shift))) return;
                const float w = expf((x - best) * inv_t);
#pragma unroll
                for (int j = 0; j < 15; ++j)
                    if (key >= (thr | (static_cast<uint32_t>(j + 1) << shift))) above[j] += w;
            });
            uint32_t digit = 0u;
#pragma unroll
            for (int j = 0; j < 15; ++j)
                if (block_sum_f(above[j], sf) >= want) digit = static_cast<uint32_t>(j + 1);
            thr |= digit << shift;
        }
        if (thr > keep) keep = thr;
    }
    // the kept mass of every wavefront's part, then the part in which the draw falls is walked by its wavefront
    float mine = 0.f;
    sweep(row, part_begin + lane, part_end, PULSE_WAVE, [&](int, float x) { mine += weight_of(x); });
    mine = wave_sum(mine);
    if (lane == 0) part_sum[wave] = mine;
    __syncthreads();
    float kept = 0.f;
    for (int w = 0; w < SAMPLE_WAVES; ++w) kept += part_sum[w];
    const float target = uniform[r] * kept;
    float run = 0.f;
    int who = -1, last_part = -1;
    for (int w = 0; w < SAMPLE_WAVES; ++w) {
        if (part_sum[w] > 0.f) {
            last_part = w;
            if (who < 0 && target < run + part_sum[w]) who = w;
        }
        if (who < 0) run += part_sum[w];
    }
    if (who < 0) {  // rounding left the target beyond the last part: its last kept entry
        who = last_part;
        run = INFINITY;
    }
    if (wave != who) return;
    int last, e;
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
        e = wave_walk(part_begin, part_end, run == INFINITY ? INFINITY : target - run,
                      [&](int i) { return weight_of(row.at<decltype(masked)::value>(i)); }, last);
    });
    if (lane == 0) out[r] = e >= 0 ? e : (last >= 0 ? last : best_i);
}

__global__ void mark_seen_kernel(uint32_t* __restrict__ masks, int mask_words, const int* __restrict__ rows,
                                 const int* __restrict__ tokens, int n, int vocab) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int tok = tokens[i];
    if (tok < 0 || tok >= vocab || rows[i] < 0) return;
    atomicOr(masks + static_cast<int64_t>(rows[i]) * mask_words + (tok >> 5), 1u << (tok & 31));
}

// Greedy choice in two stages so that a few rows of a large vocabulary use the whole chip:
// each workgroup scans one chunk of a row, then one workgroup per row merges the chunk winners.
constexpr int ARGMAX_THREADS = 256;

__global__ __launch_bounds__(ARGMAX_THREADS) void argmax_chunks_kernel(const float* __restrict__ logits, int vocab,
                                                                       int64_t row_stride, int chunk,
                                                                       float* __restrict__ part_val,
                                                                       int* __restrict__ part_idx) {
    __shared__ float sv[ARGMAX_THREADS / PULSE_WAVE];
    __shared__ int si[ARGMAX_THREADS / PULSE_WAVE];
    const int r = blockIdx.y;
    const int begin = blockIdx.x * chunk;
    const int end = min(vocab, begin + chunk);
    const float* row = logits + r * row_stride;
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    for (int i = begin + threadIdx.x; i < end; i += ARGMAX_THREADS) {
        const float x = row[i];
        if (x > best) { best = x; best_i = i; }   // NaN never wins; ascending i keeps the lowest index among equals
    }
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    wave_argmax(best, best_i);
    if (lane == 0) { sv[wave] = best; si[wave] = best_i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < ARGMAX_THREADS / PULSE_WAVE; ++w)
            if (sv[w] > best || (sv[w] == best && si[w] < best_i)) { best = sv[w]; best_i = si[w]; }
        part_val[r * gridDim.x + blockIdx.x] = best;
        part_idx[r * gridDim.x + blockIdx.x] = best_i;
    }
}

__global__ __launch_bounds__(PULSE_WAVE) void argmax_merge_kernel(const float* __restrict__ part_val,
                                                                  const int* __restrict__ part_idx, int chunks,
                                                                  int* __restrict__ out) {
    const int r = blockIdx.x;
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    for (int c = threadIdx.x; c < chunks; c += PULSE_WAVE) {
        const float v = part_val[r * chunks + c];
        const int i = part_idx[r * chunks + c];
        if (v > best || (v == best && i < best_i)) { best = v; best_i = i; }
    }
    wave_argmax(best, best_i);
    if (threadIdx.x == 0) out[r] = best_i == 0x7fffffff ? -1 : best_i;
}

// ---- rows in chunks ----------------------------------------------------------------------------------------------
// A workgroup a row reads its row at the rate of one compute unit.  Without top-k and top-p nothing has to be
// known about the row as a whole but its maximum and its mass, so the row is cut into chunks of SIMPLE_CHUNK logits
// with a workgroup each: the chunk's maximum (with its lowest index); then, the row's maximum known, the chunk's
// mass; then one wavefront a row finds the chunk in which u * mass falls (chunk masses summed in chunk order) and
// walks that chunk alone (chunked_choose_kernel).  The steps and their meaning are those of sample_kernel; sums are
// taken in another order.
constexpr int SIMPLE_CHUNK = 2048;
constexpr int SIMPLE_THREADS = 256;

__device__ __forceinline__ RowView simple_row(const float* logits, int r, int64_t row_stride, int vocab,
                                              const float* penalty, const int* seen_row, const uint32_t* seen_masks,
                                              const uint32_t* banned, int mask_words) {
    RowView row;
    row.logits = logits + r * row_stride;
    row.vocab = vocab;
    row.banned = banned;
    row.penalty = penalty ? penalty[r] : 0.f;
    row.seen = (seen_masks && seen_row && seen_row[r] >= 0 && row.penalty > 0.f)
                   ? seen_masks + static_cast<int64_t>(seen_row[r]) * mask_words : nullptr;
    return row;
}

__global__ __launch_bounds__(SIMPLE_THREADS) void simple_max_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ penalty,
    const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned,
    int mask_words, float* __restrict__ part_max, int* __restrict__ part_idx, float* __restrict__ part_min) {
    __shared__ float sv[SIMPLE_THREADS / PULSE_WAVE];
    __shared__ int si[SIMPLE_THREADS / PULSE_WAVE];
    __shared__ float sl[SIMPLE_THREADS / PULSE_WAVE];
    const int r = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const int begin = chunk * SIMPLE_CHUNK, end = min(vocab, begin + SIMPLE_CHUNK);
    float best = -INFINITY, lowest = INFINITY;
    int best_i = 0x7fffffff;
    sweep<SIMPLE_CHUNK / SIMPLE_THREADS>(row, begin + static_cast<int>(threadIdx.x), end, SIMPLE_THREADS, [&](int i, float x) {
        if (x > best) { best = x; best_i = i; }   // a thread's indices rise: the first of equals stays
        if (x != -INFINITY) lowest = fminf(lowest, x);
    });
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    wave_argmax(best, best_i);
    if (part_min) lowest = -wave_max(-lowest);
    if (lane == 0) { sv[wave] = best; si[wave] = best_i; sl[wave] = lowest; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SIMPLE_THREADS / PULSE_WAVE; ++w)
            if (sv[w] > best || (sv[w] == best && si[w] < best_i)) { best = sv[w]; best_i = si[w]; }
        if (part_min) {
            for (int w = 1; w < SIMPLE_THREADS / PULSE_WAVE; ++w) lowest = fminf(lowest, sl[w]);
            part_min[r * chunks + chunk] = lowest;
        }
        part_max[r * chunks + chunk] = best;
        part_idx[r * chunks + chunk] = best_i;
    }
}

// The row's maximum from the chunks' (every lane gets it).
__device__ __forceinline__ float simple_row_max(const float* part_max, int chunks) {
    float best = -INFINITY;
    for (int c = threadIdx.x % PULSE_WAVE; c < chunks; c += PULSE_WAVE) best = fmaxf(best, part_max[c]);
    best = wave_max(best);
    return best;
}

__global__ __launch_bounds__(SIMPLE_THREADS) void simple_mass_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, const float* __restrict__ part_max,
    float* __restrict__ part_mass) {
    __shared__ float sf[SIMPLE_THREADS / PULSE_WAVE];
    const int r = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const float temp = temperature ? temperature[r] : 0.f;
    if (!(temp > 0.f)) return;   // the largest logit wins: no mass is asked for
    if (top_k && top_k[r] > 0) return;   // what top-k keeps is weighed on the short list
    const float best = simple_row_max(part_max + r * chunks, chunks);
    if (best == -INFINITY) return;
    const float inv_t = 1.0f / temp;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const int begin = chunk * SIMPLE_CHUNK, end = min(vocab, begin + SIMPLE_CHUNK);
    float mass = 0.f;
    sweep<SIMPLE_CHUNK / SIMPLE_THREADS>(row, begin + static_cast<int>(threadIdx.x), end, SIMPLE_THREADS, [&](int, float x) {
        if (x != -INFINITY) mass += expf((x - best) * inv_t);
    });
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    mass = wave_sum(mass);
    if (lane == 0) sf[wave] = mass;
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        for (int w = 0; w < SIMPLE_THREADS / PULSE_WAVE; ++w) total += sf[w];
        part_mass[r * chunks + chunk] = total;
    }
}

// ---- rows with top-k, in chunks -------------------------------------------------------------------------------
// With a small k the candidates can be found chunk by chunk as well.  The k-th largest of the chunks' maxima is a
// lower bound of the k-th largest logit (that many logits, the maxima themselves, reach it), so everything that
// top-k keeps lies at or above it, and little else: a workgroup a chunk collects what it has there, in vocabulary
// order, into its own short segment; a wavefront a row strings the segments together in LDS and finishes on that list
// as sample_kernel does on its own (finish_on_list).  A row that does not fit (k above the number of chunks, a chunk
// with more candidates than its segment holds: many equal values) is left to sample_kernel, which runs behind and
// skips the rows that are done.
constexpr int TOPK_SEGMENT = 32;   // candidates a chunk may leave

// A row with top-p alone takes the same way with what lies at or above one of the lower chunk maxima (seven eighths
// of the chunks have a larger one): some hundreds of the largest logits of a vocabulary of 150,000, which hold the
// top_p share of a distribution as peaked as a language model's; if they do not (or a chunk has more than its segment
// holds), the row is left to sample_kernel too.  The mass of the whole row, which top_p refers to, comes from
// simple_mass_kernel.
__device__ __forceinline__ int top_p_bound_rank(int chunks) { return max(1, chunks - chunks / 8); }

__global__ __launch_bounds__(SIMPLE_THREADS) void topk_collect_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ penalty,
    const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned,
    int mask_words, const float* __restrict__ part_max, int* __restrict__ seg_i, float* __restrict__ seg_x,
    int* __restrict__ seg_n) {
    constexpr int WAVES = SIMPLE_THREADS / PULSE_WAVE;
    constexpr int PER = SIMPLE_CHUNK / SIMPLE_THREADS;   // consecutive logits a thread takes
    __shared__ float s_bound;
    __shared__ int s_count[WAVES];
    const int r = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    int k = top_k ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 0.f;
    if (k <= 0 && p > 0.f && p < 1.f) k = top_p_bound_rank(chunks);   // top-p alone: see top_p_bound_rank
    const float temp = temperature ? temperature[r] : 0.f;
    int* my_n = seg_n + r * chunks + chunk;
    if (!(temp > 0.f) || k <= 0 || k > chunks || chunks > 2 * PULSE_WAVE) {   // greedy rows need no candidates; the others are not for these kernels
        if (threadIdx.x == 0) *my_n = 0;
        return;
    }
    // the chunk's logits are asked for first: they travel while the bound is searched
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const int begin = chunk * SIMPLE_CHUNK + static_cast<int>(threadIdx.x) * PER;
    float xs[PER];
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = begin + j;
            xs[j] = i < vocab ? row.at<decltype(masked)::value>(i) : -INFINITY;
        }
    });
    // the k-th largest of the chunks' maxima, bit by bit (chunks <= 2 * 64: two a lane)
    if (wave == 0) {
        uint32_t keys[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = lane + j * PULSE_WAVE;
            keys[j] = c < chunks ? order_key(part_max[r * chunks + c]) : 0u;
        }
        uint32_t bound = 0u;
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = bound | (1u << bit);
            if (__builtin_popcountll(__ballot(keys[0] >= cand)) + __builtin_popcountll(__ballot(keys[1] >= cand)) >= k) bound = cand;
        }
        // back to the value whose key it is (a maximum of -inf, a chunk with nothing left, has the key of -inf)
        float value = -INFINITY;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = lane + j * PULSE_WAVE;
            if (c < chunks && keys[j] == bound) value = part_max[r * chunks + c];
        }
        value = wave_max(value);
        if (lane == 0) s_bound = value;
    }
    __syncthreads();
    const float bound = s_bound;
    int mine = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) mine += (xs[j] != -INFINITY && xs[j] >= bound) ? 1 : 0;
    // where this thread's candidates go: an exclusive sum over the threads, in thread order (vocabulary order)
    int pre = mine;
#pragma unroll
    for (int off = 1; off < PULSE_WAVE; off <<= 1) {
        const int up = __shfl_up(pre, off, PULSE_WAVE);
        if (lane >= off) pre += up;
    }
    if (lane == PULSE_WAVE - 1) s_count[wave] = pre;
    __syncthreads();
    int at = pre - mine, total = 0;
    for (int w = 0; w < WAVES; ++w) {
        if (w < wave) at += s_count[w];
        total += s_count[w];
    }
    int* out_i = seg_i + (static_cast<int64_t>(r) * chunks + chunk) * TOPK_SEGMENT;
    float* out_x = seg_x + (static_cast<int64_t>(r) * chunks + chunk) * TOPK_SEGMENT;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        if (xs[j] != -INFINITY && xs[j] >= bound) {
            if (at < TOPK_SEGMENT) { out_i[at] = begin + j; out_x[at] = xs[j]; }
            ++at;
        }
    }
    if (threadIdx.x == 0) *my_n = total;   // more than TOPK_SEGMENT: the row does not fit
}

// What rest_kernel adds a row's histogram to.
__device__ __forceinline__ void clear_histogram(int* rest, int lane) {
    for (int b = lane; b < 2 * HIST_BINS; b += PULSE_WAVE) rest[b] = 0;
}

// The choice of every row from what the kernels before left, a wavefront a row: the largest logit for greedy rows;
// for rows with top-k the candidates' segments strung together in LDS and finished there; for rows that draw from the
// whole vocabulary the chunk in which u * mass falls (chunk masses in chunk order), walked alone.  done[r] says
// whether the row's token is chosen; the others (rows that did not fit) are sample_kernel's.
__global__ __launch_bounds__(PULSE_WAVE) void chunked_choose_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, const float* __restrict__ part_max,
    const int* __restrict__ part_idx, const float* __restrict__ part_mass, const int* __restrict__ seg_i,
    const float* __restrict__ seg_x, const int* __restrict__ seg_n, int chunks, int* __restrict__ out,
    int* __restrict__ done, int* __restrict__ left) {
    __shared__ int list_i[LIST_CAP];
    __shared__ float list_x[LIST_CAP];
    const int r = blockIdx.x, lane = threadIdx.x;
    part_max += r * chunks;
    part_idx += r * chunks;
    part_mass += r * chunks;
    seg_n += r * chunks;
    // the largest logit, the lowest index among equals
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    for (int c = lane; c < chunks; c += PULSE_WAVE) {
        const float v = part_max[c];
        const int i = part_idx[c];
        if (v > best || (v == best && i < best_i)) { best = v; best_i = i; }
    }
    wave_argmax(best, best_i);
    const float temp = temperature ? temperature[r] : 0.f;
    if (best_i == 0x7fffffff || !(temp > 0.f)) {   // everything banned or NaN, or the largest logit wins
        if (lane == 0) { out[r] = best_i == 0x7fffffff ? -1 : best_i; done[r] = 1; }
        return;
    }
    const int k = top_k ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 0.f;
    const bool use_p = p > 0.f && p < 1.f;
    const float inv_t = 1.0f / temp;
    if (k > 0 || use_p) {
        const bool by_k = k > 0;
        // the segments' places in the list: an exclusive sum over the chunks, in chunk order (two chunks a lane)
        const int n0 = lane < chunks ? seg_n[lane] : 0, n1 = lane + PULSE_WAVE < chunks ? seg_n[lane + PULSE_WAVE] : 0;
        const bool over = n0 > TOPK_SEGMENT || n1 > TOPK_SEGMENT;
        int pre0 = n0, pre1 = n1;
#pragma unroll
        for (int off = 1; off < PULSE_WAVE; off <<= 1) {
            const int u0 = __shfl_up(pre0, off, PULSE_WAVE), u1 = __shfl_up(pre1, off, PULSE_WAVE);
            if (lane >= off) { pre0 += u0; pre1 += u1; }
        }
        const int first = __shfl(pre0, PULSE_WAVE - 1, PULSE_WAVE);      // candidates of chunks 0 .. 63
        const int n = first + __shfl(pre1, PULSE_WAVE - 1, PULSE_WAVE);
        if (k > chunks || chunks > 2 * PULSE_WAVE || __ballot(over) != 0ull || n > LIST_CAP || n < k || n == 0) {
            if (lane == 0) done[r] = 0;   // not a row for these kernels: sample_kernel takes it
            if (left) clear_histogram(left + static_cast<int64_t>(r) * REST_WORDS, lane);
            return;
        }
        float whole = 0.f;   // without top-k: the mass of the whole row, chunk masses in chunk order
        if (!by_k) {
            for (int c = lane; c < chunks; c += PULSE_WAVE) whole += part_mass[c];
            whole = wave_sum(whole);
        }
        const int64_t seg0 = (static_cast<int64_t>(r) * chunks + lane) * TOPK_SEGMENT;
        for (int e = 0; e < n0; ++e) { list_i[pre0 - n0 + e] = seg_i[seg0 + e]; list_x[pre0 - n0 + e] = seg_x[seg0 + e]; }
        const int64_t seg1 = seg0 + static_cast<int64_t>(PULSE_WAVE) * TOPK_SEGMENT;
        for (int e = 0; e < n1; ++e) { list_i[first + pre1 - n1 + e] = seg_i[seg1 + e]; list_x[first + pre1 - n1 + e] = seg_x[seg1 + e]; }
        __syncthreads();
        int token;
        const bool enough =   // (false only without top-k: the list does not hold top_p of the row)
            n <= 4 * PULSE_WAVE   // the usual case with top-k: a few dozen candidates, a few a lane
                ? finish_on_list<4>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, uniform[r], best_i, token)
                : finish_on_list<LIST_PER_LANE>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, uniform[r], best_i, token);
        if (lane == 0) {
            if (enough) out[r] = token;
            done[r] = enough ? 1 : 0;
        }
        if (left && !__shfl(enough ? 1 : 0, 0, PULSE_WAVE)) clear_histogram(left + static_cast<int64_t>(r) * REST_WORDS, lane);
        return;
    }
    // a draw from the whole vocabulary: the chunk in which it falls, chunk masses in chunk order
    float total = 0.f;
    for (int c = lane; c < chunks; c += PULSE_WAVE) total += part_mass[c];
    total = wave_sum(total);
    const float target = uniform[r] * total;
    float run = 0.f;
    int who = -1, last_chunk = -1;
    // (every lane the same few dozen additions; the masses come 64 at a time, one a lane, so that the additions do
    // not each wait for a trip to memory)
    for (int base = 0; base < chunks && who < 0; base += PULSE_WAVE) {
        const float mine = base + lane < chunks ? part_mass[base + lane] : 0.f;
        const int n = min(PULSE_WAVE, chunks - base);
        for (int j = 0; j < n; ++j) {
            const float m = __shfl(mine, j, PULSE_WAVE);
            if (m > 0.f) {
                last_chunk = base + j;
                if (target < run + m) { who = base + j; break; }
            }
            run += m;
        }
    }
    float rest = target - run;
    if (who < 0) {  // rounding left the target beyond the last chunk with mass: its last kept entry
        who = last_chunk;
        rest = INFINITY;
    }
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const int begin = who * SIMPLE_CHUNK, end = min(vocab, begin + SIMPLE_CHUNK);
    int last, e;
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
        e = wave_walk(begin, end, rest, [&](int i) {
            const float x = row.at<decltype(masked)::value>(i);
            return x != -INFINITY ? expf((x - best) * inv_t) : 0.f;
        }, last);
    });
    if (lane == 0) { out[r] = e >= 0 ? e : (last >= 0 ? last : best_i); done[r] = 1; }
}

// ---- the rows that are left, before sample_kernel ---------------------------------------------------------------
// A workgroup a row goes over its row at the rate of one compute unit; what sample_kernel needs to know of the whole row, its
// mass (a wavefront of it summed by a wavefront here, entries and order as there) and the histogram over [lowest, best], is
// made by many workgroups, in one launch: 18 us for 6 rows of 151,936 and 32 for 26, where the passes inside sample_kernel
// took 220 and two launches, the histogram behind the mass and the lowest value, 34 for 13.  (The lowest value comes with the maxima, and the
// histogram is cleared by the kernel that leaves the row.)
constexpr int REST_GROUPS = 16;                                             // workgroups for a row's histogram
constexpr int MASS_GROUPS = SAMPLE_WAVES * PULSE_WAVE / SIMPLE_THREADS;     // and for its mass

__global__ __launch_bounds__(SIMPLE_THREADS) void rest_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ penalty, const int* __restrict__ seen_row,
    const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned, int mask_words,
    const float* __restrict__ part_max, const float* __restrict__ part_min, int chunks, const int* __restrict__ done,
    int* __restrict__ rest) {
    __shared__ int hist[HIST_BINS];
    __shared__ float hist_w[HIST_BINS];
    const int r = blockIdx.y, lane = threadIdx.x % PULSE_WAVE;
    if (done[r]) return;
    rest += static_cast<int64_t>(r) * REST_WORDS;
    const float best = simple_row_max(part_max + static_cast<int64_t>(r) * chunks, chunks);
    const float inv_t = 1.0f / temperature[r];
    const int k = top_k ? top_k[r] : 0;
    const bool by_k = k > 0 && k < vocab;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    if (blockIdx.x < MASS_GROUPS) {
        const int wave = blockIdx.x * (SIMPLE_THREADS / PULSE_WAVE) + threadIdx.x / PULSE_WAVE;
        float mass = 0.f, lowest = INFINITY;
        if (!by_k)
            sweep(row, wave * PULSE_WAVE + lane, vocab, SAMPLE_THREADS, [&](int, float x) {
                if (x != -INFINITY) mass += expf((x - best) * inv_t);
            });
        for (int c = lane; c < chunks; c += PULSE_WAVE) lowest = fminf(lowest, part_min[static_cast<int64_t>(r) * chunks + c]);
        mass = wave_sum(mass);
        lowest = -wave_max(-lowest);
        if (lane == 0) {
            rest[REST_MASS + wave] = __float_as_int(mass);
            rest[REST_LOWEST + wave] = __float_as_int(lowest);
        }
        return;
    }
    for (int b = threadIdx.x; b < HIST_BINS; b += SIMPLE_THREADS) { hist[b] = 0; hist_w[b] = 0.f; }
    float lowest = INFINITY;
    for (int c = lane; c < chunks; c += PULSE_WAVE) lowest = fminf(lowest, part_min[static_cast<int64_t>(r) * chunks + c]);
    lowest = -wave_max(-lowest);
    const float scale = static_cast<float>(HIST_BINS) / (best - lowest);
    __syncthreads();
    if (!(best > lowest && scale < INFINITY)) return;    // (as sample_kernel: no histogram)
    sweep(row, (blockIdx.x - MASS_GROUPS) * SIMPLE_THREADS + threadIdx.x, vocab, REST_GROUPS * SIMPLE_THREADS, [&](int, float x) {
        if (x != -INFINITY) {
            const int b = min(HIST_BINS - 1, static_cast<int>((best - x) * scale));
            atomicAdd(&hist[b], 1);
            if (!by_k) add_in_group(&hist_w[b], expf((x - best) * inv_t));
        }
    });
    __syncthreads();
    for (int b = threadIdx.x; b < HIST_BINS; b += SIMPLE_THREADS) {
        if (hist[b] == 0) continue;
        atomicAdd(&rest[b], hist[b]);
        if (!by_k) unsafeAtomicAdd(reinterpret_cast<float*>(rest) + HIST_BINS + b, hist_w[b]);
    }
}

}  // namespace

// out[r] = index of the largest logit of row r, the lowest index among equals, -1 if none is a number.
// part_val / part_idx: scratch of rows * pulse_argmax_chunks(vocab) entries each.
extern "C" int pulse_argmax_chunks(int vocab) {
    const int chunk = 2048;
    return (vocab + chunk - 1) / chunk;
}

extern "C" int pulse_argmax(const float* logits, int rows, int vocab, int64_t row_stride, float* part_val,
                            int* part_idx, int* out, hipStream_t stream) {
    PULSE_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, "argmax: bad sizes rows=%d V=%d", rows, vocab);
    PULSE_REQUIRE(rows < 65536, "argmax: at most 65535 rows");
    PULSE_REQUIRE(logits && part_val && part_idx && out, "argmax: null pointer");
    if (rows == 0) return 0;
    const int chunks = pulse_argmax_chunks(vocab);
    hipLaunchKernelGGL(argmax_chunks_kernel, dim3(chunks, rows), dim3(ARGMAX_THREADS), 0, stream, logits, vocab,
                       row_stride, 2048, part_val, part_idx);
    PULSE_LAUNCH_CHECK("argmax_chunks");
    hipLaunchKernelGGL(argmax_merge_kernel, dim3(rows), dim3(PULSE_WAVE), 0, stream, part_val, part_idx, chunks, out);
    PULSE_LAUNCH_CHECK("argmax_merge");
    return 0;
}

// The same without a workspace argument: the chunk winners go through an array in the library's device image.
// In host code the array's name is only a stand-in for the symbol; its address on a device comes from
// hipGetSymbolAddress, once per device, and that pointer is what the kernels get.
static __device__ __align__(256) unsigned char argmax_static_scratch[PULSE_ARGMAX_STATIC_ENTRIES * 8];

namespace {
constexpr int STATIC_MAX_DEVICES = 64;
void* g_static_scratch[STATIC_MAX_DEVICES] = {};
std::mutex g_static_lock;
}  // namespace

extern "C" int pulse_argmax_static(const float* logits, int rows, int vocab, int64_t row_stride, int* out,
                                   hipStream_t stream) {
    PULSE_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, "argmax_static: bad sizes rows=%d V=%d", rows, vocab);
    PULSE_REQUIRE(rows < 65536, "argmax_static: at most 65535 rows");
    PULSE_REQUIRE(logits && out, "argmax_static: null pointer");
    const int chunks = pulse_argmax_chunks(vocab);
    PULSE_REQUIRE(static_cast<int64_t>(rows) * chunks <= PULSE_ARGMAX_STATIC_ENTRIES,
                  "argmax_static: %d rows x %d chunks of the vocabulary exceed the %d entries of the built-in scratch "
                  "array; use pulse_argmax with a workspace", rows, chunks, PULSE_ARGMAX_STATIC_ENTRIES);
    if (rows == 0) return 0;
    int device = -1;
    hipError_t err = hipGetDevice(&device);
    PULSE_REQUIRE(err == hipSuccess, "argmax_static: hipGetDevice: %s", hipGetErrorString(err));
    PULSE_REQUIRE(device >= 0 && device < STATIC_MAX_DEVICES, "argmax_static: device %d is beyond the %d this entry "
                  "point keeps an address for", device, STATIC_MAX_DEVICES);
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> hold(g_static_lock);
        if (!g_static_scratch[device]) {   // each GPU holds its own copy of the array at its own address
            void* found = nullptr;
            err = hipGetSymbolAddress(&found, HIP_SYMBOL(argmax_static_scratch));
            PULSE_REQUIRE(err == hipSuccess && found, "argmax_static: hipGetSymbolAddress on device %d: %s", device,
                          hipGetErrorString(err));
            g_static_scratch[device] = found;
        }
        base = g_static_scratch[device];
    }
    float* part_val = static_cast<float*>(base);
    int* part_idx = reinterpret_cast<int*>(static_cast<unsigned char*>(base) + PULSE_ARGMAX_STATIC_ENTRIES * 4);
    hipLaunchKernelGGL(argmax_chunks_kernel, dim3(chunks, rows), dim3(ARGMAX_THREADS), 0, stream, logits, vocab,
                       row_stride, 2048, part_val, part_idx);
    PULSE_LAUNCH_CHECK("argmax_static chunks");
    hipLaunchKernelGGL(argmax_merge_kernel, dim3(rows), dim3(PULSE_WAVE), 0, stream, part_val, part_idx, chunks, out);
    PULSE_LAUNCH_CHECK("argmax_static merge");
    return 0;
}

// out[r] = chosen token of row r, or -1 when no token is allowed.
// temperature/top_k/top_p/penalty/seen_row/banned may be null (greedy, off, off, none, none, none).
extern "C" int pulse_sample(const float* logits, int rows, int vocab, int64_t row_stride, const float* temperature,
                            const int* top_k, const float* top_p, const float* uniform, const float* penalty,
                            const int* seen_row, const uint32_t* seen_masks, const uint32_t* banned,
                            int mask_words, int* out, hipStream_t stream) {
    PULSE_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, "sample: bad sizes rows=%d V=%d", rows, vocab);
    PULSE_REQUIRE(logits && out, "sample: null pointer");
    PULSE_REQUIRE(!temperature || uniform, "sample: temperature sampling needs uniform numbers");
    PULSE_REQUIRE((!seen_masks && !banned) || mask_words * 32 >= vocab, "sample: masks cover %d tokens, vocabulary has %d",
                  mask_words * 32, vocab);
    if (rows == 0) return 0;
    hipLaunchKernelGGL(sample_kernel, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                       temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, out,
                       static_cast<const int*>(nullptr), static_cast<const float*>(nullptr),
                       static_cast<const int*>(nullptr), 0, static_cast<const int*>(nullptr));
    PULSE_LAUNCH_CHECK("sample");
    return 0;
}

// The same in chunks of the vocabulary with a workgroup each, which reads a row many times faster than the
// workgroup a row of pulse_sample does.  Greedy rows, rows that draw from the whole vocabulary at their temperature
// rows with top-k (and top-p on what it keeps) whose k is at most the number of chunks and rows with top-p alone whose
// top_p share lies in some hundreds of the largest logits are chosen by these kernels; rows that do not fit (many
// equal values around the k-th largest, a distribution too flat for top-p alone) by the kernel of pulse_sample behind
// them, which skips the rows that are done.  What a row's choice is does not depend on the
// other rows.  Scratch, with chunks = pulse_sample_chunks(vocab): part_max, part_mass (float32), part_idx, seg_n
// (int32) of rows * chunks entries; seg_i (int32), seg_x (float32) of rows * chunks * pulse_sample_segment()
// entries; done (int32) of rows entries; and, optional (null: the rows that are left are gone over by their own workgroups
// alone, with the same choices), rest (int32) of rows * (pulse_sample_rest() + chunks) entries.
extern "C" int pulse_sample_rest() { return REST_WORDS; }
extern "C" int pulse_sample_chunks(int vocab) { return (vocab + SIMPLE_CHUNK - 1) / SIMPLE_CHUNK; }
extern "C" int pulse_sample_segment() { return TOPK_SEGMENT; }

extern "C" int pulse_sample_chunked_rest(const float* logits, int rows, int vocab, int64_t row_stride, const float* temperature,
                                    const int* top_k, const float* top_p, const float* uniform, const float* penalty,
                                    const int* seen_row, const uint32_t* seen_masks, const uint32_t* banned,
                                    int mask_words, float* part_max, int* part_idx, float* part_mass, int* seg_i,
                                    float* seg_x, int* seg_n, int* done, int* rest, int* out,
                                         hipStream_t stream) {
    PULSE_REQUIRE(rows >= 0 && vocab > 0 && row_stride >= vocab, "sample_chunked: bad sizes rows=%d V=%d", rows, vocab);
    PULSE_REQUIRE(rows < 65536, "sample_chunked: at most 65535 rows");
    PULSE_REQUIRE(logits && out && part_max && part_idx && part_mass && seg_i && seg_x && seg_n && done,
                  "sample_chunked: null pointer");
    PULSE_REQUIRE(!temperature || uniform, "sample_chunked: temperature sampling needs uniform numbers");
    PULSE_REQUIRE((!seen_masks && !banned) || mask_words * 32 >= vocab, "sample_chunked: masks cover %d tokens, "
                  "vocabulary has %d", mask_words * 32, vocab);
    if (rows == 0) return 0;
    const int chunks = pulse_sample_chunks(vocab);
    const bool leaves = temperature && (top_k || top_p);    // (without them every row is done)
    // They are made while a workgroup a row leaves most of the chip idle and its passes are long: 32,000 values, flat rows
    // under top-p and others, 16 rows 103 and 80 us with them (272 and 87 without any of it), 64 rows 128 and 108, 159 and
    // 92 without; 151,936 values, 64 rows 427 and 291 (947 and 776).
    const bool prepare = rest && leaves && vocab >= 1024 * static_cast<int64_t>(rows);
    if (!prepare) rest = nullptr;
    // (behind what is made of the rows: the chunks' smallest numbers)
    float* part_min = prepare ? reinterpret_cast<float*>(rest + static_cast<int64_t>(rows) * REST_WORDS) : nullptr;
    hipLaunchKernelGGL(simple_max_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                       penalty, seen_row, seen_masks, banned, mask_words, part_max, part_idx, part_min);
    PULSE_LAUNCH_CHECK("sample_chunked (maxima)");
    if (temperature) {
        hipLaunchKernelGGL(simple_mass_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab,
                           row_stride, temperature, top_k, penalty, seen_row, seen_masks, banned, mask_words,
                           part_max, part_mass);
        PULSE_LAUNCH_CHECK("sample_chunked (masses)");
        if (top_k || top_p) {
            hipLaunchKernelGGL(topk_collect_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab,
                               row_stride, temperature, top_k, top_p, penalty, seen_row, seen_masks, banned, mask_words,
                               part_max, seg_i, seg_x, seg_n);
            PULSE_LAUNCH_CHECK("sample_chunked (candidates)");
        }
    }
    hipLaunchKernelGGL(chunked_choose_kernel, dim3(rows), dim3(PULSE_WAVE), 0, stream, logits, vocab, row_stride,
                       temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, part_max,
                       part_idx, part_mass, seg_i, seg_x, seg_n, chunks, out, done, rest);
    PULSE_LAUNCH_CHECK("sample_chunked (choice)");
    if (prepare) {
        hipLaunchKernelGGL(rest_kernel, dim3(MASS_GROUPS + REST_GROUPS, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab,
                           row_stride, temperature, top_k, penalty, seen_row, seen_masks, banned, mask_words, part_max,
                           part_min, chunks, static_cast<const int*>(done), rest);
        PULSE_LAUNCH_CHECK("sample_chunked (what is left)");
    }
    if (leaves) {
        hipLaunchKernelGGL(sample_kernel, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                           temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, out,
                           static_cast<const int*>(done), part_max, part_idx, chunks, static_cast<const int*>(rest));
        PULSE_LAUNCH_CHECK("sample_chunked (the rest)");
    }
    return 0;
}

extern "C" int pulse_sample_chunked(const float* logits, int rows, int vocab, int64_t row_stride, const float* temperature,
                                    const int* top_k, const float* top_p, const float* uniform, const float* penalty,
                                    const int* seen_row, const uint32_t* seen_masks, const uint32_t* banned,
                                    int mask_words, float* part_max, int* part_idx, float* part_mass, int* seg_i,
                                    float* seg_x, int* seg_n, int* done, int* out, hipStream_t stream) {
    return pulse_sample_chunked_rest(logits, rows, vocab, row_stride, temperature, top_k, top_p, uniform, penalty, seen_row,
                                     seen_masks, banned, mask_words, part_max, part_idx, part_mass, seg_i, seg_x, seg_n, done,
                                     nullptr, out, stream);
}

// Set the bit of tokens[i] in the mask row rows[i] (the per-request "seen" set of the presence penalty).
extern "C" int pulse_mark_seen(uint32_t* masks, int mask_words, const int* rows, const int* tokens, int n, int vocab,
                               hipStream_t stream) {
    PULSE_REQUIRE(masks && rows && tokens && n >= 0 && mask_words * 32 >= vocab, "mark_seen: bad arguments");
    if (n == 0) return 0;
    hipLaunchKernelGGL(mark_seen_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, masks, mask_words, rows,
                       tokens, n, vocab);
    PULSE_LAUNCH_CHECK("mark_seen");
    return 0;
}
