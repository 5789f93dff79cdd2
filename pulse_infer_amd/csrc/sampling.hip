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
#include <string.h>

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

// The sum of a step's 64 weights is the prefix's at its last lane, to the bit, and a third of the prefix's instructions without a trip
// through LDS: the prefix is made for the step in which the sum comes near `rest` only (chunked_choose_kernel, 32 rows of 151,936,
// 28 -> 22 us).
__device__ __forceinline__ float pairs_sum(float v) {     // neighbours first, then pairs of neighbours, ..
    const auto moved = [&](auto code) __attribute__((always_inline)) {
        return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(code)::value, 0xF, 0xF, true)));
    };
    v += moved(Int<0xB1>());      // quad_perm [1, 0, 3, 2]
    v += moved(Int<0x4E>());      // quad_perm [2, 3, 0, 1]
    v += moved(Int<0x141>());     // row_half_mirror: the other four of eight
    v += moved(Int<0x140>());     // row_mirror: the other eight of sixteen
    return across_rows(v, LaneSum());
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
        float sums[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) sums[u] = pairs_sum(ws[u]);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int base = first + u * PULSE_WAVE;
            const float w = ws[u];
            const unsigned long long has = __ballot(w > 0.f);
            if (has == 0ull) continue;
            last = base + (63 - __builtin_clzll(has));
            // (a prefix may round up to a few units in its last place beyond the sum)
            if (!(rest < (run + sums[u]) * 1.00001f)) {
                run += sums[u];
                continue;
            }
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

// The same over STEPS * 64 weights in LDS whose steps' sums (as pairs_sum makes them) are there, step q's in lane q.
template <int STEPS>
__device__ int wave_walk_summed(const float* weights, float sums, float rest, int& last) {
    const int lane = threadIdx.x % PULSE_WAVE;
    float run = 0.f;
    last = -1;
    for (int q = 0; q < STEPS; ++q) {
        const float sum = __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_readlane(__float_as_int(sums), q)));
        if (sum == 0.f) continue;      // (no weight above zero)
        if (!(rest < (run + sum) * 1.00001f)) {
            run += sum;
            continue;
        }
        const float w = weights[q * PULSE_WAVE + lane];
        float pre = w;
#pragma unroll
        for (int off = 1; off < PULSE_WAVE; off <<= 1) {
            const float up = __shfl_up(pre, off, PULSE_WAVE);
            if (lane >= off) pre += up;
        }
        const unsigned long long hit = __ballot(w > 0.f && rest < run + pre);
        if (hit != 0ull) return q * PULSE_WAVE + __builtin_ctzll(hit);
        run += __shfl(pre, PULSE_WAVE - 1, PULSE_WAVE);
    }
    for (int q = STEPS - 1; q >= 0 && last < 0; --q) {
        const unsigned long long has = __ballot(weights[q * PULSE_WAVE + lane] > 0.f);
        if (has != 0ull) last = q * PULSE_WAVE + 63 - __builtin_clzll(has);
    }
    return -1;
}

constexpr int HIST_BINS = 2048;                         // bins of the value histogram that locates the k-th largest
constexpr int WAVE_CAP = 128;                           // candidates a wavefront may collect
constexpr int LIST_CAP = SAMPLE_WAVES * WAVE_CAP;       // candidates of a row
constexpr int LIST_PER_LANE = LIST_CAP / PULSE_WAVE;

// The first bit (from the top) in which two keys differ, -1 for none; what of a key lies above a bit.
__device__ __forceinline__ int first_bit(uint32_t a, uint32_t b) { return a == b ? -1 : 31 - __builtin_clz(a ^ b); }
__device__ __forceinline__ uint32_t above_bit(uint32_t key, int bit) { return bit >= 31 ? 0u : key & ~((2u << bit) - 1u); }

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
    // The searches go bit by bit, from the first bit on in which the list's largest and smallest key (then the largest and the k-th
    // largest) differ: what is above is in all of them.  (32 rows of 151,936 with top-k 50, the list's choice alone on its wavefront: 10.3 us from
    // the top bit and by lanes' counts, 9.1 so; left_kernel's top-k of mixed rows 16.8 and 14.0.)
    uint32_t most = 0u, least = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        most = max(most, keys[j]);
        least = min(least, lane + j * PULSE_WAVE < n ? keys[j] : 0xffffffffu);
    }
    most = wave_reduce(most, [](uint32_t a, uint32_t b) { return max(a, b); });
    least = wave_reduce(least, [](uint32_t a, uint32_t b) { return min(a, b); });
    // the k-th largest key
    uint32_t keep = 0u;
    if (by_k) {
        const int from = first_bit(most, least);
        keep = from < 0 ? most : above_bit(most, from);
        for (int bit = from; bit >= 0; --bit) {
            const uint32_t cand = keep | (1u << bit);
            int c = 0;      // (a key past the list is below every candidate)
#pragma unroll
            for (int j = 0; j < PER; ++j) c += __builtin_popcountll(__ballot(keys[j] >= cand));
            if (c >= k) keep = cand;
        }
    }
    if (use_p) {
        float mass = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) mass += keys[j] >= keep ? wts[j] : 0.f;
        mass = wave_sum(mass);
        const float want = p * (by_k ? mass : whole);
        if (!by_k && !(mass >= want)) return false;   // without top-k the list must hold all of the top_p set
        const uint32_t lowest = by_k ? keep : least;
        const int from = first_bit(most, lowest);
        uint32_t thr = from < 0 ? most : above_bit(most, from);
        for (int bit = from; bit >= 0; --bit) {
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

// ---- top-p alone on rows whose share is no short list -------------------------------------------------------------
// The masses here are whole numbers: an entry's weight, at most 1, in units of 2^-40 (2^-31 from 2^23 entries on, so that a row's
// sum fits 64 bits).  Their sums are the same in any order, so a row's threshold and draw are one choice whoever sums, a
// workgroup a row or many, and need no second pass over the row in one fixed order; and they are nearer to the exact masses
// than float32 sums: 152,000 roundings of 2^-41 against sums good to 2^-24.
typedef unsigned long long mass_t;

struct Weigh {
    float best, inv_t, low_scale;
    int low;
    __device__ __forceinline__ Weigh(float best_, float inv_t_, int vocab) : best(best_), inv_t(inv_t_) {
        low = vocab < (1 << 23) ? 20 : 11;
        low_scale = static_cast<float>(1 << low);
    }
    __device__ __forceinline__ mass_t operator()(float x) const {
        const float w = expf((x - best) * inv_t) * 1048576.f;
        const uint32_t high = static_cast<uint32_t>(w);      // (the rest of w is exact)
        return (static_cast<mass_t>(high) << low) + static_cast<uint32_t>(rintf((w - static_cast<float>(high)) * low_scale));
    }
};

__device__ __forceinline__ mass_t mass_sum(mass_t v) {      // (by lane moves: shuffles are trips through LDS)
    auto step = [&](auto apart) __attribute__((always_inline)) {
        const WaveTwo low = wave_two<decltype(apart)::value>(static_cast<uint32_t>(v)), high = wave_two<decltype(apart)::value>(static_cast<uint32_t>(v >> 32));
        v = ((static_cast<mass_t>(high.a) << 32) | low.a) + ((static_cast<mass_t>(high.b) << 32) | low.b);
    };
    step(Int<32>()); step(Int<16>()); step(Int<8>()); step(Int<4>()); step(Int<2>()); step(Int<1>());
    return v;
}
// The sum over the lanes up to this one.
__device__ __forceinline__ mass_t mass_through(mass_t v) {
#pragma unroll
    for (int off = 1; off < PULSE_WAVE; off <<= 1) {
        const mass_t up = __shfl_up(v, off, PULSE_WAVE);
        if (static_cast<int>(threadIdx.x % PULSE_WAVE) >= off) v += up;
    }
    return v;
}

// What the kernels in front of left_kernel leave of a row that the chunks could not choose for, in 32-bit words: the histogram
// over [lowest, best] (rows with top-k: counts; top-p alone: masses; 64 bits each), the row's smallest number, whether its token was
// chosen from what they left (the tests ask; no kernel does), the mass of the bins above the one with top-p's edge, that of the row, and
// every chunk's of the former.
constexpr int REST_LOWEST = 2 * HIST_BINS, REST_CHOSEN = REST_LOWEST + 1, REST_BASE = REST_LOWEST + 2, REST_WHOLE = REST_LOWEST + 4;
constexpr int REST_CHUNKS = REST_LOWEST + 6, REST_MOST_CHUNKS = 2 * PULSE_WAVE;
constexpr int REST_WORDS = REST_CHUNKS + 2 * REST_MOST_CHUNKS;
static_assert(REST_WORDS % 2 == 0 && REST_CHUNKS % 2 == 0, "64-bit words");

__device__ __forceinline__ int bin_at(float x, float best, float scale) { return min(HIST_BINS - 1, static_cast<int>((best - x) * scale)); }

// The bin in which the masses from the top reach p of the whole (or, k > 0, the counts reach k; or, given, `want`), the mass above it
// and the whole: thread t of THREADS sums HIST_BINS / THREADS neighbouring bins.  `base` is on the way in the mass above them all, on
// the way out that above the bin.  -1 if there is no such bin.  Called by a whole workgroup.
template <int THREADS>
__device__ int edge_bin(const mass_t* hist, float p, int k, mass_t* waves, int* at, mass_t* above, mass_t& base, mass_t& whole, double want = -1.) {
    constexpr int PER = HIST_BINS / THREADS, WAVES = THREADS / PULSE_WAVE;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    mass_t bins[PER], mine = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        bins[j] = hist[threadIdx.x * PER + j];
        mine += bins[j];
    }
    const mass_t through = mass_through(mine);
    if (lane == PULSE_WAVE - 1) waves[wave] = through;
    if (threadIdx.x == 0) *at = -1;
    __syncthreads();
    mass_t before = base + through - mine;
    whole = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        if (w < wave) before += waves[w];
        whole += waves[w];
    }
    if (want < 0.) want = k > 0 ? static_cast<double>(k) : static_cast<double>(p) * static_cast<double>(whole);
    if (static_cast<double>(before) < want && static_cast<double>(before + mine) >= want) {      // one thread
        int j = 0;
        while (j < PER - 1 && static_cast<double>(before + bins[j]) < want) before += bins[j++];
        *at = threadIdx.x * PER + j;
        *above = before;
    }
    __syncthreads();
    base = *above;
    return *at;
}

// The largest of the keys at or above which the mass is at least p of the whole: `n` tokens of the edge's bin, `base` the mass
// above it (the masses through the bin reach that share, so there is one).  Every token's own sum, no order, by as many neighbouring lanes
// as there are for each (32 flat rows of 151,936, some 250 tokens in the bin, a lane each: 24 us of left_kernel, so 17.6).  Called by
// a whole workgroup, `best` (LDS) cleared before and read behind a barrier.
__device__ void edge_key(const uint32_t* keys, const mass_t* masses, int n, int threads, mass_t base, mass_t whole, float p, uint32_t* best) {
    const double want = static_cast<double>(p) * static_cast<double>(whole);
    int each = 1;
    while (each < PULSE_WAVE && 2 * each * n <= threads) each *= 2;
    const int sub = threadIdx.x & (each - 1);
    for (int e0 = 0; e0 < n; e0 += threads / each) {
        const int e = e0 + static_cast<int>(threadIdx.x) / each;
        const uint32_t key = keys[min(e, n - 1)];
        mass_t through = 0;
#pragma unroll 8
        for (int j = sub; j < n; j += each) through += keys[j] >= key ? masses[j] : 0;
        for (int off = 1; off < each; off *= 2) through += __shfl_xor(through, off, PULSE_WAVE);
        if (sub == 0 && e < n && static_cast<double>(base + through) >= want) atomicMax(best, key);
    }
}

// u of the kept mass, as a number below it.
__device__ __forceinline__ mass_t draw_from(float u, mass_t kept) {
    const mass_t t = static_cast<mass_t>(static_cast<double>(u) * static_cast<double>(kept));
    return t < kept ? t : kept - 1;
}

constexpr int EDGE_CAP = 1024;   // tokens of the edge's bin that are ranked

// A row by a workgroup of SAMPLE_THREADS.  `chunked`: behind the kernels that work in chunks, which left the chunks' maxima, and in
// `rest` what they have been over the row for, or null.
__device__ __forceinline__ void sample_row(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, int* __restrict__ out, const bool chunked,
    const float* __restrict__ part_max, const int* __restrict__ part_idx, int chunks, const int* __restrict__ rest) {
    __shared__ float sf[SAMPLE_WAVES];
    __shared__ int si[SAMPLE_WAVES];
    __shared__ mass_t hist_m[HIST_BINS];    // top-p alone: the bins' masses
    int* const hist = reinterpret_cast<int*>(hist_m);
    if (rest) rest += static_cast<int64_t>(blockIdx.x) * REST_WORDS;
    __shared__ int wave_bins[SAMPLE_WAVES];
    __shared__ int region_i[SAMPLE_WAVES][WAVE_CAP];
    __shared__ float region_x[SAMPLE_WAVES][WAVE_CAP];
    __shared__ int region_n[SAMPLE_WAVES];
    __shared__ int list_i[LIST_CAP];
    __shared__ float list_x[LIST_CAP];
    __shared__ float part_sum[SAMPLE_WAVES];
    __shared__ int list_done;
    __shared__ mass_t edge_m[EDGE_CAP], part_m[SAMPLE_WAVES], edge_above;
    __shared__ uint32_t edge_best;
    __shared__ int edge_n;

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
    // Top-p alone takes the same way with the LIST_TRY largest values, if their mass reaches top_p of the whole.  (Behind the
    // kernels in chunks it does not: their list was as long.)
    constexpr int LIST_TRY = 1024;
    const bool by_k = k > 0 && k < vocab;
    const int k_list = by_k ? k : min(vocab - 1, LIST_TRY);
    float whole = 0.f;   // without top-k: the mass of the whole vocabulary, which top_p refers to
    if (by_k || (use_p && k_list > 0 && !chunked)) {
        if (rest) {      // (the kernels before have been over the row)
            lowest = __int_as_float(rest[REST_LOWEST]);
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
                hist[b] = rest ? rest[2 * b] : 0;
            }
            __syncthreads();
            if (!rest) {
                sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    if (x != -INFINITY) atomicAdd(&hist[bin_of(x)], 1);
                });
                __syncthreads();
            }
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
        if (edge >= 0 && listed <= LIST_CAP) {
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
    if (use_p && !by_k) {
        const Weigh weigh(best, inv_t, vocab);
        float least = rest ? __int_as_float(rest[REST_LOWEST]) : lowest;
        if (least == INFINITY) {      // (nobody has been over the row for it)
            sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                if (x != -INFINITY) least = fminf(least, x);
            });
            least = -block_max_f(-least, sf);
        }
        const float scale = static_cast<float>(HIST_BINS) / (best - least);
        mass_t base = 0, whole_m = 0;
        uint32_t thr = 0u;
        bool found = false;
        if (best > least && scale < INFINITY) {
            // The bin in which the masses from the top reach top-p's share, and of its tokens the one that does it.  (Whole
            // masses and one pass for that token take the place of float32 sums, good for a bracket only, and of a pass over
            // the row for the sums at the five or fifteen tokens round that place.)
            __syncthreads();
            for (int b = threadIdx.x; b < HIST_BINS; b += SAMPLE_THREADS) hist_m[b] = rest ? reinterpret_cast<const mass_t*>(rest)[b] : 0;
            if (threadIdx.x == 0) { edge_n = 0; edge_best = 0u; }
            __syncthreads();
            if (!rest) {
                sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    if (x != -INFINITY) atomicAdd(&hist_m[bin_at(x, best, scale)], weigh(x));
                });
                __syncthreads();
            }
            const int at = edge_bin<SAMPLE_THREADS>(hist_m, p, 0, part_m, si, &edge_above, base, whole_m);
            if (at >= 0) {
                uint32_t* const keys = reinterpret_cast<uint32_t*>(list_i);
                sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    if (x == -INFINITY || bin_at(x, best, scale) != at) return;
                    const int e = atomicAdd(&edge_n, 1);
                    if (e < EDGE_CAP) { keys[e] = order_key(x); edge_m[e] = weigh(x); }
                });
                __syncthreads();
                const int n = edge_n;
                if (n <= EDGE_CAP) {
                    edge_key(keys, edge_m, n, SAMPLE_THREADS, base, whole_m, p, &edge_best);
                    __syncthreads();
                    thr = edge_best;
                    found = thr != 0u;
                }
            }
        }
        auto block_mass = [&](mass_t v) {
            v = mass_sum(v);
            __syncthreads();
            if (lane == 0) part_m[wave] = v;
            __syncthreads();
            mass_t total = 0;
            for (int w = 0; w < SAMPLE_WAVES; ++w) total += part_m[w];
            return total;
        };
        if (!found) {
            // Too many tokens in a bin, or no range: the threshold's bits, eleven a pass, by a histogram over them.  (Four bits a pass,
            // the masses above the fifteen candidates of a digit side by side in 64 bits, took eight passes and spilled 395 registers:
            // a row of 151,936 with ties at the edge 1,855 us, so 408.)
            double want = -1.;
            base = 0;
            thr = 0u;
            for (int pass = 0; pass < 3; ++pass) {
                const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0, known = pass == 0 ? 32 : pass == 1 ? 21 : 10;
                const uint32_t most = pass == 2 ? 1023u : 2047u;
                __syncthreads();
                for (int b = threadIdx.x; b < HIST_BINS; b += SAMPLE_THREADS) hist_m[b] = 0;
                __syncthreads();
                sweep<8>(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) {
                    const uint32_t key = order_key(x);
                    if (x == -INFINITY || (known < 32 && (key ^ thr) >> known != 0u)) return;
                    mass_t w = weigh(x);
                    // (one entry for lanes that all hold the same value, which would wait for one another)
                    const unsigned long long here = __ballot(1);
                    if (__ballot(key == static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(key))) == here) {
                        if (lane != __builtin_ctzll(here)) return;
                        w *= static_cast<mass_t>(__builtin_popcountll(here));
                    }
                    atomicAdd(&hist_m[most - ((key >> shift) & most)], w);
                });
                __syncthreads();
                const int at = edge_bin<SAMPLE_THREADS>(hist_m, p, 0, part_m, si, &edge_above, base, whole_m, want);
                if (at < 0) { thr = 0xffffffffu; break; }     // (no weight is a number)
                if (pass == 0) want = static_cast<double>(p) * static_cast<double>(whole_m);
                thr |= (most - at) << shift;
            }
        }
        // the kept mass of every wavefront's part, then the part in which the draw falls is walked by its wavefront
        mass_t mine = 0;
        sweep(row, part_begin + lane, part_end, PULSE_WAVE, [&](int, float x) { if (x != -INFINITY && order_key(x) >= thr) mine += weigh(x); });
        const mass_t kept = block_mass(mine);
        if (kept == 0) {     // (an infinite logit: no weight is a number)
            if (threadIdx.x == 0) out[r] = best_i;
            return;
        }
        const mass_t target = draw_from(uniform[r], kept);
        mass_t run = 0;
        int who = 0;
        while (target >= run + part_m[who]) run += part_m[who++];      // (target < kept: there is such a part)
        if (wave != who) return;
        int token = -1;
        by_mask(row, [&](auto masked) __attribute__((always_inline)) {
            constexpr int AHEAD = 8;     // steps of 64 entries whose values are asked for together
            for (int first = part_begin; first < part_end && token < 0; first += AHEAD * PULSE_WAVE) {
                float xs[AHEAD];
#pragma unroll
                for (int q = 0; q < AHEAD; ++q) {
                    const int i = first + q * PULSE_WAVE + lane;
                    xs[q] = i < part_end ? row.at<decltype(masked)::value>(i) : -INFINITY;
                }
#pragma unroll
                for (int q = 0; q < AHEAD; ++q) {
                    if (token >= 0) continue;
                    const mass_t through = run + mass_through(xs[q] != -INFINITY && order_key(xs[q]) >= thr ? weigh(xs[q]) : 0);
                    const unsigned long long hit = __ballot(target < through);
                    if (hit != 0ull) token = first + q * PULSE_WAVE + __builtin_ctzll(hit);
                    run = __shfl(through, PULSE_WAVE - 1, PULSE_WAVE);
                }
            }
        });
        if (lane == 0) out[r] = token;
        return;
    }
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
        float mass = 0.f;
        sweep(row, threadIdx.x, vocab, SAMPLE_THREADS, [&](int, float x) { mass += weight_of(x); });
        const float want = p * block_sum_f(mass, sf);
        // The largest threshold whose kept mass still reaches `want`, four bits of it a pass over the row: the masses
        // above the fifteen candidates of a digit are summed side by side (each in the order in which a pass for it
        // alone would sum it, so the choice is that of a search bit by bit, in an eighth of the passes).
        uint32_t thr = 0u;
        for (int shift = 28; shift >= 0; shift -= 4) {
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
        if (last_part < 0) {      // (no weight is a number above zero)
            if (threadIdx.x == 0) out[r] = best_i;
            return;
        }
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

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, int* __restrict__ out) {
    sample_row(logits, vocab, row_stride, temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, out,
               false, nullptr, nullptr, 0, nullptr);
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
// walks that chunk alone (chunked_choose_kernel).  The steps and their meaning are those of sample_row; sums are
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

// ---- rows with top-k, in chunks -------------------------------------------------------------------------------
// With a small k the candidates can be found chunk by chunk as well.  The k-th largest of the chunks' maxima is a
// lower bound of the k-th largest logit (that many logits, the maxima themselves, reach it), so everything that
// top-k keeps lies at or above it, and little else: a workgroup a chunk collects what it has there, in vocabulary
// order, into its own short segment; a wavefront a row strings the segments together in LDS and finishes on that list
// as sample_row does on its own (finish_on_list).  A row that does not fit (k above the number of chunks, a chunk
// with more candidates than its segment holds: many equal values) is left to left_kernel, which runs behind and
// skips the rows that are done.
constexpr int TOPK_SEGMENT = 32;   // candidates a chunk may leave

// A row with top-p alone takes the same way with what lies at or above one of the lower chunk maxima (seven eighths
// of the chunks have a larger one): some hundreds of the largest logits of a vocabulary of 150,000, which hold the
// top_p share of a distribution as peaked as a language model's; if they do not (or a chunk has more than its segment
// holds), the row is left to left_kernel too.  The mass of the whole row, which top_p refers to, is the chunks' masses'.
__device__ __forceinline__ int top_p_bound_rank(int chunks) { return max(1, chunks - chunks / 8); }

// Where a chunk's entries go that are taken, entry u * SIMPLE_THREADS + t being thread t's u-th: the number of those before it in that
// order (vocabulary order), -1 for what is not taken; `total`: all of them.  Called by a whole workgroup, `counts` of its own each time.
constexpr int CHUNK_PER = SIMPLE_CHUNK / SIMPLE_THREADS;
__device__ __forceinline__ void chunk_places(const bool (&taken)[CHUNK_PER], int (*counts)[SIMPLE_THREADS / PULSE_WAVE], int (&place)[CHUNK_PER], int& total) {
    constexpr int WAVES = SIMPLE_THREADS / PULSE_WAVE;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    unsigned long long has[CHUNK_PER];
#pragma unroll
    for (int u = 0; u < CHUNK_PER; ++u) {
        has[u] = __ballot(taken[u]);
        if (lane == u) counts[u][wave] = __builtin_popcountll(has[u]);
    }
    __syncthreads();
    total = 0;
#pragma unroll
    for (int u = 0; u < CHUNK_PER; ++u) {
        place[u] = total + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(has[u] >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(has[u]), 0u));
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            if (w < wave) place[u] += counts[u][w];
            total += counts[u][w];
        }
        if (!taken[u]) place[u] = -1;
    }
}

// A chunk's logits, entry u * SIMPLE_THREADS + t with thread t (-inf past the end), all asked for together.
__device__ __forceinline__ void chunk_values(const RowView& row, int begin, float (&xs)[CHUNK_PER]) {
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < CHUNK_PER; ++u) {
            const int i = begin + u * SIMPLE_THREADS + static_cast<int>(threadIdx.x);
            const float x = row.at<decltype(masked)::value>(min(i, row.vocab - 1));
            xs[u] = i < row.vocab ? x : -INFINITY;
        }
    });
}

// What a chunk adds, the row's maxima known: its mass (rows without top-k) and its candidates (rows with top-k or top-p), from one reading
// of its logits.  What bounds it: the trips to memory of 9 workgroups a unit; the logits are asked for first, in whole lines.  (Two
// kernels, the candidates' a thread with eight neighbouring logits, 32 rows of 151,936: all options 5.6 + 11.0 us, 8.9 in one; top-p alone
// 6.8 + 18.8 and 12.6.)
__global__ __launch_bounds__(SIMPLE_THREADS) void chunk_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ penalty,
    const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned,
    int mask_words, const float* __restrict__ part_max, float* __restrict__ part_mass, int* __restrict__ seg_i, float* __restrict__ seg_x,
    int* __restrict__ seg_n) {
    constexpr int WAVES = SIMPLE_THREADS / PULSE_WAVE;
    __shared__ float s_bound, s_mass[WAVES];
    __shared__ int s_count[CHUNK_PER][WAVES];
    const int r = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    const int own_k = top_k ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 0.f, temp = temperature[r];
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const bool any = top_k || top_p, weighed = temp > 0.f && own_k <= 0;      // (what top-k keeps is weighed on the short list)
    const int k = own_k <= 0 && p > 0.f && p < 1.f ? top_p_bound_rank(chunks) : own_k;      // top-p alone: see top_p_bound_rank
    int* my_n = seg_n + r * chunks + chunk;
    // (greedy rows need no candidates; k beyond the chunks is not for these kernels)
    const bool listed = any && temp > 0.f && k > 0 && k <= chunks && chunks <= 2 * PULSE_WAVE;
    if (any && !listed && threadIdx.x == 0) *my_n = 0;
    if (!listed && !weighed) return;
    float xs[CHUNK_PER];
    chunk_values(row, chunk * SIMPLE_CHUNK, xs);
    const float best = simple_row_max(part_max + r * chunks, chunks);
    if (listed && wave == 0) {     // the k-th largest of the chunks' maxima, bit by bit (chunks <= 2 * 64: two a lane)
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
    if (weighed && best != -INFINITY) {
        const float inv_t = 1.0f / temp;
        float mass = 0.f;
#pragma unroll
        for (int u = 0; u < CHUNK_PER; ++u)
            if (xs[u] != -INFINITY) mass += expf((xs[u] - best) * inv_t);
        mass = wave_sum(mass);
        if (lane == 0) s_mass[wave] = mass;
    }
    __syncthreads();
    if (weighed && best != -INFINITY && threadIdx.x == 0) {
        float total = 0.f;
        for (int w = 0; w < WAVES; ++w) total += s_mass[w];
        part_mass[r * chunks + chunk] = total;
    }
    if (!listed) return;
    const float bound = s_bound;
    bool taken[CHUNK_PER];
#pragma unroll
    for (int u = 0; u < CHUNK_PER; ++u) taken[u] = xs[u] != -INFINITY && xs[u] >= bound;
    int place[CHUNK_PER], total;
    chunk_places(taken, s_count, place, total);
    const int64_t segment = (static_cast<int64_t>(r) * chunks + chunk) * TOPK_SEGMENT;
#pragma unroll
    for (int u = 0; u < CHUNK_PER; ++u)
        if (place[u] >= 0 && place[u] < TOPK_SEGMENT) {
            seg_i[segment + place[u]] = chunk * SIMPLE_CHUNK + u * SIMPLE_THREADS + static_cast<int>(threadIdx.x);
            seg_x[segment + place[u]] = xs[u];
        }
    if (threadIdx.x == 0) *my_n = total;   // more than TOPK_SEGMENT: the row does not fit
}

// The chunks' segments strung together in LDS: chunk c's entries go to places first[c] .. first[c + 1] - 1.  Eight a thread are asked
// for together (a lane that fetched its chunk's entries one after the other took 15 of the choice's 26 us).
template <int THREADS>
__device__ __forceinline__ void string_segments(const int* seg_i, const float* seg_x, const int* first, int chunks, int* list_i, float* list_x) {
    constexpr int AHEAD = 8;
    for (int q0 = threadIdx.x; q0 < chunks * TOPK_SEGMENT; q0 += AHEAD * THREADS) {
        int to[AHEAD], i[AHEAD];
        float x[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int q = q0 + u * THREADS, c = min(q / TOPK_SEGMENT, chunks - 1), e = q - c * TOPK_SEGMENT;
            to[u] = e < first[c + 1] - first[c] ? first[c] + e : -1;
            i[u] = to[u] >= 0 ? seg_i[q] : 0;
            x[u] = to[u] >= 0 ? seg_x[q] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (to[u] >= 0) { list_i[to[u]] = i[u]; list_x[to[u]] = x[u]; }
    }
}

// How the choice in chunks leaves a row, in `done`: its token is chosen; left; left with so large a k that no segments will hold its
// list (half full on average), for a workgroup alone, which goes by the histogram of the whole row, or, where a workgroup's own
// passes over a short row cost no more than that, without it.
enum { LEFT = 0, CHOSEN = 1, LEFT_COUNTED = 2, LEFT_ALONE = 3 };

// What rest_kernel adds a row's histogram to, and that the row's token is not chosen.
__device__ __forceinline__ void clear_rest(int* rest) {
    for (int b = threadIdx.x; b <= REST_CHOSEN; b += blockDim.x) rest[b] = 0;
}

// The choice of every row from what the kernels before left, a workgroup a row: the largest logit for greedy rows;
// for rows with top-k the candidates' segments strung together in LDS and finished there; for rows that draw from the
// whole vocabulary the chunk in which u * mass falls (chunk masses in chunk order), walked alone.  done[r] says
// whether the row's token is chosen; the others (rows that did not fit) are left_kernel's.
// The four wavefronts fetch (segments, the walked chunk's logits and their weights) and make the steps' sums; what is chosen is one
// wavefront's business, the others reach the same decisions up to there.  (A wavefront alone on its row waited out five trips to memory
// for the segments and branched on every chunk's mass: 32 rows 20.6 -> 10.9 us at a temperature, 13.1 -> 10.6 with top-k 50, 21.7 -> 11.7
// with all options.)
constexpr int CHOOSE_THREADS = 256;
__global__ __launch_bounds__(CHOOSE_THREADS) void chunked_choose_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, const float* __restrict__ part_max,
    const int* __restrict__ part_idx, const float* __restrict__ part_mass, const int* __restrict__ seg_i,
    const float* __restrict__ seg_x, const int* __restrict__ seg_n, int chunks, int* __restrict__ out,
    int* __restrict__ done, int* __restrict__ left) {
    __shared__ int list_i[LIST_CAP];
    __shared__ float list_x[LIST_CAP];
    __shared__ int first_s[2 * PULSE_WAVE + 1];
    constexpr int STEPS = SIMPLE_CHUNK / PULSE_WAVE, MINE = STEPS / (CHOOSE_THREADS / PULSE_WAVE);
    static_assert(LIST_CAP >= SIMPLE_CHUNK && STEPS <= PULSE_WAVE, "a chunk's weights fit the list, its steps' sums a wavefront");
    __shared__ float sums_s[STEPS];
    const int r = blockIdx.x, lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    // (the row's options, and what its chunks left, are asked for together)
    const float temp = temperature ? temperature[r] : 0.f;
    const int k = top_k ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 0.f;
    const float u = temperature ? uniform[r] : 0.f;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    part_max += r * chunks;
    part_idx += r * chunks;
    part_mass += r * chunks;
    seg_n += r * chunks;
    const int at1 = lane + PULSE_WAVE;
    const float mass0 = lane < chunks ? part_mass[lane] : 0.f, mass1 = at1 < chunks ? part_mass[at1] : 0.f;     // (a greedy row's: not written, not used)
    const int n0 = lane < chunks ? seg_n[lane] : 0, n1 = at1 < chunks ? seg_n[at1] : 0;                         // (without top-k and top-p: nor these)
    // the largest logit, the lowest index among equals
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    for (int c = lane; c < chunks; c += PULSE_WAVE) {
        const float v = part_max[c];
        const int i = part_idx[c];
        if (v > best || (v == best && i < best_i)) { best = v; best_i = i; }
    }
    wave_argmax(best, best_i);
    if (best_i == 0x7fffffff || !(temp > 0.f)) {   // everything banned or NaN, or the largest logit wins
        if (threadIdx.x == 0) { out[r] = best_i == 0x7fffffff ? -1 : best_i; done[r] = 1; }
        return;
    }
    const bool use_p = p > 0.f && p < 1.f;
    const float inv_t = 1.0f / temp;
    if (k > 0 || use_p) {
        const bool by_k = k > 0;
        // the segments' places in the list: an exclusive sum over the chunks, in chunk order (two chunks a lane)
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
            // not a row for these kernels
            if (threadIdx.x == 0) done[r] = !by_k || k <= chunks * (TOPK_SEGMENT / 2) ? LEFT : vocab >= 1024 * static_cast<int64_t>(gridDim.x) ? LEFT_COUNTED : LEFT_ALONE;
            if (left) clear_rest(left + static_cast<int64_t>(r) * REST_WORDS);
            return;
        }
        float whole = 0.f;   // without top-k: the mass of the whole row, chunk masses in chunk order
        if (!by_k) {
            whole = wave_sum(mass0 + mass1);     // (at most 2 * 64 chunks here)
        }
        if (wave == 0) {
            first_s[lane] = pre0 - n0;
            first_s[lane + PULSE_WAVE] = first + pre1 - n1;
            if (lane == 0) first_s[2 * PULSE_WAVE] = n;
        }
        __syncthreads();
        const int64_t segment = static_cast<int64_t>(r) * chunks * TOPK_SEGMENT;
        string_segments<CHOOSE_THREADS>(seg_i + segment, seg_x + segment, first_s, chunks, list_i, list_x);
        __syncthreads();
        if (wave != 0) return;
        int token;
        const bool enough =   // (false only without top-k: the list does not hold top_p of the row)
            n <= 4 * PULSE_WAVE   // the usual case with top-k: a few dozen candidates, a few a lane; top-p alone has some hundreds
                ? finish_on_list<4>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, u, best_i, token)
                : n <= 12 * PULSE_WAVE
                ? finish_on_list<12>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, u, best_i, token)
                : finish_on_list<LIST_PER_LANE>(list_i, list_x, n, by_k, k, use_p, p, whole, best, inv_t, u, best_i, token);
        if (lane == 0) {
            if (enough) out[r] = token;
            done[r] = enough ? 1 : 0;
        }
        if (left && !enough)      // (by this wavefront alone)
            for (int b = lane; b <= REST_CHOSEN; b += PULSE_WAVE) left[static_cast<int64_t>(r) * REST_WORDS + b] = 0;
        return;
    }
    // a draw from the whole vocabulary: the chunk in which it falls, chunk masses in chunk order
    float total = mass0;
    for (int c = lane + PULSE_WAVE; c < chunks; c += PULSE_WAVE) total += c < 2 * PULSE_WAVE ? mass1 : part_mass[c];
    total = wave_sum(total);
    const float target = u * total;
    float run = 0.f, rest = 0.f;
    int who = -1, last_chunk = -1;
    // (every lane the same additions, 64 masses at a time, lane j keeping the sum before the j-th: a branch an addition took three times as long)
    for (int base = 0; base < chunks && who < 0; base += PULSE_WAVE) {
        const float mine = base == 0 ? mass0 : base == PULSE_WAVE ? mass1 : base + lane < chunks ? part_mass[base + lane] : 0.f;
        float before = 0.f;
#pragma unroll 8
        for (int j = 0; j < PULSE_WAVE; ++j) {
            before = lane == j ? run : before;
            run += __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_readlane(__float_as_int(mine), j)));
        }
        const unsigned long long has = __ballot(mine > 0.f), hit = __ballot(mine > 0.f && target < before + mine);
        if (hit != 0ull) {
            const int j = __builtin_ctzll(hit);
            who = base + j;
            rest = target - __shfl(before, j, PULSE_WAVE);
        } else if (has != 0ull) {
            last_chunk = base + 63 - __builtin_clzll(has);
        }
    }
    if (who < 0 && last_chunk < 0) {      // (no weight is a number above zero)
        if (threadIdx.x == 0) { out[r] = best_i; done[r] = CHOSEN; }
        return;
    }
    if (who < 0) {  // rounding left the target beyond the last chunk with mass: its last kept entry
        who = last_chunk;
        rest = INFINITY;
    }
    // The chunk's walk, as wave_walk's: the wavefronts make the weights and the sums of a share of its steps each.
    const int begin = who * SIMPLE_CHUNK;
    float* const weights = list_x;
    float ws[MINE];
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < MINE; ++j) ws[j] = row.at<decltype(masked)::value>(min(begin + (wave * MINE + j) * PULSE_WAVE + lane, vocab - 1));
    });
#pragma unroll
    for (int j = 0; j < MINE; ++j) {
        const int at = (wave * MINE + j) * PULSE_WAVE + lane;
        ws[j] = begin + at < vocab && ws[j] != -INFINITY ? expf((ws[j] - best) * inv_t) : 0.f;
        weights[at] = ws[j];
        const float sum = pairs_sum(ws[j]);
        if (lane == 0) sums_s[wave * MINE + j] = sum;
    }
    __syncthreads();
    if (wave != 0) return;
    int last;
    const int e = wave_walk_summed<STEPS>(weights, sums_s[min(lane, STEPS - 1)], rest, last);
    if (lane == 0) { out[r] = e >= 0 ? begin + e : (last >= 0 ? begin + last : best_i); done[r] = 1; }
}

// ---- the rows that are left ---------------------------------------------------------------------------------------
// A workgroup a row goes over its row at the rate of one compute unit.  What has to be known of the whole row, the histogram
// over [lowest, best], is made by many (the lowest value comes with the maxima, and the histogram is cleared by the kernel that
// leaves the row); with it a row is finished in chunks as well (left_collect_kernel, left_choose), unless a chunk has more
// tokens at the edge than its segment holds: those rows a workgroup goes over alone (sample_row), in the launch that chooses.
// (left_choose by a kernel of its own: every call waits for one launch more, top-p or top-k in 33 to 37 us, 37 to 41.)
// 32 rows of 151,936, six of them flat under top-p alone and six with a k above the number of chunks: these three kernels 35 us,
// where the histogram with float32 masses and sample_kernel's passes took 31 and 128.
// Workgroups for a row's histogram: each adds its bins to the row's, which is what bounds them (32 rows of 151,936 under top-p alone:
// 8 groups 15.1 us, 16 13.4, 32 15.9, 64 24.6; of 32,000: 7.2, 9.0, 12.6, 18.8), unless the rows are few (a whole step of one: 32 groups
// 70.2 us, 16 72.6; of three of 32,000 72.3, 8 groups 74.4).
constexpr int REST_GROUPS = 16, REST_GROUPS_FEW = 32, REST_SPAN = 4096, REST_FEW_ROWS = 8;

// Whether a row is left, and what is known of it.
struct LeftRow {
    bool by_p, ranged;
    int k;               // 0: without top-k
    float p, best, lowest, inv_t, scale;
    __device__ __forceinline__ LeftRow(int r, int vocab, int chunks, const float* temperature, const int* top_k, const float* top_p,
                                       const float* part_max, const float* part_min) {
        const int lane = threadIdx.x % PULSE_WAVE;
        k = top_k ? top_k[r] : 0;
        if (k < 0 || k >= vocab) k = 0;
        p = top_p ? top_p[r] : 0.f;
        by_p = k == 0 && p > 0.f && p < 1.f;
        inv_t = 1.0f / temperature[r];
        best = simple_row_max(part_max + static_cast<int64_t>(r) * chunks, chunks);
        lowest = INFINITY;
        for (int c = lane; c < chunks; c += PULSE_WAVE) lowest = fminf(lowest, part_min[static_cast<int64_t>(r) * chunks + c]);
        lowest = -wave_max(-lowest);
        scale = static_cast<float>(HIST_BINS) / (best - lowest);
        ranged = best > lowest && scale < INFINITY;
    }
};

__global__ __launch_bounds__(SIMPLE_THREADS) void rest_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ penalty, const int* __restrict__ seen_row,
    const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned, int mask_words,
    const float* __restrict__ part_max, const float* __restrict__ part_min, int chunks, const int* __restrict__ done,
    int* __restrict__ rest) {
    __shared__ mass_t hist[HIST_BINS];
    const int r = blockIdx.y;
    if (done[r] == CHOSEN || done[r] == LEFT_ALONE) return;
    rest += static_cast<int64_t>(r) * REST_WORDS;
    for (int b = threadIdx.x; b < HIST_BINS; b += SIMPLE_THREADS) hist[b] = 0;
    const LeftRow left(r, vocab, chunks, temperature, top_k, top_p, part_max, part_min);
    if (blockIdx.x == 0 && threadIdx.x == 0) rest[REST_LOWEST] = __float_as_int(left.lowest);
    __syncthreads();
    if (!left.ranged) return;    // (as sample_row: no histogram)
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    const Weigh weigh(left.best, left.inv_t, vocab);
    const int first = blockIdx.x * SIMPLE_THREADS + threadIdx.x;
    if (left.k > 0)
        sweep(row, first, vocab, static_cast<int>(gridDim.x) * SIMPLE_THREADS, [&](int, float x) {
            if (x != -INFINITY) atomicAdd(&hist[bin_at(x, left.best, left.scale)], static_cast<mass_t>(1));
        });
    else
        sweep(row, first, vocab, static_cast<int>(gridDim.x) * SIMPLE_THREADS, [&](int, float x) {
            if (x != -INFINITY) atomicAdd(&hist[bin_at(x, left.best, left.scale)], weigh(x));
        });
    __syncthreads();
    for (int b = threadIdx.x; b < HIST_BINS; b += SIMPLE_THREADS)
        if (hist[b] != 0) atomicAdd(reinterpret_cast<mass_t*>(rest) + b, hist[b]);
}

// A workgroup a chunk, into the chunk's segment.  Rows with top-k: the entries in the bin in which the k-th largest lies and above
// it, in vocabulary order.  Top-p alone: the entries in the bin of the edge, in any order, and the mass of those above it.  (More
// entries than a segment holds, or no edge: the number says so.)
__global__ __launch_bounds__(SIMPLE_THREADS) void left_collect_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ penalty, const int* __restrict__ seen_row,
    const uint32_t* __restrict__ seen_masks, const uint32_t* __restrict__ banned, int mask_words,
    const float* __restrict__ part_max, const float* __restrict__ part_min, const int* __restrict__ done,
    int* __restrict__ seg_i, float* __restrict__ seg_x, int* __restrict__ seg_n, int* __restrict__ rest) {
    constexpr int WAVES = SIMPLE_THREADS / PULSE_WAVE, PER = CHUNK_PER;
    __shared__ mass_t waves[WAVES], above_s;
    __shared__ int at_s, counts[PER][WAVES];
    const int r = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const int lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    if (done[r] != LEFT) return;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    float xs[PER];        // (asked for first: they travel while the edge is searched)
    chunk_values(row, chunk * SIMPLE_CHUNK, xs);
    const LeftRow left(r, vocab, chunks, temperature, top_k, top_p, part_max, part_min);
    if (left.k == 0 && !left.by_p) return;
    rest += static_cast<int64_t>(r) * REST_WORDS;
    mass_t base = 0, whole = 0;
    const int at = edge_bin<SIMPLE_THREADS>(reinterpret_cast<const mass_t*>(rest), left.p, left.k, waves, &at_s, &above_s, base, whole);
    int* const my_n = seg_n + static_cast<int64_t>(r) * chunks + chunk;
    if (at < 0) {
        if (threadIdx.x == 0) *my_n = TOPK_SEGMENT + 1;
        return;
    }
    const Weigh weigh(left.best, left.inv_t, vocab);
    bool taken[PER];
    mass_t mass = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int bin = xs[j] == -INFINITY ? HIST_BINS : bin_at(xs[j], left.best, left.scale);
        taken[j] = bin == at || (left.k > 0 && bin < at);
        if (!taken[j] && bin < at) mass += weigh(xs[j]);
    }
    mass = mass_sum(mass);
    __syncthreads();      // (what edge_bin left has been read)
    if (lane == PULSE_WAVE - 1) waves[wave] = mass;
    int place[PER], total;
    chunk_places(taken, counts, place, total);
    mass = 0;
    for (int w = 0; w < WAVES; ++w) mass += waves[w];
    const int64_t segment = (static_cast<int64_t>(r) * chunks + chunk) * TOPK_SEGMENT;
#pragma unroll
    for (int j = 0; j < PER; ++j)
        if (place[j] >= 0 && place[j] < TOPK_SEGMENT) {
            seg_i[segment + place[j]] = chunk * SIMPLE_CHUNK + j * SIMPLE_THREADS + static_cast<int>(threadIdx.x);
            seg_x[segment + place[j]] = xs[j];
        }
    if (threadIdx.x != 0) return;
    *my_n = total;
    *reinterpret_cast<mass_t*>(rest + REST_CHUNKS + 2 * chunk) = mass;
    if (chunk == 0) {
        *reinterpret_cast<mass_t*>(rest + REST_BASE) = base;
        *reinterpret_cast<mass_t*>(rest + REST_WHOLE) = whole;
    }
}

// The choice of such a row by a workgroup of THREADS; false if it does not fit.  Top-k: on the strung segments, as sample_row's.
// Top-p alone: the edge among the collected tokens, the chunk in which the draw falls, its token.
template <int THREADS>
__device__ __forceinline__ bool left_choose(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, const float* __restrict__ part_max, const float* __restrict__ part_min,
    const int* __restrict__ part_idx, int chunks, const int* __restrict__ seg_i, const float* __restrict__ seg_x,
    const int* __restrict__ seg_n, int* __restrict__ rest, int* __restrict__ out) {
    constexpr int WAVES = THREADS / PULSE_WAVE, PER = SIMPLE_CHUNK / THREADS;
    __shared__ int list_i[LIST_CAP];
    __shared__ float list_x[LIST_CAP];
    __shared__ int first_s[REST_MOST_CHUNKS + 1], n_s;
    __shared__ mass_t masses[EDGE_CAP], chunk_m[REST_MOST_CHUNKS], waves[WAVES], target_s;
    __shared__ uint32_t keys[EDGE_CAP], best_s;
    __shared__ int who_s;
    const int r = blockIdx.x, lane = threadIdx.x % PULSE_WAVE, wave = threadIdx.x / PULSE_WAVE;
    const LeftRow left(r, vocab, chunks, temperature, top_k, top_p, part_max, part_min);
    if (left.k == 0 && !left.by_p) return false;
    rest += static_cast<int64_t>(r) * REST_WORDS;
    seg_n += static_cast<int64_t>(r) * chunks;
    const int64_t segment = static_cast<int64_t>(r) * chunks * TOPK_SEGMENT;
    if (wave == 0) {      // the segments' places in the list, two neighbouring chunks a lane
        const int n0 = 2 * lane < chunks ? seg_n[2 * lane] : 0, n1 = 2 * lane + 1 < chunks ? seg_n[2 * lane + 1] : 0;
        int pre = n0 + n1;
#pragma unroll
        for (int off = 1; off < PULSE_WAVE; off <<= 1) {
            const int up = __shfl_up(pre, off, PULSE_WAVE);
            if (lane >= off) pre += up;
        }
        first_s[2 * lane] = pre - n0 - n1;
        first_s[2 * lane + 1] = pre - n1;
        const bool over = __ballot(n0 > TOPK_SEGMENT || n1 > TOPK_SEGMENT) != 0ull;
        if (lane == PULSE_WAVE - 1) { n_s = over ? LIST_CAP + 1 : pre; first_s[REST_MOST_CHUNKS] = pre; }
        if (lane == 0) best_s = 0u;
    }
    if (static_cast<int>(threadIdx.x) < chunks) chunk_m[threadIdx.x] = *reinterpret_cast<const mass_t*>(rest + REST_CHUNKS + 2 * threadIdx.x);
    __syncthreads();
    const int n = n_s;
    if (n == 0 || n > (left.k > 0 ? LIST_CAP : EDGE_CAP)) return false;
    string_segments<THREADS>(seg_i + segment, seg_x + segment, first_s, chunks, list_i, list_x);
    __syncthreads();
    if (left.k > 0) {
        if (wave != 0) return true;
        // (where no weight is a number above zero, the largest logit)
        float largest = -INFINITY;
        int best_i = 0x7fffffff;
        for (int c = lane; c < chunks; c += PULSE_WAVE) {
            const float v = part_max[static_cast<int64_t>(r) * chunks + c];
            const int i = part_idx[static_cast<int64_t>(r) * chunks + c];
            if (v > largest || (v == largest && i < best_i)) { largest = v; best_i = i; }
        }
        wave_argmax(largest, best_i);
        const bool use_p = left.p > 0.f && left.p < 1.f;
        int token;            // (with top-k every list is enough)
        if (n <= 8 * PULSE_WAVE) finish_on_list<8>(list_i, list_x, n, true, left.k, use_p, left.p, 0.f, left.best, left.inv_t, uniform[r], best_i, token);
        else finish_on_list<LIST_PER_LANE>(list_i, list_x, n, true, left.k, use_p, left.p, 0.f, left.best, left.inv_t, uniform[r], best_i, token);
        if (lane == 0) { out[r] = token; rest[REST_CHOSEN] = 1; }
        return true;
    }
    const Weigh weigh(left.best, left.inv_t, vocab);
    const float p = left.p;
    for (int e = threadIdx.x; e < n; e += THREADS) {
        keys[e] = order_key(list_x[e]);
        masses[e] = weigh(list_x[e]);
    }
    __syncthreads();
    edge_key(keys, masses, n, THREADS, *reinterpret_cast<const mass_t*>(rest + REST_BASE),
             *reinterpret_cast<const mass_t*>(rest + REST_WHOLE), p, &best_s);
    __syncthreads();
    const uint32_t thr = best_s;
    if (thr == 0u) return false;
    for (int e = threadIdx.x; e < n; e += THREADS)
        if (keys[e] >= thr) atomicAdd(&chunk_m[list_i[e] / SIMPLE_CHUNK], masses[e]);
    __syncthreads();
    if (wave == 0) {      // the chunk in which u of the kept mass falls, two chunks a lane
        const mass_t m0 = 2 * lane < chunks ? chunk_m[2 * lane] : 0, m1 = 2 * lane + 1 < chunks ? chunk_m[2 * lane + 1] : 0;
        const mass_t through = mass_through(m0 + m1), target = draw_from(uniform[r], __shfl(through, PULSE_WAVE - 1, PULSE_WAVE));
        mass_t before = through - m0 - m1;
        if (target >= before && target < through) {                    // (target is less than all of it: one lane)
            const bool second = target >= before + m0;
            who_s = 2 * lane + (second ? 1 : 0);
            target_s = target - before - (second ? m0 : 0);
        }
    }
    __syncthreads();
    const int begin = who_s * SIMPLE_CHUNK + static_cast<int>(threadIdx.x) * PER;
    const RowView row = simple_row(logits, r, row_stride, vocab, penalty, seen_row, seen_masks, banned, mask_words);
    mass_t ms[PER], mine = 0;
    by_mask(row, [&](auto masked) __attribute__((always_inline)) {
        float xs[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) xs[j] = begin + j < vocab ? row.at<decltype(masked)::value>(begin + j) : -INFINITY;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            ms[j] = xs[j] != -INFINITY && order_key(xs[j]) >= thr ? weigh(xs[j]) : 0;
            mine += ms[j];
        }
    });
    const mass_t through = mass_through(mine);
    if (lane == PULSE_WAVE - 1) waves[wave] = through;
    __syncthreads();
    mass_t before = through - mine;
    for (int w = 0; w < wave; ++w) before += waves[w];
    const mass_t target = target_s;
    if (target >= before && target < before + mine) {                  // one thread has it
        int j = 0;
        while (target >= before + ms[j]) before += ms[j++];
        out[r] = begin + j;
        rest[REST_CHOSEN] = 1;
    }
    return true;
}

// The rows that are left: by what the kernels before collected, else by their workgroup alone.
__global__ __launch_bounds__(SAMPLE_THREADS) void left_kernel(
    const float* __restrict__ logits, int vocab, int64_t row_stride, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ uniform,
    const float* __restrict__ penalty, const int* __restrict__ seen_row, const uint32_t* __restrict__ seen_masks,
    const uint32_t* __restrict__ banned, int mask_words, const float* __restrict__ part_max, const float* __restrict__ part_min,
    const int* __restrict__ part_idx, int chunks, const int* __restrict__ done, const int* __restrict__ seg_i, const float* __restrict__ seg_x,
    const int* __restrict__ seg_n, int* __restrict__ rest, int* __restrict__ out) {
    const int how = done[blockIdx.x];
    if (how == CHOSEN) return;
    if (rest && how == LEFT && chunks <= REST_MOST_CHUNKS &&
        left_choose<SAMPLE_THREADS>(logits, vocab, row_stride, temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned,
                                    mask_words, part_max, part_min, part_idx, chunks, seg_i, seg_x, seg_n, rest, out)) return;
    __syncthreads();
    sample_row(logits, vocab, row_stride, temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, out, true,
               part_max, part_idx, chunks, how == LEFT_ALONE ? nullptr : rest);
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
                       temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, out);
    PULSE_LAUNCH_CHECK("sample");
    return 0;
}

// A request's options, as its rows bring them to every step.
struct SampleRow {
    float temperature;
    int32_t top_k;
    float top_p, penalty;
    uint64_t seed;
    int32_t seeded, unused;
};
static_assert(sizeof(SampleRow) == 32, "the rows lie one after the other");

static uint64_t splitmix64(uint64_t x) {
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// The options of a step's rows as the kernels read them, host memory [6, room]: temperature, top_k, top_p, the uniform number that
// depends on the row's seed and counter alone, penalty, slot (-1 without a penalty).
// `numbers`: the rows' slots, then their counters; `seeds`: for rows without one of their own (null: none is).  `kinds`: 1 if a row uses top-k, 2
// top-p, 4 a penalty.  (The host's part of a step of 32 rows up to its last launch, 78 us with this in the interpreter, 43 so.)
extern "C" int pulse_sample_options(const void* params, const int64_t* numbers, const uint64_t* seeds, int rows, int32_t* host, int64_t room,
                                    int* kinds) {
    PULSE_REQUIRE(rows >= 0 && room >= rows && host && kinds && (rows == 0 || (params && numbers)), "sample_options: bad arguments");
    float* const floats = reinterpret_cast<float*>(host);
    *kinds = 0;
    for (int r = 0; r < rows; ++r) {
        SampleRow p;
        memcpy(&p, static_cast<const char*>(params) + sizeof(SampleRow) * r, sizeof(p));
        PULSE_REQUIRE(p.seeded || seeds, "sample_options: row %d has no seed", r);
        const uint64_t z = splitmix64(splitmix64(p.seeded ? p.seed : seeds[r]) ^
                                      (static_cast<uint64_t>(numbers[static_cast<int64_t>(rows) + r]) * 0xD1342543DE82EF95ull));
        const bool penalized = p.penalty > 0.f;
        floats[r] = p.temperature;
        host[room + r] = p.top_k;
        floats[2 * room + r] = p.top_p;
        floats[3 * room + r] = static_cast<float>(z >> 40) / static_cast<float>(1 << 24);
        floats[4 * room + r] = p.penalty;
        host[5 * room + r] = penalized ? static_cast<int32_t>(numbers[r]) : -1;
        *kinds |= (p.top_k > 0 ? 1 : 0) | (p.top_p > 0.f && p.top_p < 1.f ? 2 : 0) | (penalized ? 4 : 0);
    }
    return 0;
}

// The same in chunks of the vocabulary with a workgroup each, which reads a row many times faster than the
// workgroup a row of pulse_sample does.  Greedy rows, rows that draw from the whole vocabulary at their temperature
// rows with top-k (and top-p on what it keeps) whose k is at most the number of chunks and rows with top-p alone whose
// top_p share lies in some hundreds of the largest logits are chosen by these kernels; rows that do not fit (a larger k, a
// distribution too flat for top-p alone) by three more that go by a histogram of the row, the last of which takes what does not fit
// these either (many equal values at the edge, a k beyond half of what the segments hold) as pulse_sample does.  What a row's choice
// is does not depend on the other rows.  Whole steps of rows with
// mixed options, the host's part among it, us, before the histogram's kernels finished rows: 32,000 values, 3 / 16 / 64 rows
// 139 / 155 / 191 -> 93 / 119 / 162; 151,936 values 212 / 247 / 331 -> 101 / 130 / 202.  (32 rows of 151,936 since masses and candidates
// come from one reading and the options are put together in native code: 160 -> 101.)
// Scratch, with chunks = pulse_sample_chunks(vocab): part_max, part_mass (float32), part_idx, seg_n (int32) of rows * chunks entries; seg_i (int32), seg_x (float32) of rows * chunks * pulse_sample_segment()
// entries; done (int32) of rows entries; and, optional (null: the rows that are left are gone over by their own workgroups
// alone, with the same choices, as where it does not start at a multiple of 8 bytes), rest (int32) of rows *
// (pulse_sample_rest() + chunks) entries.
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
    const bool prepare = rest && leaves && reinterpret_cast<uintptr_t>(rest) % alignof(mass_t) == 0;
    if (!prepare) rest = nullptr;
    // (behind what is made of the rows: the chunks' smallest numbers)
    float* part_min = prepare ? reinterpret_cast<float*>(rest + static_cast<int64_t>(rows) * REST_WORDS) : nullptr;
    hipLaunchKernelGGL(simple_max_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                       penalty, seen_row, seen_masks, banned, mask_words, part_max, part_idx, part_min);
    PULSE_LAUNCH_CHECK("sample_chunked (maxima)");
    if (temperature) {
        hipLaunchKernelGGL(chunk_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab, row_stride, temperature,
                           top_k, top_p, penalty, seen_row, seen_masks, banned, mask_words, part_max, part_mass, seg_i, seg_x, seg_n);
        PULSE_LAUNCH_CHECK("sample_chunked (masses and candidates)");
    }
    hipLaunchKernelGGL(chunked_choose_kernel, dim3(rows), dim3(CHOOSE_THREADS), 0, stream, logits, vocab, row_stride,
                       temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, part_max,
                       part_idx, part_mass, seg_i, seg_x, seg_n, chunks, out, done, rest);
    PULSE_LAUNCH_CHECK("sample_chunked (choice)");
    if (prepare) {
        const int groups = rows <= REST_FEW_ROWS ? REST_GROUPS_FEW : min(REST_GROUPS, (vocab + REST_SPAN - 1) / REST_SPAN);
        hipLaunchKernelGGL(rest_kernel, dim3(groups, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab, row_stride, temperature,
                           top_k, top_p, penalty, seen_row, seen_masks, banned, mask_words, part_max, part_min, chunks,
                           static_cast<const int*>(done), rest);
        if (chunks <= REST_MOST_CHUNKS) {
            hipLaunchKernelGGL(left_collect_kernel, dim3(chunks, rows), dim3(SIMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                               temperature, top_k, top_p, penalty, seen_row, seen_masks, banned, mask_words, part_max, part_min,
                               static_cast<const int*>(done), seg_i, seg_x, seg_n, rest);
        }
        PULSE_LAUNCH_CHECK("sample_chunked (what is left)");
    }
    if (leaves) {
        hipLaunchKernelGGL(left_kernel, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, logits, vocab, row_stride,
                           temperature, top_k, top_p, uniform, penalty, seen_row, seen_masks, banned, mask_words, part_max, part_min,
                           static_cast<const int*>(part_idx), chunks, static_cast<const int*>(done), static_cast<const int*>(seg_i),
                           static_cast<const float*>(seg_x), static_cast<const int*>(seg_n), rest, out);
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
