// One pass over the fused projection output of a step: per-head RMSNorm of q
// and k, rotation of q and k by the position table, q written back in place,
// k and v written into their cache pages.
//
// Cache layout per (page, kv head): K is [page_size, head_dim] (a key's
// elements contiguous), V is [head_dim, page_size] (a channel's keys
// contiguous), which is what the attention kernels' matrix-core operands want.
//
// Replaces five launches of the reference (q_norm, k_norm, two rotations, the
// page write: src/model/qwen3/model.cpp:815-848; formulas
// src/ops/kernels/cuda/rmsnorm_kernel.cu:97-157, rope_kernel.cu:76-132,
// paged_kv_write.cu:31-52).  Norm and rotation are float32 with one rounding.
//
// Options beyond that: the norm may have no weights (a division by the head's root mean square alone); q may be
// multiplied by a temperature that grows with the position, 1 + coef * ln(floor((pos + 1) / every) + 1), in float32
// after the norm; and the values may be taken from any head-sized columns of the row (`v_head0`: the head number at
// which they start), e.g. from the raw key columns for a design whose values are its keys as projected.
#include "common.h"

#include <algorithm>

namespace {

constexpr int MAX_PAIRS_PER_LANE = 4;  // head_dim <= 512

struct QkRopeArgs {
    int nq, nkv, d;
    int64_t row_stride;
    float eps;
    int rotary_dim;  // 0: no rotation
    int pairing;     // 0: (2i, 2i+1)   1: (i, i + rotary_dim/2)
    int page_size, num_pages, bt_width;
    int write_kv;
    int norm;        // 0: none   1: with the weights q_w / k_w   2: without weights
    int v_head0;     // the values of kv head g are columns (v_head0 + g) * d .. of the row
    float temp_coef; // query temperature: q *= 1 + temp_coef * ln(floor((pos + 1) / temp_every) + 1); temp_every 0: none
    int temp_every;
    const float* parts;      // the rows as float32 shares of the projection, added up here in their order; null: qkv's
    int shares;
    int64_t part_stride, part_row;
};

// The factor of the query temperature at a position (1 when there is none).
__device__ __forceinline__ float query_temperature(const QkRopeArgs& a, int pos) {
    if (a.temp_every <= 0) return 1.f;
    return 1.f + a.temp_coef * logf(static_cast<float>((pos + 1) / a.temp_every) + 1.f);
}

template <typename TX, typename TW, typename TC>
__global__ __launch_bounds__(64) void qk_rope_kv_kernel(TX* __restrict__ qkv, const TW* __restrict__ q_w,
                                                        const TW* __restrict__ k_w, const float* __restrict__ cos_t,
                                                        const float* __restrict__ sin_t, TC* __restrict__ kcache,
                                                        TC* __restrict__ vcache, const int* __restrict__ positions,
                                                        const int* __restrict__ token_entry,
                                                        const int* __restrict__ block_table, QkRopeArgs a) {
    const int t = blockIdx.x;
    const int hh = blockIdx.y;
    const int lane = threadIdx.x;
    const int d = a.d;
    const int half_rot = a.rotary_dim / 2;
    const bool is_q = hh < a.nq;
    const int g = hh - a.nq;
    TX* row = qkv + static_cast<int64_t>(t) * a.row_stride;
    TX* x = is_q ? row + static_cast<int64_t>(hh) * d : row + static_cast<int64_t>(a.nq + g) * d;
    const TW* w = is_q ? q_w : k_w;

    // Every load is issued before anything waits for one: the head's elements, the norm weight, cos and sin, the
    // value head, and the chain position -> block table -> page.  A wavefront lives for little more than one trip
    // to memory then, and the kernel is bound by that time.
    int ia[MAX_PAIRS_PER_LANE], ib[MAX_PAIRS_PER_LANE];
    float xa[MAX_PAIRS_PER_LANE], xb[MAX_PAIRS_PER_LANE], wa[MAX_PAIRS_PER_LANE], wb[MAX_PAIRS_PER_LANE];
    float cs[MAX_PAIRS_PER_LANE], sn[MAX_PAIRS_PER_LANE];
    const int npairs = d / 2;
#pragma unroll
    for (int r = 0; r < MAX_PAIRS_PER_LANE; ++r) {
        const int p = lane + r * PULSE_WAVE;
        ia[r] = ib[r] = 0;
        xa[r] = xb[r] = 0.f;
        wa[r] = wb[r] = cs[r] = 1.f;
        sn[r] = 0.f;
        if (p < npairs) {
            if (p < half_rot) {
                ia[r] = a.pairing == 0 ? 2 * p : p;
                ib[r] = a.pairing == 0 ? 2 * p + 1 : p + half_rot;
                if (cos_t) {
                    cs[r] = cos_t[static_cast<int64_t>(t) * half_rot + p];
                    sn[r] = sin_t[static_cast<int64_t>(t) * half_rot + p];
                }
            } else {
                ia[r] = a.rotary_dim + 2 * (p - half_rot);
                ib[r] = ia[r] + 1;
            }
            xa[r] = to_f32<TX>(x[ia[r]]);
            xb[r] = to_f32<TX>(x[ib[r]]);
            if (w) {
                wa[r] = to_f32<TW>(w[ia[r]]);
                wb[r] = to_f32<TW>(w[ib[r]]);
            }
        }
    }
    float vv[2 * MAX_PAIRS_PER_LANE];
    int pos = 0, entry = 0;
    if (is_q && a.temp_every > 0) pos = positions[t];
    if (!is_q) {
        pos = positions[t];
        entry = token_entry[t];
        const TX* v = row + static_cast<int64_t>(a.v_head0 + g) * d;
#pragma unroll
        for (int r = 0; r < 2 * MAX_PAIRS_PER_LANE; ++r) {
            const int i = lane + r * PULSE_WAVE;
            vv[r] = i < d ? to_f32<TX>(v[i]) : 0.f;
        }
    }

    // where a key goes
    int64_t kbase = 0, vbase = 0;
    bool store_kv = false;
    if (!is_q) {
        const int page = block_table[static_cast<int64_t>(entry) * a.bt_width + pos / a.page_size];
        const int slot = pos % a.page_size;
        store_kv = page >= 0 && page < a.num_pages;
        const int64_t pg = static_cast<int64_t>(page) * a.nkv + g;
        kbase = (pg * a.page_size + slot) * d;
        vbase = pg * d * a.page_size + slot;
    }

    float inv = 1.f;
    if (a.norm) {
        float ss = 0.f;
#pragma unroll
        for (int r = 0; r < MAX_PAIRS_PER_LANE; ++r) ss += xa[r] * xa[r] + xb[r] * xb[r];
        ss = wave_sum(ss);
        inv = 1.0f / sqrtf(ss / static_cast<float>(d) + a.eps);
    }
    const float temp = is_q ? query_temperature(a, pos) : 1.f;

#pragma unroll
    for (int r = 0; r < MAX_PAIRS_PER_LANE; ++r) {
        const int p = lane + r * PULSE_WAVE;
        if (p < npairs) {
            float va = xa[r], vb = xb[r];
            if (a.norm) {
                va = va * inv * wa[r];
                vb = vb * inv * wb[r];
            }
            if (a.temp_every > 0) {
                va *= temp;
                vb *= temp;
            }
            if (p < half_rot && cos_t) {
                const float ra = va * cs[r] - vb * sn[r];
                const float rb = va * sn[r] + vb * cs[r];
                va = ra;
                vb = rb;
            }
            if (is_q) {
                x[ia[r]] = from_f32<TX>(va);
                x[ib[r]] = from_f32<TX>(vb);
            } else if (store_kv) {
                kcache[kbase + ia[r]] = from_f32<TC>(va);
                kcache[kbase + ib[r]] = from_f32<TC>(vb);
            }
        }
    }

    if (!is_q && store_kv) {
#pragma unroll
        for (int r = 0; r < 2 * MAX_PAIRS_PER_LANE; ++r) {
            const int i = lane + r * PULSE_WAVE;
            if (i < d) vcache[vbase + static_cast<int64_t>(i) * a.page_size] = from_f32<TC>(vv[r]);
        }
    }
}


// The bfloat16 path: a head's row of d elements is taken by d / 8 lanes with 16-byte accesses (8 elements a lane),
// so a wavefront takes 64 / LPH heads of one token at once and runs a tenth of the instructions of the kernel
// above, which is what that kernel's time goes to on long prompts.  The sum of squares runs over the LPH lanes of
// a head.  Needs d and rotary_dim to be multiples of 8, LPH = the power of two >= d / 8 (at most 64).
// PAIRING 0: a lane's pairs are (e0, e1) .. (e6, e7) of 8 consecutive elements.  PAIRING 1: a lane takes elements
// 4c .. 4c+3 and their partners half a rotary_dim further on.  Elements beyond rotary_dim are not rotated.
typedef __attribute__((ext_vector_type(4))) float vf4;
typedef __attribute__((ext_vector_type(4))) uint32_t vu4;
typedef __attribute__((ext_vector_type(2))) uint32_t vu2;

template <typename TW>
__device__ __forceinline__ void load8(const TW* p, float (&out)[8]);
template <>
__device__ __forceinline__ void load8<bf16_t>(const bf16_t* p, float (&out)[8]) {
    const vu4 raw = *reinterpret_cast<const vu4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[2 * i] = __uint_as_float(raw[i] << 16);
        out[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
    }
}
template <>
__device__ __forceinline__ void load8<float>(const float* p, float (&out)[8]) {
    const vf4 lo = *reinterpret_cast<const vf4*>(p);
    const vf4 hi = *reinterpret_cast<const vf4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[i] = lo[i];
        out[4 + i] = hi[i];
    }
}
template <typename TW>
__device__ __forceinline__ void load4(const TW* p, float* out);
template <>
__device__ __forceinline__ void load4<bf16_t>(const bf16_t* p, float* out) {
    const vu2 raw = *reinterpret_cast<const vu2*>(p);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        out[2 * i] = __uint_as_float(raw[i] << 16);
        out[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
    }
}
template <>
__device__ __forceinline__ void load4<float>(const float* p, float* out) {
    const vf4 v = *reinterpret_cast<const vf4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = v[i];
}

// Four neighbouring values of a row's shares, added up in their order (four shares are asked for together; past the last: the last
// again, for nobody).
__device__ __forceinline__ vf4 sum4(const float* p, int shares, int64_t part_stride) {
    constexpr int AHEAD = 4;
    vf4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < shares; s0 += AHEAD) {
        vf4 v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = *reinterpret_cast<const vf4*>(p + min(s0 + u, shares - 1) * part_stride);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (s0 + u < shares) sum += v[u];
    }
    return sum;
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return static_cast<uint32_t>(f32_to_bf16(lo)) | (static_cast<uint32_t>(f32_to_bf16(hi)) << 16);
}

// One wavefront of it: the heads from number `y` * 64 / LPH on of token t.
template <typename TW, int PAIRING, int LPH, bool PARTS>
__device__ __forceinline__ void qk_rope_rows(int t, int y, int lane, bf16_t* __restrict__ qkv, const TW* __restrict__ q_w,
                                             const TW* __restrict__ k_w, const float* __restrict__ cos_t,
                                             const float* __restrict__ sin_t, bf16_t* __restrict__ kcache,
                                             const int* __restrict__ positions, const int* __restrict__ token_entry,
                                             const int* __restrict__ block_table, const QkRopeArgs& a) {
    constexpr int HPW = PULSE_WAVE / LPH;
    const int c = lane % LPH;
    const int hh = y * HPW + lane / LPH;
    const int heads = a.write_kv ? a.nq + a.nkv : a.nq;
    const int d = a.d;
    const int half_rot = a.rotary_dim / 2;
    const bool on = hh < heads && c * 8 < d;
    const bool is_q = hh < a.nq;
    const int g = hh - a.nq;
    bf16_t* row = qkv + static_cast<int64_t>(t) * a.row_stride;
    bf16_t* x = row + static_cast<int64_t>(on ? hh : 0) * d;  // q heads, then k heads, one after the other
    const TW* w = is_q ? q_w : k_w;

    // which elements: two groups of four
    const bool rotated = c * 8 < a.rotary_dim;
    int oa = c * 8, ob = c * 8 + 4;  // PAIRING 0, and everything beyond rotary_dim
    if (PAIRING == 1 && rotated) {
        oa = c * 4;
        ob = c * 4 + half_rot;
    }
    if (!on) oa = 0, ob = 4;

    // every load before anything waits for one
    float e[8], wv[8], cs[4], sn[4];
    if constexpr (PARTS) {
        const float* part = a.parts + static_cast<int64_t>(t) * a.part_row + static_cast<int64_t>(on ? hh : 0) * d;
        const vf4 lo = sum4(part + oa, a.shares, a.part_stride), hi = sum4(part + ob, a.shares, a.part_stride);
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = lo[i], e[4 + i] = hi[i];
    } else if (PAIRING == 0) {
        load8<bf16_t>(x + oa, e);
    } else {
        load4<bf16_t>(x + oa, e);
        load4<bf16_t>(x + ob, e + 4);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) wv[i] = 1.f;
    if (w) {
        if (PAIRING == 0) {
            load8<TW>(w + oa, wv);
        } else {
            load4<TW>(w + oa, wv);
            load4<TW>(w + ob, wv + 4);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) cs[i] = 1.f, sn[i] = 0.f;
    if (cos_t && rotated && on) {
        load4<float>(cos_t + static_cast<int64_t>(t) * half_rot + c * 4, cs);
        load4<float>(sin_t + static_cast<int64_t>(t) * half_rot + c * 4, sn);
    }
    const bool is_k = on && !is_q;
    int pos = 0, entry = 0;
    if (a.temp_every > 0) pos = positions[t];
    if (is_k) {
        pos = positions[t];
        entry = token_entry[t];
    }
    bool store_kv = false;
    int64_t kbase = 0;
    if (is_k) {
        const int page = block_table[static_cast<int64_t>(entry) * a.bt_width + pos / a.page_size];
        const int slot = pos % a.page_size;
        store_kv = page >= 0 && page < a.num_pages;
        const int64_t pg = static_cast<int64_t>(page) * a.nkv + g;
        kbase = (pg * a.page_size + slot) * d;
    }

    if (!on) {
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = 0.f;
    }
    float inv = 1.f;
    if (a.norm) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += e[i] * e[i];
        if constexpr (LPH == 16) {
            ss = row_reduce(ss, LaneSum());
        } else {
#pragma unroll
            for (int off = LPH / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, PULSE_WAVE);
        }
        inv = 1.0f / sqrtf(ss / static_cast<float>(d) + a.eps);
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = e[i] * inv * wv[i];
    }
    if (a.temp_every > 0 && is_q) {
        const float temp = query_temperature(a, pos);
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] *= temp;
    }
    if (rotated) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ia = PAIRING == 0 ? 2 * i : i;
            const int ib = PAIRING == 0 ? 2 * i + 1 : i + 4;
            const float va = e[ia], vb = e[ib];
            e[ia] = va * cs[i] - vb * sn[i];
            e[ib] = va * sn[i] + vb * cs[i];
        }
    }
    if (!on) return;
    const vu2 lo = {pack2(e[0], e[1]), pack2(e[2], e[3])};
    const vu2 hi = {pack2(e[4], e[5]), pack2(e[6], e[7])};
    if (is_q) {
        *reinterpret_cast<vu2*>(x + oa) = lo;
        *reinterpret_cast<vu2*>(x + ob) = hi;
    } else if (store_kv) {
        *reinterpret_cast<vu2*>(kcache + kbase + oa) = lo;
        *reinterpret_cast<vu2*>(kcache + kbase + ob) = hi;
    }
}

// The values of the step's tokens into their pages, whose layout has the slots of a page side by side for every
// channel: a workgroup takes 16 consecutive tokens of one kv head, a thread one token (tid % 16) and eight channels
// at a time, so that the 16 lanes of a store write the 16 two-byte slots of one channel, 32 contiguous bytes when
// the tokens fill a page in order (a thread finds its own token's page and slot: any other arrangement is written
// just as correctly, only in smaller pieces).  Written from the kernel above, a token at a time, the same bytes
// took twice as long as everything else that kernel does.
constexpr int VW_TOKENS = 16;
constexpr int VEC_THREADS = 256;

template <bool PARTS>
__device__ __forceinline__ void v_page_rows(int tile, int g, const bf16_t* __restrict__ qkv, bf16_t* __restrict__ vcache,
                                            const int* __restrict__ positions, const int* __restrict__ token_entry,
                                            const int* __restrict__ block_table, const QkRopeArgs& a, int tokens) {
    const int t = tile * VW_TOKENS + threadIdx.x % VW_TOKENS;
    const int cg = threadIdx.x / VW_TOKENS;
    if (t >= tokens) return;
    const int pos = positions[t];
    const int page = block_table[static_cast<int64_t>(token_entry[t]) * a.bt_width + pos / a.page_size];
    if (page < 0 || page >= a.num_pages) return;
    const int slot = pos % a.page_size;
    const int64_t column = static_cast<int64_t>(a.v_head0 + g) * a.d;
    const bf16_t* src = qkv + static_cast<int64_t>(t) * a.row_stride + column;
    bf16_t* dst = vcache + (static_cast<int64_t>(page) * a.nkv + g) * a.d * a.page_size + slot;
    for (int c0 = cg * 8; c0 < a.d; c0 += 8 * (VEC_THREADS / VW_TOKENS)) {
        if constexpr (PARTS) {
            const float* part = a.parts + static_cast<int64_t>(t) * a.part_row + column + c0;
            const vf4 lo = sum4(part, a.shares, a.part_stride), hi = sum4(part + 4, a.shares, a.part_stride);
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[static_cast<int64_t>(c0 + i) * a.page_size] = f32_to_bf16(i < 4 ? lo[i % 4] : hi[i % 4]);
            continue;
        }
        const uint4 raw = *reinterpret_cast<const uint4*>(src + c0);
        const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int i = 0; i < 8; ++i)
            dst[static_cast<int64_t>(c0 + i) * a.page_size] = static_cast<bf16_t>(words[i / 2] >> (16 * (i % 2)));
    }
}

// With PARTS the rows come as float32 shares of the projection (4 bytes a value and share): the lanes ask for four
// shares' pieces of 16 bytes together.  40 heads of 128 at 97 / 160 / 357 tokens: 3.6 / 4.2 / 4.4 us from rounded rows, 4.5 / 5.0 / 8.5
// from four shares (figures of the product and the rotation together, by which it is decided, are at Linear.parts_shares_for).
//
// Both in one launch: the first `rope_groups` workgroups are four wavefronts of rows each, the others 16 tokens' values of a
// kv head.  (Neither reads what the other writes: q's columns are the only ones written in place, and the values are never
// among them.)  Two launches took 4.0 + 2.9 us at 97 tokens, 5.6 + 4.8 at 509, 12.3 + 5.3 at 2,048 (32 + 8 heads of 128);
// one 4.0, 5.7, 15.6.
template <typename TW, int PAIRING, int LPH, bool PARTS>
__global__ __launch_bounds__(VEC_THREADS) void qk_rope_kv_vec_kernel(bf16_t* __restrict__ qkv, const TW* __restrict__ q_w,
                                                                     const TW* __restrict__ k_w,
                                                                     const float* __restrict__ cos_t,
                                                                     const float* __restrict__ sin_t,
                                                                     bf16_t* __restrict__ kcache, bf16_t* __restrict__ vcache,
                                                                     const int* __restrict__ positions,
                                                                     const int* __restrict__ token_entry,
                                                                     const int* __restrict__ block_table, QkRopeArgs a,
                                                                     int tokens, int per_token, int rope_groups) {
    const int b = blockIdx.x;
    if (b < rope_groups) {
        // (fewer than 2^30 rows, see the entry point: a division of 32 bits, by one number for the whole wavefront)
        const unsigned row = __builtin_amdgcn_readfirstlane(b * (VEC_THREADS / PULSE_WAVE) + threadIdx.x / PULSE_WAVE);
        const unsigned t = row / static_cast<unsigned>(per_token);
        if (t >= static_cast<unsigned>(tokens)) return;
        qk_rope_rows<TW, PAIRING, LPH, PARTS>(static_cast<int>(t), static_cast<int>(row - t * per_token), threadIdx.x % PULSE_WAVE, qkv, q_w,
                                       k_w, cos_t, sin_t, kcache, positions, token_entry, block_table, a);
    } else {
        v_page_rows<PARTS>((b - rope_groups) / a.nkv, (b - rope_groups) % a.nkv, qkv, vcache, positions, token_entry, block_table, a,
                    tokens);
    }
}

template <typename TW, int PAIRING, bool PARTS>
void launch_vec(int lph, hipStream_t stream, int tokens, int heads, bf16_t* qkv, const TW* q_w, const TW* k_w,
                const float* cos_t, const float* sin_t, bf16_t* kcache, bf16_t* vcache, const int* positions,
                const int* token_entry, const int* block_table, const QkRopeArgs& a) {
    const int value_groups = a.write_kv ? (tokens + VW_TOKENS - 1) / VW_TOKENS * a.nkv : 0;
#define PULSE_VEC(L)                                                                                                    \
    do {                                                                                                                \
        const int per_token = (heads + 64 / L - 1) / (64 / L);                                                          \
        const int rope_groups = static_cast<int>((static_cast<int64_t>(tokens) * per_token + 3) / 4);                   \
        hipLaunchKernelGGL((qk_rope_kv_vec_kernel<TW, PAIRING, L, PARTS>), dim3(rope_groups + value_groups), dim3(VEC_THREADS), 0, \
                           stream, qkv, q_w, k_w, cos_t, sin_t, kcache, vcache, positions, token_entry, block_table, a,  \
                           tokens, per_token, rope_groups);                                                             \
    } while (0)
    if (lph <= 2) PULSE_VEC(2);
    else if (lph <= 4) PULSE_VEC(4);
    else if (lph <= 8) PULSE_VEC(8);
    else if (lph <= 16) PULSE_VEC(16);
    else if (lph <= 32) PULSE_VEC(32);
    else PULSE_VEC(64);
#undef PULSE_VEC
}

}  // namespace

static int qk_rope_kv(const float* parts, int shares, int64_t part_stride, int64_t part_row, void* qkv, int x_dtype, int64_t row_stride, const void* q_w, const void* k_w,
                                int w_dtype, float eps, const float* cos_t, const float* sin_t, int rotary_dim,
                                int pairing, void* kcache, void* vcache, int c_dtype, const int* positions,
                                const int* token_entry, const int* block_table, int bt_width, int tokens, int nq,
                                int nkv, int d, int page_size, int num_pages, int write_kv, int plain_norm,
                                int v_head0, float temp_coef, int temp_every, hipStream_t stream) {
    PULSE_REQUIRE(tokens >= 0 && nq > 0 && nkv >= 0 && d > 0, "qk_rope_kv: bad sizes");
    PULSE_REQUIRE(d % 2 == 0 && d <= 2 * PULSE_WAVE * MAX_PAIRS_PER_LANE,
                  "qk_rope_kv: head_dim %d must be even and at most %d", d, 2 * PULSE_WAVE * MAX_PAIRS_PER_LANE);
    PULSE_REQUIRE(rotary_dim >= 0 && rotary_dim <= d && rotary_dim % 2 == 0,
                  "qk_rope_kv: rotary_dim %d must be even and at most head_dim %d", rotary_dim, d);
    PULSE_REQUIRE(pairing == 0 || pairing == 1, "qk_rope_kv: unknown pairing %d", pairing);
    PULSE_REQUIRE((q_w == nullptr) == (k_w == nullptr), "qk_rope_kv: give both norm weights or neither");
    PULSE_REQUIRE(!(plain_norm && q_w), "qk_rope_kv: a norm without weights was asked for and weights were given");
    PULSE_REQUIRE(temp_every >= 0, "qk_rope_kv: the query temperature's interval must not be negative");
    PULSE_REQUIRE(rotary_dim == 0 || (cos_t && sin_t), "qk_rope_kv: rotation needs the cos/sin tables");
    PULSE_REQUIRE(pulse_dtype_ok(x_dtype) && pulse_dtype_ok(w_dtype) && pulse_dtype_ok(c_dtype), "qk_rope_kv: bad dtype tag");
    PULSE_REQUIRE(qkv && positions, "qk_rope_kv: null pointer");
    if (write_kv) {
        PULSE_REQUIRE(kcache && vcache && token_entry && block_table, "qk_rope_kv: cache pointers missing");
        PULSE_REQUIRE(page_size > 0 && num_pages > 0 && bt_width > 0 && nkv > 0, "qk_rope_kv: bad cache geometry");
        PULSE_REQUIRE(v_head0 >= 0 && row_stride >= static_cast<int64_t>(nq + nkv) * d &&
                      row_stride >= static_cast<int64_t>(v_head0 + nkv) * d, "qk_rope_kv: row stride too small");
    } else {
        PULSE_REQUIRE(row_stride >= static_cast<int64_t>(nq) * d, "qk_rope_kv: row stride too small");
    }
    if (parts) {
        const int columns = write_kv ? std::max(nq + nkv, v_head0 + nkv) : nq;
        PULSE_REQUIRE(shares > 0 && part_row >= static_cast<int64_t>(columns) * d && part_row % 4 == 0 && part_stride % 4 == 0 &&
                      (shares == 1 || part_stride >= static_cast<int64_t>(tokens - 1) * part_row + static_cast<int64_t>(columns) * d) &&
                      reinterpret_cast<uintptr_t>(parts) % 16 == 0, "qk_rope_kv: %d shares of rows %lld apart overlap or are not aligned",
                      shares, static_cast<long long>(part_row));
    }
    if (tokens == 0) return 0;
    QkRopeArgs a;
    a.parts = parts; a.shares = shares; a.part_stride = part_stride; a.part_row = part_row;
    a.nq = nq; a.nkv = nkv; a.d = d; a.row_stride = row_stride; a.eps = eps;
    a.rotary_dim = (cos_t ? rotary_dim : 0); a.pairing = pairing;
    a.page_size = page_size; a.num_pages = num_pages; a.bt_width = bt_width; a.write_kv = write_kv;
    a.norm = q_w ? 1 : (plain_norm ? 2 : 0); a.v_head0 = v_head0; a.temp_coef = temp_coef; a.temp_every = temp_every;
    const int heads = write_kv ? nq + nkv : nq;
    PULSE_REQUIRE(static_cast<int64_t>(tokens) * heads < (1ll << 30), "qk_rope_kv: %d tokens of %d heads are too many", tokens, heads);
    // the 16-byte path: bfloat16 activations and cache, 8-element chunks that the rotation does not cut
    const bool vec = x_dtype == PULSE_BF16 && (!write_kv || c_dtype == PULSE_BF16) && d % 8 == 0 && a.rotary_dim % 8 == 0 && row_stride % 8 == 0 &&
                     (reinterpret_cast<uintptr_t>(qkv) % 16) == 0 && (reinterpret_cast<uintptr_t>(kcache) % 16) == 0 &&
                     (q_w == nullptr || ((reinterpret_cast<uintptr_t>(q_w) % 16) == 0 && (reinterpret_cast<uintptr_t>(k_w) % 16) == 0)) &&
                     (cos_t == nullptr || ((reinterpret_cast<uintptr_t>(cos_t) % 16) == 0 && (reinterpret_cast<uintptr_t>(sin_t) % 16) == 0));
    if (vec) {
        const int lph = d / 8;
#define PULSE_ROPE(P, S)                                                                                                  \
    launch_vec<TW, P, S>(lph, stream, tokens, heads, static_cast<bf16_t*>(qkv), static_cast<const TW*>(q_w),              \
                         static_cast<const TW*>(k_w), cos_t, sin_t, static_cast<bf16_t*>(kcache),                         \
                         static_cast<bf16_t*>(vcache), positions, token_entry, block_table, a)
        PULSE_DISPATCH_DTYPE(w_dtype, TW,
            if (pairing == 0) { if (parts) PULSE_ROPE(0, true); else PULSE_ROPE(0, false); }
            else { if (parts) PULSE_ROPE(1, true); else PULSE_ROPE(1, false); });
#undef PULSE_ROPE
        PULSE_LAUNCH_CHECK("qk_rope_kv");
        return 0;
    }
    PULSE_REQUIRE(!parts, "qk_rope_kv: shares need bfloat16 rows and pages, aligned and in chunks of eight values");
    const dim3 grid(tokens, heads);
    PULSE_DISPATCH_DTYPE(x_dtype, TX, PULSE_DISPATCH_DTYPE(w_dtype, TW, PULSE_DISPATCH_DTYPE(c_dtype, TC,
        hipLaunchKernelGGL((qk_rope_kv_kernel<TX, TW, TC>), grid, dim3(64), 0, stream, static_cast<TX*>(qkv),
                           static_cast<const TW*>(q_w), static_cast<const TW*>(k_w), cos_t, sin_t,
                           static_cast<TC*>(kcache), static_cast<TC*>(vcache), positions, token_entry,
                           block_table, a))));
    PULSE_LAUNCH_CHECK("qk_rope_kv");
    return 0;
}

extern "C" int pulse_qk_rope_kv(void* qkv, int x_dtype, int64_t row_stride, const void* q_w, const void* k_w,
                                int w_dtype, float eps, const float* cos_t, const float* sin_t, int rotary_dim,
                                int pairing, void* kcache, void* vcache, int c_dtype, const int* positions,
                                const int* token_entry, const int* block_table, int bt_width, int tokens, int nq,
                                int nkv, int d, int page_size, int num_pages, int write_kv, int plain_norm,
                                int v_head0, float temp_coef, int temp_every, hipStream_t stream) {
    return qk_rope_kv(nullptr, 0, 0, 0, qkv, x_dtype, row_stride, q_w, k_w, w_dtype, eps, cos_t, sin_t, rotary_dim, pairing, kcache, vcache, c_dtype, positions,
                      token_entry, block_table, bt_width, tokens, nq, nkv, d, page_size, num_pages, write_kv, plain_norm, v_head0, temp_coef,
                      temp_every, stream);
}

// The same with the projection's rows as `shares` float32 results [tokens, part_row], `part_stride` values apart, that are added up
// in their order (a product whose inner dimension was shared out over workgroups); qkv only receives q.
extern "C" int pulse_qk_rope_kv_parts(const float* parts, int shares, int64_t part_stride, int64_t part_row, void* qkv, int x_dtype, int64_t row_stride, const void* q_w, const void* k_w,
                                int w_dtype, float eps, const float* cos_t, const float* sin_t, int rotary_dim,
                                int pairing, void* kcache, void* vcache, int c_dtype, const int* positions,
                                const int* token_entry, const int* block_table, int bt_width, int tokens, int nq,
                                int nkv, int d, int page_size, int num_pages, int write_kv, int plain_norm,
                                int v_head0, float temp_coef, int temp_every, hipStream_t stream) {
    PULSE_REQUIRE(parts, "qk_rope_kv: null pointer");
    return qk_rope_kv(parts, shares, part_stride, part_row, qkv, x_dtype, row_stride, q_w, k_w, w_dtype, eps, cos_t, sin_t, rotary_dim, pairing, kcache, vcache, c_dtype, positions,
                      token_entry, block_table, bt_width, tokens, nq, nkv, d, page_size, num_pages, write_kv, plain_norm, v_head0, temp_coef,
                      temp_every, stream);
}
