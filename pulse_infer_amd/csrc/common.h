// Shared helpers for the gfx950 kernels: storage types, wave64 reductions and
// the error channel of the C entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include <utility>

// f(0), f(1) .. f(N - 1) with constants (an unrolled loop whatever its size).
template <typename F, int... I>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>()), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each(f, std::make_integer_sequence<int, N>()); }

// Storage type tags used across the C ABI.
enum PulseDType : int { PULSE_F32 = 0, PULSE_BF16 = 1 };

typedef uint16_t bf16_t;  // raw bfloat16 bits

#define PULSE_WAVE 64

// Every entry point returns 0 on success; otherwise a message is left for
// pulse_last_error().  Arguments are checked on the host before any launch.
extern "C" const char* pulse_last_error();
void pulse_set_error(const char* fmt, ...);
int pulse_compute_units();  // of the current device, asked once

#define PULSE_REQUIRE(cond, ...)            \
    do {                                    \
        if (!(cond)) {                      \
            pulse_set_error(__VA_ARGS__);   \
            return 1;                       \
        }                                   \
    } while (0)

#define PULSE_LAUNCH_CHECK(name)                                                  \
    do {                                                                          \
        hipError_t e_ = hipGetLastError();                                        \
        if (e_ != hipSuccess) {                                                   \
            pulse_set_error("%s: launch failed: %s", name, hipGetErrorString(e_)); \
            return 2;                                                             \
        }                                                                         \
    } while (0)

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
    return __uint_as_float(static_cast<uint32_t>(v) << 16);
}

// Round to nearest, ties to even; NaN stays NaN.  (The conversion instruction of gfx950, v_cvt_pk_bf16_f32: one
// instruction for two values where the rounding written out in integer arithmetic takes six a value.)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    return __builtin_bit_cast(bf16_t, static_cast<__bf16>(f));
}

// 16 bytes of a tensor that a kernel reads once (weights, the cache): a load marked nontemporal, which the memory
// system streams instead of keeping in its caches.  A plain read of 2 GB runs at 5.9 TB/s with ordinary loads and at
// 6.4 to 6.6 TB/s with these.
typedef __attribute__((ext_vector_type(4))) int pulse_i32x4;
__device__ __forceinline__ pulse_i32x4 stream_load16(const void* p) {
    return __builtin_nontemporal_load(static_cast<const pulse_i32x4*>(p));
}

// 16 bytes a lane from memory straight into LDS: lane i's piece lands at lds_base + 16 i (a wavefront-wide address), from a
// pointer a lane, or from `offset` bytes behind a base in scalar registers.  The compiler knows nothing of these copies, so
// the waits for them are written out where they are used.
__device__ __forceinline__ void load_to_lds(const void* p, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_base), "v"(p) : "memory", "m0");
}
__device__ __forceinline__ void stream_to_lds(const void* p, uint32_t lds_base) {   // (nontemporal, see stream_load16)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" : : "s"(lds_base), "v"(p) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_base), "v"(offset), "s"(base) : "memory", "m0");
}

// The same in a row: `lds_place` says where, the copies behind it bring 16 bytes a lane from `offset` + BYTES behind the base to BYTES
// behind that place (-4,096 <= BYTES < 4,096), an instruction each.  (The place is kept in M0 from statement to statement, which the compiler does
// not know: the build looks through what it made and refuses kernels in which anything else touches M0, check_m0 of build.py.)
__device__ __forceinline__ void lds_place(uint32_t lds_base) { asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" : : "s"(lds_base) : "memory", "m0"); }
template <int BYTES, bool STREAM = false>
__device__ __forceinline__ void copy_to_place(const void* base, uint32_t offset) {
    if constexpr (STREAM) asm volatile("global_load_lds_dwordx4 %0, %1 offset:%c2 nt" : : "v"(offset), "s"(base), "n"(BYTES) : "memory");
    else asm volatile("global_load_lds_dwordx4 %0, %1 offset:%c2" : : "v"(offset), "s"(base), "n"(BYTES) : "memory");
}

template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t v) { return bf16_to_f32(v); }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return f32_to_bf16(v); }

// The two operands of a step of a reduction over the wavefront: what lanes i and i ^ STEP hold, the same pair (in one order or the
// other) for both.  Steps go 32, 16, 8, 4, 2, 1; below 8 the pair is right once the steps before have been taken (lanes that
// differ in the higher bits then hold the same).  By lane moves in the vector unit: a trip through LDS, which `__shfl_xor` takes,
// is waited for six times a sum.  (The same bits.  Decoding steps of the 8B shape, the norms, the attention's maxima and the sums of
// squares among it: 32 requests 4,790 -> 4,749 us, one 3,263 -> 3,239 where runs of one side differ by 2 us; less than runs differ by on
// a card where that is more.)
struct WaveTwo { uint32_t a, b; };
template <int STEP>
__device__ __forceinline__ WaveTwo wave_two(uint32_t v) {
    if constexpr (STEP == 32 || STEP == 16) {
        const auto both = STEP == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false) : __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return {both[0], both[1]};
    } else {
        return {v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x120 + STEP /* row_ror:STEP */, 0xF, 0xF, true))};
    }
}

// op over all lanes, lanes 32 apart first (every lane gets it; op must not care for its operands' order)
template <typename T, typename F>
__device__ __forceinline__ T wave_reduce(T v, F op) {
    static_assert(sizeof(T) == 4, "a register a lane");
    auto step = [&](WaveTwo t) __attribute__((always_inline)) { v = op(__builtin_bit_cast(T, t.a), __builtin_bit_cast(T, t.b)); };
    step(wave_two<32>(__builtin_bit_cast(uint32_t, v)));
    step(wave_two<16>(__builtin_bit_cast(uint32_t, v)));
    step(wave_two<8>(__builtin_bit_cast(uint32_t, v)));
    step(wave_two<4>(__builtin_bit_cast(uint32_t, v)));
    step(wave_two<2>(__builtin_bit_cast(uint32_t, v)));
    step(wave_two<1>(__builtin_bit_cast(uint32_t, v)));
    return v;
}
// op over the sixteen lanes of a row of lanes, 8 apart first.
template <typename F>
__device__ __forceinline__ float row_reduce(float v, F op) {
    auto step = [&](WaveTwo t) __attribute__((always_inline)) { v = op(__uint_as_float(t.a), __uint_as_float(t.b)); };
    step(wave_two<8>(__float_as_uint(v)));
    step(wave_two<4>(__float_as_uint(v)));
    step(wave_two<2>(__float_as_uint(v)));
    step(wave_two<1>(__float_as_uint(v)));
    return v;
}
// op over the four lanes that hold the same place of their row of sixteen, neighbouring rows first.
template <typename F>
__device__ __forceinline__ float across_rows(float v, F op) {
    const WaveTwo near = wave_two<16>(__float_as_uint(v));
    const WaveTwo far = wave_two<32>(__float_as_uint(op(__uint_as_float(near.a), __uint_as_float(near.b))));
    return op(__uint_as_float(far.a), __uint_as_float(far.b));
}
struct LaneSum { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
struct LaneMax { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
__device__ __forceinline__ float wave_sum(float v) { return wave_reduce(v, LaneSum()); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce(v, LaneMax()); }

__device__ __forceinline__ int wave_sum(int v) { return wave_reduce(v, [](int a, int b) { return a + b; }); }

// The largest value over all lanes and its number, the lowest among equals (numbers only: no NaN).
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
    auto step = [&](WaveTwo x, WaveTwo n) __attribute__((always_inline)) {
        const float a = __uint_as_float(x.a), b = __uint_as_float(x.b);
        const int ia = static_cast<int>(n.a), ib = static_cast<int>(n.b);
        const bool second = b > a || (b == a && ib < ia);
        v = second ? b : a;
        i = second ? ib : ia;
    };
    step(wave_two<32>(__float_as_uint(v)), wave_two<32>(static_cast<uint32_t>(i)));
    step(wave_two<16>(__float_as_uint(v)), wave_two<16>(static_cast<uint32_t>(i)));
    step(wave_two<8>(__float_as_uint(v)), wave_two<8>(static_cast<uint32_t>(i)));
    step(wave_two<4>(__float_as_uint(v)), wave_two<4>(static_cast<uint32_t>(i)));
    step(wave_two<2>(__float_as_uint(v)), wave_two<2>(static_cast<uint32_t>(i)));
    step(wave_two<1>(__float_as_uint(v)), wave_two<1>(static_cast<uint32_t>(i)));
}

// Sum over a block of up to 1024 threads; `scratch` holds one float per wave (>= 16).
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x % PULSE_WAVE;
    const int wave = threadIdx.x / PULSE_WAVE;
    const int nwaves = (blockDim.x + PULSE_WAVE - 1) / PULSE_WAVE;
    v = wave_sum(v);
    __syncthreads();  // scratch may still be read from an earlier call
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < nwaves; ++w) total += scratch[w];  // same order in every thread
    return total;
}

// Eight neighbouring bfloat16 channels of a head, rotated: (u, p) -> u cos - p sin for a pair's first channel, u cos + p sin for
// its second.  Pairs are neighbours (`other` unused; cs, sn: four angles) or, `apart`, half the rotated channels apart (`other`: the
// partners' eight; eight angles; `lower`: the first channels).  The angles come in whole pieces: one by one, each was waited for.
__device__ __forceinline__ uint4 turned_piece(uint4 own, uint4 other, bool apart, bool lower, const float* cs, const float* sn) {
    const float4 c0 = *reinterpret_cast<const float4*>(cs), c1 = *reinterpret_cast<const float4*>(cs + (apart ? 4 : 0));
    const float4 s0 = *reinterpret_cast<const float4*>(sn), s1 = *reinterpret_cast<const float4*>(sn + (apart ? 4 : 0));
    const uint32_t u[4] = {own.x, own.y, own.z, own.w}, o[4] = {other.x, other.y, other.z, other.w};
    const float c[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w}, s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    uint32_t to[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float a = __uint_as_float(u[j] << 16), b = __uint_as_float(u[j] & 0xffff0000u);
        const float pa = apart ? __uint_as_float(o[j] << 16) : b, pb = apart ? __uint_as_float(o[j] & 0xffff0000u) : a;
        const float ca = apart ? c[2 * j] : c[j], cb = apart ? c[2 * j + 1] : c[j], sa = apart ? s[2 * j] : s[j], sb = apart ? s[2 * j + 1] : s[j];
        const float qa = !apart || lower ? -pa : pa, qb = apart && lower ? -pb : pb;
        to[j] = static_cast<uint32_t>(f32_to_bf16(a * ca + qa * sa)) | (static_cast<uint32_t>(f32_to_bf16(b * cb + qb * sb)) << 16);
    }
    return make_uint4(to[0], to[1], to[2], to[3]);
}

// Dispatch a two-way storage tag to a template argument.
#define PULSE_DISPATCH_DTYPE(tag, T, ...)                 \
    do {                                                  \
        if ((tag) == PULSE_F32) {                         \
            using T = float;                              \
            __VA_ARGS__;                                  \
        } else {                                          \
            using T = bf16_t;                             \
            __VA_ARGS__;                                  \
        }                                                 \
    } while (0)

static inline bool pulse_dtype_ok(int tag) { return tag == PULSE_F32 || tag == PULSE_BF16; }
