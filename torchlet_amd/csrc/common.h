// Shared device helpers of the torchlet_amd kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// ---------------------------------------------------------------- element types
// bfloat16 is carried as its 16 raw bits; every kernel widens to float on load and
// rounds to nearest-even on store.
struct bf16_t { uint16_t bits; };

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }

template <typename T> __device__ __forceinline__ T from_float(float v);
template <> __device__ __forceinline__ float from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_float<bf16_t>(float v) {
    // gfx950 converts in hardware (v_cvt_pk_bf16_f32): round to nearest, ties to even, NaN kept
    const __bf16 h = (__bf16)v;
    bf16_t r;
    __builtin_memcpy(&r.bits, &h, sizeof(r.bits));
    return r;
}

// A vector (norm weight, bias) is stored either as bfloat16 or as float; read element i.
__device__ __forceinline__ float load_vec(const void* p, int is_f32, size_t i) {
    return is_f32 ? ((const float*)p)[i] : to_float(((const bf16_t*)p)[i]);
}

// Four neighbouring numbers (16-byte aligned floats, 8-byte aligned bfloat16).
__device__ __forceinline__ float4 load4(const float* p) { return *(const float4*)p; }
__device__ __forceinline__ float4 load4(const bf16_t* p) {
    const uint2 t = *(const uint2*)p;
    return make_float4(__uint_as_float(t.x << 16), __uint_as_float(t.x & 0xffff0000u), __uint_as_float(t.y << 16), __uint_as_float(t.y & 0xffff0000u));
}
__device__ __forceinline__ void store4(float* p, float4 v) { *(float4*)p = v; }
__device__ __forceinline__ void store4(bf16_t* p, float4 v) {
    uint2 t;
    t.x = (uint32_t)from_float<bf16_t>(v.x).bits | ((uint32_t)from_float<bf16_t>(v.y).bits << 16);
    t.y = (uint32_t)from_float<bf16_t>(v.z).bits | ((uint32_t)from_float<bf16_t>(v.w).bits << 16);
    *(uint2*)p = t;
}

// Four: four neighbouring numbers as they are stored, widened where they are used (half the registers of a piece on its way).
template <typename T> struct Four;
template <> struct Four<float> { typedef float4 type; };
template <> struct Four<bf16_t> { typedef ushort4 type; };
__device__ __forceinline__ float4 widen4(float4 v) { return v; }
__device__ __forceinline__ float4 widen4(ushort4 v) {
    return make_float4(to_float(bf16_t{v.x}), to_float(bf16_t{v.y}), to_float(bf16_t{v.z}), to_float(bf16_t{v.w}));
}

// ---------------------------------------------------------------- reductions
#define TL_WAVE 64

// A lane's value and that of lane ^ 32 (lane ^ 16), joined: the halves (the rows of 16 lanes) change places in the vector unit, where a shuffle would go through shared
// memory and the step would wait for the trip.  All lanes of the wave take part.
__device__ __forceinline__ float sum_across_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_across_rows(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float max_across_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_across_rows(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// The value of the lane BY places on in its row of 16, in a circle.
template <int BY>
__device__ __forceinline__ float row_turned(float v) {
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x120 + BY, 0xF, 0xF, false));
}
// Sums over neighbouring LANES (a power of two) and maxima over the wave, the same in each of the lanes.  The sums are those of a butterfly of exchanges with lane ^ 32, ^ 16, .. ^ 1, to
// the bit: once the halves of a row hold the same sums, the lane 4 places on holds what lane ^ 4 does, and so on.  (As a butterfly of six shuffles a sum took 0.25 us longer: a
// decode step's norm of 16 rows of 2048 numbers, which takes two, 4.1 -> 3.6 us, launch included.)
template <int LANES>
__device__ __forceinline__ float lanes_sum(float v) {
    if constexpr (LANES > 32) v = sum_across_halves(v);
    if constexpr (LANES > 16) v = sum_across_rows(v);
    static_assert(LANES >= 16, "whole rows of the wave");
    v += row_turned<8>(v);
    v += row_turned<4>(v);
    v += row_turned<2>(v);
    v += row_turned<1>(v);
    return v;
}
__device__ __forceinline__ float wave_sum(float v) { return lanes_sum<TL_WAVE>(v); }
__device__ __forceinline__ float wave_max(float v) {
    v = max_across_rows(max_across_halves(v));
    v = fmaxf(v, row_turned<8>(v));
    v = fmaxf(v, row_turned<4>(v));
    v = fmaxf(v, row_turned<2>(v));
    return fmaxf(v, row_turned<1>(v));
}

__device__ __forceinline__ float sigmoid(float v) { return 1.f / (1.f + expf(-v)); }

// z / 2 (1 + tanh(y)), y = sqrt(2 / pi) (z + 0.044715 z^3), with (1 + tanh(y)) / 2 = sigmoid(2 y).
__device__ __forceinline__ float gelu_tanh(float z) { return z * sigmoid(1.5957691216057308f * fmaf(0.044715f * z * z, z, z)); }

// One pair turned by its angle, in a fixed sequence of roundings (one product, one fused
// multiply-add per result), so that every kernel here gives the same bits for the same input.
__device__ __forceinline__ void rope_turn(float& x1, float& x2, float c, float sn) {
    const float y1 = __fmaf_rn(x1, c, -__fmul_rn(x2, sn));
    const float y2 = __fmaf_rn(x2, c, __fmul_rn(x1, sn));
    x1 = y1;
    x2 = y2;
}

// Sum over a block of up to 1024 threads; every thread gets the result.
// `red` points to at least 16 floats of shared memory.
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int wave = threadIdx.x / TL_WAVE, lane = threadIdx.x % TL_WAVE;
    const int nw = (blockDim.x + TL_WAVE - 1) / TL_WAVE;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < nw; ++i) t += red[i];
    return t;
}

// ---------------------------------------------------------------- host side
// Every entry point returns 0 on success, else an error code; the text of the last
// error of the calling thread is read with tl_last_error().
#define TL_OK 0
#define TL_ERR_ARG 1
#define TL_ERR_HIP 2

#include <stdarg.h>
#include <stdio.h>

// Each shared library is one translation unit and carries its own error text.
static thread_local char tl_error_text[512];

static inline void tl_set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(tl_error_text, sizeof(tl_error_text), fmt, ap);
    va_end(ap);
}

extern "C" const char* tl_last_error() { return tl_error_text; }

#define TL_REQUIRE(cond, ...)                 \
    do {                                      \
        if (!(cond)) {                        \
            tl_set_error(__VA_ARGS__);        \
            return TL_ERR_ARG;                \
        }                                     \
    } while (0)

#define TL_CHECK_LAUNCH(name)                                                    \
    do {                                                                         \
        hipError_t e_ = hipGetLastError();                                       \
        if (e_ != hipSuccess) {                                                  \
            tl_set_error("%s: launch failed: %s", name, hipGetErrorString(e_));  \
            return TL_ERR_HIP;                                                   \
        }                                                                        \
    } while (0)

#define TL_DT_F32 0
#define TL_DT_BF16 1
