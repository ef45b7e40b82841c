// Shared host/device helpers for the gfx950 kernels of libfastmoe_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdarg>
#include <cstdio>

#include "../../include/fast_moe_amd.h"

namespace fmoe {

// ---------------------------------------------------------------- host side
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);

#define FMOE_REQUIRE(cond, ...)                                   \
    do {                                                          \
        if (!(cond)) return ::fmoe::fail(FMOE_ERR_ARGUMENT, __VA_ARGS__); \
    } while (0)

__host__ __device__ static inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }
__host__ __device__ static inline bool aligned16(const void* p) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}
__host__ __device__ static inline bool aligned_ok(const void* a, const void* b, const void* c) {
    return aligned16(a) && aligned16(b) && aligned16(c);
}

// -------------------------------------------------------------- device side
constexpr int kWave = 64;

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) int i32x8;

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

// round-to-nearest-even fp32 -> bf16 bit pattern; NaN stays NaN (quiet)
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float round_bf16(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }

// two fp32 -> two bf16 (round to nearest even) in one v_cvt_pk_bf16_f32, `lo` in the low half: for
// loops that round every element they touch (with the integer sequence above, which also keeps a
// NaN's payload, the rounding is most of such a loop's instructions and the loop is bound by them,
// not by the memory it streams)
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    const bf16x2_t r = __builtin_convertvector(v, bf16x2_t);
    return __builtin_bit_cast(uint32_t, r);
}
// both values rounded to bf16 and back
__device__ __forceinline__ void round_bf16_pair(float& a, float& b) {
    const uint32_t pk = cvt_pk_bf16(a, b);
    a = __uint_as_float(pk << 16);
    b = __uint_as_float(pk & 0xffff0000u);
}

__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + expf(-x)); }

// round(silu(x)) to bf16 for two bf16-valued x, equal on every one of the 65536 inputs to what
// x / (1 + exp(-x)) gives when it is evaluated in fp32 with correctly rounded steps and then rounded
// to bf16 (F.silu on a bf16 tensor).  v_exp_f32 and v_rcp_f32 give that rounding on every input with two
// corrections: at x = 5.9375 the fp32 quotient comes out on the midpoint of two bf16 values, one unit in the last
// place above the exact one, which the addend one unit above 1 takes back (it moves no other input's rounding);
// and at -87.5, -88 and -88.5 the reciprocal lies below the normal range and is flushed: x * exp(x), scaled through
// the exponent, rounds right there.  Further down exp(-x) overflows and the quotient is -0, as in the fp32 formula.
// (Library expf, a division and a double-precision second look bound the passes that call this by VALU work and by the
// size of their unrolled code: 33 M hidden elements took the SiLU quantiser 54 us, 24 M silu_mul 32 us.)
__device__ __forceinline__ void silu_round_bf16_pair(float& a, float& b) {
    constexpr float kLog2e = 1.44269504088896341f, kOnePlus = 1.00000012f;
    float ya = a * __builtin_amdgcn_rcpf(kOnePlus + __builtin_amdgcn_exp2f(a * -kLog2e));
    float yb = b * __builtin_amdgcn_rcpf(kOnePlus + __builtin_amdgcn_exp2f(b * -kLog2e));
    if (fminf(a, b) < -87.0f) {
        auto low = [](float x, float y) {
            const float scaled = x * __builtin_amdgcn_exp2f(__builtin_fmaf(x, kLog2e, 32.0f));
            return x < -87.0f && x > -88.7f ? scaled * 0x1p-32f : y;
        };
        ya = low(a, ya);
        yb = low(b, yb);
    }
    round_bf16_pair(ya, yb);
    a = ya;
    b = yb;
}
// The same for a 16-byte chunk of eight values, with one look for the low end: a branch behind every pair leaves its chain of v_exp_f32 and
// v_rcp_f32 nothing to overlap with.
__device__ __forceinline__ u32x4 silu_round_bf16_x8(u32x4 v) {
    constexpr float kLog2e = 1.44269504088896341f, kOnePlus = 1.00000012f;
    float x[8], y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        x[j] = j & 1 ? __uint_as_float(v[j / 2] & 0xffff0000u) : __uint_as_float(v[j / 2] << 16);
        y[j] = x[j] * __builtin_amdgcn_rcpf(kOnePlus + __builtin_amdgcn_exp2f(x[j] * -kLog2e));
    }
    if (fminf(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])), fminf(fminf(x[4], x[5]), fminf(x[6], x[7]))) < -87.0f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float scaled = x[j] * __builtin_amdgcn_exp2f(__builtin_fmaf(x[j], kLog2e, 32.0f));
            y[j] = x[j] < -87.0f && x[j] > -88.7f ? scaled * 0x1p-32f : y[j];
        }
    }
    return u32x4{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3]), cvt_pk_bf16(y[4], y[5]), cvt_pk_bf16(y[6], y[7])};
}
__device__ __forceinline__ float silu_round_bf16(float x) {
    float other = 0.0f;
    silu_round_bf16_pair(x, other);
    return x;
}

// SiLU from the hardware exp / reciprocal (about 2 ulp in fp32): for values that
// are rounded to bf16 right afterwards.
__device__ __forceinline__ float fast_silu_f32(float x) {
    // v_exp_f32 and v_rcp_f32 only: a true division costs ten more VALU instructions
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896341f));
}

__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

template <typename T>
__device__ __forceinline__ T wave_bcast(T v, int src_lane) {
    return __shfl(v, src_lane, kWave);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

// inclusive prefix sum over the 64 lanes
__device__ __forceinline__ int wave_inclusive_scan(int v) {
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        int n = __shfl_up(v, o, kWave);
        if (lane >= o) v += n;
    }
    return v;
}
__device__ __forceinline__ long long wave_inclusive_scan(long long v) {
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        long long n = __shfl_up(v, o, kWave);
        if (lane >= o) v += n;
    }
    return v;
}

}  // namespace fmoe
