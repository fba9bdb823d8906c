// The operand formats of the floating-point path and their conversions from and to float32.
#pragma once

#include "common.hpp"

namespace a4g {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned f32_to_bf16_bits(float f) {  // round to nearest even; NaN stays NaN
    const unsigned u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_bits_to_f32(unsigned h) { return __uint_as_float(h << 16); }

// float32 -> fp8 e4m3 code, the integer recipe of the reference's packer (_float32_to_fp8_scalar,
// op_impls/families/matmul/common.py:262-276): round half away from zero at mantissa bit 20, exponent bias 7,
// gradual underflow below 2^-6, magnitudes from 480 up map to the code 0x7f.
__host__ __device__ __forceinline__ unsigned f32_bits_to_fp8(unsigned bits) {
    const unsigned h = bits + 0x00080000u;
    const unsigned e = (h & 0x7F800000u) >> 23, m = h & 0x007FFFFFu, sign = (h & 0x80000000u) >> 24;
    if (e > 135u) return sign | 0x7Fu;
    if (e > 120u) return sign | (((e - 120u) << 3) & 0x78u) | (m >> 20);
    if (e > 116u) return sign | ((((0x00780000u + m) >> (140u - e)) + 1u) >> 1);
    return sign;
}
__device__ __forceinline__ unsigned f32_to_fp8_bits(float f) { return f32_bits_to_fp8(__float_as_uint(f)) & 0xFFu; }
// fp8 e4m3 (OCP "fn": bias 7, no infinities, 0x7f / 0xff are NaN) -> float32, exact
__device__ __forceinline__ float fp8_bits_to_f32(unsigned c) {
    const unsigned sign = (c & 0x80u) << 24, e = (c >> 3) & 0xFu, m = c & 7u;
    if (e == 15u && m == 7u) return __uint_as_float(sign | 0x7FC00000u);
    if (e == 0u) return __uint_as_float(sign) + (sign ? -1.f : 1.f) * static_cast<float>(m) * 0.001953125f;  // m * 2^-9
    return __uint_as_float(sign | ((e + 120u) << 23) | (m << 20));
}

__device__ __forceinline__ float load_float(const void* p, int64_t i, int fmt) {
    if (fmt == A4G_F32) return static_cast<const float*>(p)[i];
    if (fmt == A4G_FP8) return fp8_bits_to_f32(static_cast<const uint8_t*>(p)[i]);
    return bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
}
__device__ __forceinline__ void store_float(void* p, int64_t i, int fmt, float v) {
    if (fmt == A4G_F32) static_cast<float*>(p)[i] = v;
    else if (fmt == A4G_FP8) static_cast<uint8_t*>(p)[i] = static_cast<uint8_t>(f32_to_fp8_bits(v));
    else static_cast<uint16_t*>(p)[i] = static_cast<uint16_t>(f32_to_bf16_bits(v));
}
static inline int fmt_bytes(int fmt) { return fmt == A4G_F32 ? 4 : (fmt == A4G_FP8 ? 1 : 2); }
static inline bool fmt_ok(int fmt) { return fmt == A4G_F32 || fmt == A4G_BF16 || fmt == A4G_FP8; }

}  // namespace a4g
