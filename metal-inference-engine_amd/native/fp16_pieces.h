// fp16 pieces of fp32 values, for the fp32 prefill attention (paged_prefill.hip).
#pragma once

#include "rk_device.h"
#include "rk_internal.h"

namespace rk {

constexpr int kTop = 14;                           // a row's largest value lies in [2^kTop, 2^(kTop + 1))

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// the power of two that puts the magnitude m into [2^kTop, 2^(kTop + 1)): its exponent (0 for m = 0; inf and NaN as
// the largest finite exponent, so that they stay inf and NaN in the pieces)
__device__ __forceinline__ int top_exponent(float m) {
    const int e = (int)(__float_as_uint(m) >> 23) - 127;
    return m == 0.0f ? 0 : kTop - max(min(e, 127), -112);
}

// hi and lo pieces of a pair (already scaled), packed: hi = fp16(v), lo = fp16((v - hi) up). up = 2^kUp, where lo's
// products have sums of their own, keeps its bits 2^kUp further down
constexpr int kUp = 12;
struct Pieces {
    uint32_t hi, lo;
};
__device__ __forceinline__ Pieces split_pair(float a, float b, float up = 1.0f) {
    const f16x2 h = __builtin_convertvector((f32x2_t){a, b}, f16x2);
    const f16x2 l = __builtin_convertvector((f32x2_t){(a - (float)h[0]) * up, (b - (float)h[1]) * up}, f16x2);
    return {__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l)};
}
// Where a value was infinite: it is all in lo, which meets only the other operand's hi, whose sign is the value's (hi times
// the other's lo, of either sign or 0, would make it NaN).
__device__ __forceinline__ Pieces infinite_in_lo(Pieces p) {
    const uint32_t m = p.hi & 0x7fff7fffu;           // exponent 31 with mantissa 0
    const uint32_t inf = ((m & 0xffffu) == 0x7c00u ? 0xffffu : 0u) | (m >> 16 == 0x7c00u ? 0xffff0000u : 0u);
    return {p.hi & ~inf, (p.lo & ~inf) | (p.hi & inf)};
}

// Rows of 32 fp16 (64 bytes) in LDS: the 16-byte unit u of row R sits at u ^ swizzle(R). A read of lane l: row l % 16,
// unit l / 16, is served 16 lanes at a time, rows 0-3 and 12-15 of one unit with rows 4-11 of the next, and these then
// lie on all 16 units of the 256-byte bank line.
__device__ __forceinline__ int swizzle(int R) { return (0x78 >> (2 * ((R >> 2) & 3))) & 3; }

}  // namespace rk
