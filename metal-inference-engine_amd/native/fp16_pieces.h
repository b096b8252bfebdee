// fp16 pieces of fp32 values: shared by the linears of many rows (linear_gemm.hip, linear_mid.hip) and the fp32
// prefill attention (paged_prefill.hip).
#pragma once

#include "rk_device.h"
#include "rk_internal.h"

namespace rk {

// linear_mid.hip: the form for up to a few hundred rows, behind rk_linear_gemm
bool mid_takes(int M, int K, int w_type, const void* scales, const void* mins);
size_t mid_workspace_bytes(int M, int N, int K, int w_type, int glu);
int mid_linear(float* y, const float* x, long long x_ld, int M, int N, int K, const void* w, int w_type,
               const void* scales, const void* mins, const float* bias, const float* residual, int glu,
               void* workspace, hipStream_t stream);

constexpr int kQB = 32;                            // weights per quantization block = one MFMA's k-extent
constexpr int kTop = 14;                           // a row's largest value lies in [2^kTop, 2^(kTop + 1))

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

__device__ __forceinline__ uint32_t pack_f16(float a, float b) {   // round to nearest even
    return __builtin_bit_cast(uint32_t, (f16x2){(_Float16)a, (_Float16)b});
}

__device__ __forceinline__ float half_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// the power of two that puts the magnitude m into [2^kTop, 2^(kTop + 1)): its exponent (0 for m = 0; inf and NaN as
// the largest finite exponent, so that they stay inf and NaN in the pieces)
__device__ __forceinline__ int top_exponent(float m) {
    const int e = (int)(__float_as_uint(m) >> 23) - 127;
    return m == 0.0f ? 0 : kTop - max(min(e, 127), -112);
}

// hi and lo pieces of a pair (already scaled), packed: hi = fp16(v), lo = fp16(v - hi)
struct Pieces {
    uint32_t hi, lo;
};
__device__ __forceinline__ Pieces split_pair(float a, float b) {
    const f16x2 h = __builtin_convertvector((f32x2_t){a, b}, f16x2);
    const f16x2 l = __builtin_convertvector((f32x2_t){a - (float)h[0], b - (float)h[1]}, f16x2);
    return {__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l)};
}
// the same where a value may be infinite: an infinite hi has no rest (inf - inf would make it NaN)
__device__ __forceinline__ uint32_t rest_of(Pieces p) {
    const uint32_t e = p.hi & 0x7c007c00u, m = p.hi & 0x03ff03ffu;   // exponent 31 with mantissa 0
    const uint32_t drop = ((e & 0xffffu) == 0x7c00u && !(m & 0xffffu) ? 0xffffu : 0u) |
                          (e >> 16 == 0x7c00u && !(m >> 16) ? 0xffff0000u : 0u);
    return p.lo & ~drop;
}

// largest |v| of a 256-thread workgroup, in every thread
__device__ __forceinline__ float block_absmax(float m, float* red) {
    m = row16_max(m);
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    m = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    m = fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__device__ __forceinline__ float silu_times(float g, float u) {
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * kLog2e)) * u;
}


// Rows of 32 fp16 (64 bytes) in LDS: the 16-byte unit u of row R sits at u ^ swizzle(R). A read of lane l: row l % 16,
// unit l / 16, is served 16 lanes at a time, rows 0-3 and 12-15 of one unit with rows 4-11 of the next, and these then
// lie on all 16 units of the 256-byte bank line.
__device__ __forceinline__ int swizzle(int R) { return (0x78 >> (2 * ((R >> 2) & 3))) & 3; }

}  // namespace rk
