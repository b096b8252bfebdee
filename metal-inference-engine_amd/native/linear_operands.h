// MFMA operands of the linears (linear.hip, linear_mid.hip, linear_gemm.hip). Activations enter v_mfma_f32_16x16x32_bf16
// as the exact three-piece bf16 split of their fp32 values, weights exactly (bf16 as stored, INT8 / INT4 codes as small
// integers), so every product is exact and is summed in fp32.
#pragma once

#include "rk_device.h"
#include "rk_internal.h"

namespace rk {

// linear_mid.hip: the form for up to a few hundred rows, behind rk_linear_gemm
struct MidPlan {
    int MB, MT, NT, G, S, SB, WB;  // row blocks and their tiles; weight tiles and groups of them; K-splits and their blocks
    double us;                     // the estimated time; 0: not for this form
    size_t sums, part, total;      // the workspace
};
MidPlan mid_plan(int M, int N, int K, int w_type, int glu);
bool mid_reads(const void* scales, const void* mins);   // their addresses allow it
int mid_linear(const MidPlan& p, float* y, const float* x, long long x_ld, int M, int N, int K, const void* w, int w_type,
               const void* scales, const void* mins, const float* bias, const float* residual, int glu,
               void* workspace, hipStream_t stream);

constexpr int kQB = 32;            // weights per quantization block = the MFMA k-extent

__device__ __forceinline__ float half_to_f32(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// silu(g) * u = g / (1 + exp(-g)) * u with the hardware exp2 and reciprocal: SwiGLU's product, in the one form that
// the silu * up input transform and the paired [gate; up] outputs compute, so they give equal bits.
// The result is the rounded fp32 product, as the reference hands silu * up to the next op as an fp32 tensor: the
// empty asm makes it opaque, since an inlined product would otherwise be contracted into the activation split that
// consumes it (x - hi as fma(a, u, -hi)), whose pieces would then carry the unrounded product.
__device__ __forceinline__ float silu_times(float g, float u) {
    const float d = 1.0f + __builtin_amdgcn_exp2f(-g * 1.4426950408889634f);
    float h = g * __builtin_amdgcn_rcpf(d) * u;
    asm("" : "+v"(h));
    return h;
}

// 8 INT8 codes (one lane's MFMA slots of one block: bytes of lo then hi) as bf16 bits; q in [-127, 127] is exact in
// bf16, and the top half of the fp32 value is its bf16 pattern
__device__ __forceinline__ u32x4 int8_bf16(uint32_t lo, uint32_t hi) {
    u32x4 o;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t w = h ? hi : lo;
            const float f0 = (float)(int)__builtin_amdgcn_sbfe(w, 16 * e, 8);
            const float f1 = (float)(int)__builtin_amdgcn_sbfe(w, 16 * e + 8, 8);
            o[2 * h + e] = pack_hi2(__float_as_uint(f0), __float_as_uint(f1));
        }
    return o;
}

// 8 INT4 codes (4 bytes; byte j holds elements 2j in the low nibble, 2j+1 in the high one) as bf16 bits, in the
// element order 0 2 4 6 1 3 5 7 (kInt4Order; the activations are staged in the same order, so the MFMA's k-sum
// is unchanged). A code q alone in a byte, read as an fp8 e4m3 pattern 0000qqqq, is exactly q * 2^-9 (codes 0-7
// are subnormals m * 2^-9, 8-15 the first normal binade (8 + m) * 2^-9), so v_cvt_scalef32_pk_bf16_fp8 with the
// scale 2^9 turns two such bytes into two exact bf16 integers: 7 instructions for 8 codes.
__device__ __forceinline__ u32x4 int4_bf16(uint32_t v) {
    const uint32_t lo = v & 0x0F0F0F0Fu, hi = (v >> 4) & 0x0F0F0F0Fu;   // codes 0 2 4 6 | 1 3 5 7, one per byte
    u32x4 o;
    o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
    o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
    o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
    o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
    return o;
}
// element pairs of the four bf16-pair registers of an INT4 operand (int4_bf16), and of the activation pieces staged
// against it
constexpr int kInt4Order[4][2] = {{0, 2}, {4, 6}, {1, 3}, {5, 7}};

// The same of code - 8 (as signed bytes of the e4m3 pattern: 0 .. 7 as they are, -8 .. -1 from a table), for the linears
// that take an INT4 weight as s (q - 8) + (8 s + min)
__device__ __forceinline__ uint32_t int4_centred(uint32_t t) {   // codes, one per byte
    const uint32_t x = t & 0x08080808u, m = (x << 5) - (x >> 3), low = t & 0x07070707u;   // m: 0xff for codes 8 .. 15
    return (low & m) | (__builtin_amdgcn_perm(0x81828384u, 0x85868788u, low) & ~m);
}
__device__ __forceinline__ u32x4 int4_bf16_centred(uint32_t v) {
    const uint32_t lo = int4_centred(v & 0x0F0F0F0Fu), hi = int4_centred((v >> 4) & 0x0F0F0F0Fu);
    u32x4 o;
    o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
    o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
    o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
    o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
    return o;
}

// split3 where a value may be infinite: an infinity has no rest (inf - inf would make it NaN)
__device__ __forceinline__ Split3 split3_any(float x) {
    Split3 s = split3(x);
    if (__builtin_isinf(x)) s.mid = s.lo = 0u;
    return s;
}

// 4 x 4 transpose over the wave's four 16-lane groups: afterwards register d of lane group g holds what register g
// of lane group d held. v_permlane32_swap exchanges the upper 32 lanes of its first operand with the lower 32 of its
// second, v_permlane16_swap the odd 16-lane groups of the first with the even ones of the second; all 64 lanes must
// be active.
__device__ __forceinline__ u32x4 xpose4(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
    const auto s02 = __builtin_amdgcn_permlane32_swap(a0, a2, false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(a1, a3, false, false);
    const auto s01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    const auto s23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    return (u32x4){s01[0], s01[1], s23[0], s23[1]};
}

}  // namespace rk
