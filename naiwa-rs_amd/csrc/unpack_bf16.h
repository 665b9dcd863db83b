// Quantised weights as bf16 operands of the matrix cores: computed in f32 and rounded once.
#pragma once

#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Element i of a laid-out Q4_K run holds byte q4_elem(i) of the run (an involution).
__host__ __device__ constexpr int q4_elem(int i) { return (i == 1 || i == 2 || i == 5 || i == 6) ? (i ^ 3) : i; }

// Two f32 values rounded to nearest-even bf16 (v_cvt_pk_bf16_f32), as one word.
__device__ __forceinline__ uint32_t bf16x2_bits(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{a, b}, bf16x2));
}
// Eight f32 values as the bf16 MFMA operand.
__device__ __forceinline__ bf16x8 to_bf16x8(const float (&f)[8]) {
    const u32x4 w = {bf16x2_bits(f[0], f[1]), bf16x2_bits(f[2], f[3]), bf16x2_bits(f[4], f[5]),
                     bf16x2_bits(f[6], f[7])};
    return __builtin_bit_cast(bf16x8, w);
}

// (d * scale, -dmin * min) of 32-value sub-block j of a Q4_K block whose first 16
// bytes are hd (ggml's get_scale_min_k4), exact in f32 (an f16 times a 6-bit integer).
__device__ __forceinline__ void q4k_scale_min(const u32x4& hd, int j, float& sc, float& mn) {
    const uint32_t s3[3] = {hd.y, hd.z, hd.w};
    auto sb = [&](int i) -> int { return (int)((s3[i >> 2] >> (8 * (i & 3))) & 0xFFu); };
    int s, m;
    if (j < 4) {
        s = sb(j) & 63;
        m = sb(j + 4) & 63;
    } else {
        s = (sb(j + 4) & 0xF) | ((sb(j - 4) >> 6) << 4);
        m = (sb(j + 4) >> 4) | ((sb(j) >> 6) << 4);
    }
    sc = naiwa_f16_to_f32(hd.x & 0xffffu) * (float)s;
    mn = -(naiwa_f16_to_f32(hd.x >> 16) * (float)m);
}

// Nibble masks held in registers.  A nibble masked into the mantissa of an f16 magic
// number reads as magic + q exactly: a low nibble (bits 0-3) in 1024.0 (0x6400), a
// high one left at bits 4-7 in 64.0 (0x5400).  With the mask in a VGPR,
// (w & mask) | magic is one v_and_or_b32 (a VOP3 here takes at most one literal or
// SGPR, so two immediates would cost a separate and and or).
struct NibMask {
    uint32_t m[2]; // low nibbles 0x000F000F, high nibbles 0x00F000F0
};
__device__ __forceinline__ NibMask nib_mask() {
    NibMask n{{0x000F000Fu, 0x00F000F0u}};
    asm("" : "+v"(n.m[0]));
    asm("" : "+v"(n.m[1]));
    return n;
}

// The 8 weights q * sc + mn of quant words da, db (bytes 0-7 of a run), the low
// nibbles when hi = 0 and the high ones when hi = 1, in byte order 0 2 1 3 4 6 5 7,
// rounded once to bf16.  Each pair of nibbles becomes two f16 magic + q (one
// v_and_or_b32), and each weight one v_fma_mix_f32: (magic + q) * sc + (mn - magic
// * sc) in f32.  The folded offset is rounded once in f32 (an error below 2^-14 sc,
// far under the bf16 rounding of the weight).
__device__ __forceinline__ bf16x8 q4k_unpack(uint32_t da, uint32_t db, int hi, const NibMask& nm, float sc,
                                             float mn) {
    const uint32_t mk = nm.m[hi], magic = hi ? 0x54005400u : 0x64006400u;
    const float m2 = __builtin_fmaf(hi ? -64.0f : -1024.0f, sc, mn);
    const uint32_t p[4] = {(da & mk) | magic, ((da >> 8) & mk) | magic, (db & mk) | magic,
                           ((db >> 8) & mk) | magic};
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const half2v v = __builtin_bit_cast(half2v, p[i]);
        f[2 * i] = __builtin_fmaf((float)v[0], sc, m2);
        f[2 * i + 1] = __builtin_fmaf((float)v[1], sc, m2);
    }
    return to_bf16x8(f);
}

// The 8 weights d * q of the signed bytes of words d0, d1 (values in order): the
// product is exact in f32 and rounded once to bf16.
__device__ __forceinline__ bf16x8 q8_unpack(uint32_t d0, uint32_t d1, float d) {
    float f[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[k] = (float)(int8_t)(d0 >> (8 * k)) * d;
        f[4 + k] = (float)(int8_t)(d1 >> (8 * k)) * d;
    }
    return to_bf16x8(f);
}

} // namespace
