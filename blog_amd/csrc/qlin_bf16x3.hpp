// qlin_bf16x3.hpp -- f32 activations times small-integer weights on the bf16 matrix cores, with nothing of
// the operands lost (gfx950 device code).
//
// x = hi + mid + lo, each the leading 8 significant bits of what is left (truncated), holds the 24 bits of an
// f32 exactly, whatever the other values of the token are: bf16 has f32's exponents, so there is no scale.
// Weights enter as integers of at most 8 bits, exact in bf16; the three products of a pair are exact and
// v_mfma adds them in f32; the block's scale comes by one fma per sum.  hi's products go first, or to a sum of their
// own: what an MFMA's C has below the products' last place is cut off towards minus infinity, so with the small
// parts' sum as hi's C every output was low by 3e-8 to 8e-8 of the mean magnitude (hi first: 1e-9 to 8e-9; apart: 2e-10).
//
// What does not fit: sums of integers times |x| >= 2^100 could overflow before the scale, parts of values
// below 2^-100 leave bf16's range, and an infinite x has no parts.  Those (out_of_range over the values one
// lane supplies), and weights whose scale is not finite, are multiplied as f32 values d q on
// v_mfma_f32_16x16x4_f32 instead, a uniform and rare branch.  A value below 2^-110 among larger ones of its
// lane keeps what lies above 2^-126.
//
// (An fp16 pair under a power-of-two scale per token took two products instead of three, but rounded what is
// far below the token's largest value: 1e-6 next to 1e6 was lost where the weight at the latter is 0.)
#pragma once

#include "qlin_device.hpp"
#include "qlin_mfma.hpp"

namespace qlin {

// the bf16 pair of two f32 values' upper halves
__device__ __forceinline__ uint32_t bf16_tops(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}
// the three parts of two values, as bf16 pairs
__device__ __forceinline__ void split3(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    hi = bf16_tops(a, b);
    const float a1 = a - bf16_hi_val(__builtin_bit_cast(uint32_t, a)), b1 = b - bf16_hi_val(__builtin_bit_cast(uint32_t, b));
    mid = bf16_tops(a1, b1);
    const float a2 = a1 - bf16_hi_val(__builtin_bit_cast(uint32_t, a1)), b2 = b1 - bf16_hi_val(__builtin_bit_cast(uint32_t, b1));
    lo = bf16_tops(a2, b2);
}
// ... of 8 values: a lane's operands of v_mfma_f32_16x16x32_bf16
__device__ __forceinline__ void split3(const f32x4 &a, const f32x4 &b, u32x4 &hi, u32x4 &mid, u32x4 &lo) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f32x4 &v = i < 2 ? a : b;
        uint32_t h, m, l;
        split3(v[2 * (i & 1)], v[2 * (i & 1) + 1], h, m, l);
        hi[i] = h;
        mid[i] = m;
        lo[i] = l;
    }
}

// max(|a|, |b|, c) in one instruction
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// whether values of largest magnitude am (NaNs aside, which the parts carry) go as f32
__device__ __forceinline__ bool out_of_range(float am) { return !(am < 0x1p100f) || (am < 0x1p-100f && am > 0.0f); }

// the bf16 values of the 8 bytes a, b: signed, or unsigned less off
__device__ __forceinline__ u32x4 bf16_of_i8(uint32_t a, uint32_t b) {
    asm("" : "+v"(a), "+v"(b));  // (a loop that loads them ahead carries dwords, not a byte per register)
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = i < 2 ? a : b;
        r[i] = bf16_tops(static_cast<float>(static_cast<int8_t>(v >> (16 * (i & 1)))),
                         static_cast<float>(static_cast<int8_t>(v >> (16 * (i & 1) + 8))));
    }
    return r;
}
// byte I of v as a float in one instruction (a compiler's choice is a shift, a mask and a conversion)
template <int I>
__device__ __forceinline__ float f32_of_byte(uint32_t v) {
    float f;
    if constexpr (I == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(v));
    else if constexpr (I == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(v));
    else if constexpr (I == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(v));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(v));
    return f;
}
__device__ __forceinline__ u32x4 bf16_of_u8(uint32_t a, uint32_t b, float off) {
    return u32x4{bf16_tops(f32_of_byte<0>(a) - off, f32_of_byte<1>(a) - off),
                 bf16_tops(f32_of_byte<2>(a) - off, f32_of_byte<3>(a) - off),
                 bf16_tops(f32_of_byte<0>(b) - off, f32_of_byte<1>(b) - off),
                 bf16_tops(f32_of_byte<2>(b) - off, f32_of_byte<3>(b) - off)};
}
// value i of packed bf16 values
template <class V>
__device__ __forceinline__ float bf16_at(const V &v, int i) {
    return i & 1 ? bf16_hi_val(v[i >> 1]) : bf16_val(v[i >> 1] & 0xffffu);
}

// bits 0..3 of b to bit 4 of bytes 0..3
__device__ __forceinline__ uint32_t bit4_of_bytes(uint32_t b) { return spread4(b) << 4; }

}  // namespace qlin
