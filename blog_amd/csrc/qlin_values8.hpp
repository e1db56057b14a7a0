// qlin_values8.hpp -- eight consecutive weights of a packed row at a time: the raw bytes, then their
// canonical values (gfx950 device code).
//
// Elements k0 .. k0+7 (k0 a multiple of 8) lie in one block and under one scale in every format.  The
// raw words are read first, so that a wave can have several pieces' loads in flight; blocks are only
// 2-byte aligned, so the pieces are read as wide loads off their natural alignment (which the hardware
// takes) rather than as 16-bit loads.  Values are those of the per-element decoders
// (kernel.cu:1122-1185, ggml's Q4_0), bit for bit.
#pragma once

#include "qlin_device.hpp"

namespace qlin {

// dwords at a 2-byte aligned address
__device__ __forceinline__ uint32_t ld4_a2(const uint8_t *p) {
    uint32_t v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 4);
    return v;
}
__device__ __forceinline__ uint2 ld8_a2(const uint8_t *p) {
    uint2 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 8);
    return v;
}
__device__ __forceinline__ u32x4 ld16_a2(const uint8_t *p) {
    u32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 16);
    return v;
}

__device__ __forceinline__ uint32_t byte_of(uint2 v, int i) { return ((i < 4 ? v.x : v.y) >> (8 * (i & 3))) & 0xffu; }

// q: the 8 quant bytes; a: d (low half; Q6_K: the scale byte above it); b: Q5_0's qh, Q6_K's qh bytes;
// hdr: Q4_K's d, dmin and scale bytes.
template <int T>
struct Raw8 {
    uint2 q;
    uint32_t a;
    uint2 b;
};
template <>
struct Raw8<T_Q4_K> {
    uint2 q;
    u32x4 hdr;
};

template <int T>
__device__ __forceinline__ void raw8(const uint8_t *row, int k0, Raw8<T> &r) {
    if constexpr (T == T_Q4_K) {
        const uint8_t *b = row + static_cast<size_t>(k0 >> 8) * 144;
        const int e = k0 & 255;
        r.hdr = ld16_a2(b);
        r.q = ld8_a2(b + 16 + (e >> 6) * 32 + (e & 31));
    } else if constexpr (T == T_Q6_K) {  // half, group of 32, elements l0 .. l0+7 (one 16-element scale)
        const uint8_t *b = row + static_cast<size_t>(k0 >> 8) * 210;
        const int e = k0 & 255, half = e >> 7, grp = (e & 127) >> 5, l0 = e & 31;
        r.q = ld8_a2(b + half * 64 + l0 + 32 * (grp & 1));
        r.b = ld8_a2(b + 128 + half * 32 + l0);
        r.a = ld_u16(b + 208) | (static_cast<uint32_t>(b[192 + half * 8 + l0 / 16 + 2 * grp]) << 16);
    } else if constexpr (T == T_Q8_0) {
        const uint8_t *b = row + static_cast<size_t>(k0 >> 5) * 34;
        r.a = ld_u16(b);
        r.q = ld8_a2(b + 2 + (k0 & 31));
    } else {
        constexpr int BB = T == T_Q4_0 ? 18 : 22, QS = T == T_Q4_0 ? 2 : 6;
        const uint8_t *b = row + static_cast<size_t>(k0 >> 5) * BB;
        r.a = ld_u16(b);
        r.q = ld8_a2(b + QS + (k0 & 15));
        if constexpr (T == T_Q5_0) r.b.x = ld4_a2(b + 2);
    }
}

template <int T>
__device__ __forceinline__ void values8(const Raw8<T> &r, int k0, float (&v)[8]) {
    if constexpr (T == T_Q4_K) {
        const int j = (k0 & 255) >> 5;
        int sc, m;
        q4k_scale_min(j, r.hdr.y, r.hdr.z, r.hdr.w, sc, m);
        const float dsc = mul_rn(f16_bits_to_f32(r.hdr.x & 0xffffu), static_cast<float>(sc));
        const float dm = mul_rn(f16_bits_to_f32(r.hdr.x >> 16), static_cast<float>(m));
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = sub_rn(mul_rn(dsc, static_cast<float>((byte_of(r.q, i) >> (4 * (j & 1))) & 15u)), dm);
    } else if constexpr (T == T_Q6_K) {
        const int grp = (k0 & 127) >> 5;
        const int sc = static_cast<int8_t>(r.a >> 16);
        const float dsc = mul_rn(f16_bits_to_f32(r.a & 0xffffu), static_cast<float>(sc));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t lb = byte_of(r.q, i), hb = byte_of(r.b, i);
            const int q = static_cast<int>(((grp < 2 ? lb : lb >> 4) & 15u) | (((hb >> (2 * grp)) & 3u) << 4)) - 32;
            v[i] = mul_rn(dsc, static_cast<float>(q));
        }
    } else if constexpr (T == T_Q8_0) {
        const float d = f16_bits_to_f32(r.a);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = mul_rn(d, static_cast<float>(static_cast<int8_t>(byte_of(r.q, i))));
    } else {
        const int e0 = k0 & 31, sh = e0 >= 16 ? 4 : 0;
        const float d = f16_bits_to_f32(r.a);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int q = static_cast<int>((byte_of(r.q, i) >> sh) & 15u);
            if constexpr (T == T_Q5_0) q |= static_cast<int>(((r.b.x >> (e0 + i)) & 1u) << 4);
            v[i] = mul_rn(d, static_cast<float>(q - (T == T_Q4_0 ? 8 : 16)));
        }
    }
}

}  // namespace qlin
