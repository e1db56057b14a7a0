// qlin_gemm.hip -- the prefill GEMM of the 32-block formats: Q8_0, Q5_0 and Q4_0 weights times many rows of
// activations, f32 or Q8_1, on the fp16 matrix cores of gfx950.
//
//   y[r, o] (=|+=) sum_k w(o, k) x[r, k]                          (kernel.cu:1254-1279, quant_matmul_kernel)
//   y[r, o]  =     sum over 32-blocks of the Q8_1 block dots      (kernel.cu:2305-2402, quant_matmul_q8_1)
//   act[r, o] = g / (1 + expf(-g)) * u, g, u the rows of two matrices (SharedExperts.cpp:34-40)
//
// Operands (v_mfma_f32_16x16x32_f16: products exact, f32 accumulation).
//   A (activations): a token's values times a power of two 2^s, split into hi = fp16(x 2^s) and
//     lo = fp16(x 2^s - hi), which together hold x 2^s to 2^-22 of its value down to 2^-16 of the
//     token's largest; two MFMAs into one accumulator.  s comes from the token's largest magnitude so
//     far (in [2^12, 2^13) after scaling), and only a value 4 times that or more changes it: then that
//     token's sums are rescaled, exactly, before the step that brought it.  The result takes 2^-s at the
//     end.  A Q8_1 activation is the value d8 q, its fp16 pair formed the same way (128 d8 bounds it).
//   B (weights): q less its offset, an integer exact in fp16; the block's d by one fma per output.
//
// Tiling.  A workgroup of 8 waves computes BM tokens x BN weight rows in steps of 64 values of K.  Both
// operands of a step are staged in LDS once per workgroup -- each weight decoded once for all BM
// tokens, each activation split once for all BN rows -- in the MFMA lane layout, two buffers.  The
// waves form a WM x WN grid, each MT x NT tiles of 16 x 16.  Between two barriers waves 0-3 (one per
// SIMD) multiply step k and then stage their share of step k + 1, while waves 4-7 stage theirs of
// step k + 1 and then multiply step k, so that one half's matrix instructions run beside the other's
// vector ones.  Global loads are one step ahead (activations, from L2) and two (weights).
//
// Slots of the LDS planes are permuted within a row group by an XOR with the k-group (A) or the chunk
// (B), so that the staging writes and the fragment reads both spread over the banks.
//
// Measured (f32 activations): Q8_0 [14336, 4096] at 512 tokens 1738 -> 177 us (340 TFLOP/s) and Q4_0
// [18944, 3584] at 203 tokens 618 -> 133 us against the f32 matrix cores with the weights decoded per 16
// tokens; Q8_1 activations, Q8_0 [14336, 4096] at 512 tokens 315 -> 165 us against the 64-token tiles
// that scale every block's products twice.  Matrix cores, vector ALU and LDS are each busy 35-45% of
// the time: what bounds it is the step's chain (barrier, fragment reads, products, staging writes).
//
// Blocks and rows are only 2-byte aligned in general; weights are read as wide loads at that alignment.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_values8.hpp"

#include <type_traits>

namespace qlin {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum : int { kStore = 0, kAdd = 1, kSwiGLU = 2 };

constexpr int kWaves = 8, kThreads = kWaves * 64, kStep = 64;

template <int MT_, int NT_, int WM_, int WN_>
struct Geo {
    static constexpr int MT = MT_, NT = NT_, WM = WM_, WN = WN_;
    static constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN;
    static constexpr int waves = MT * NT > 8 ? 2 : 4;  // per SIMD: two workgroups on a CU where LDS has room for them
    static_assert(WM * WN == kWaves, "8 waves");
};

// LDS, in uint4: two step buffers (hi and lo planes, weights, block scales, rescale factors), then the
// tokens' final scales and the steps that rescale.
template <class G>
struct Lds {
    static constexpr int a = G::BM / 16 * 2 * 64, b = G::BN / 16 * 2 * 64;
    static constexpr int hi = 0, lo = a, w = 2 * a, dw = w + b, fac = dw + 2 * G::BN / 4;
    static constexpr int buf = fac + G::BM / 4;
    static constexpr int inv = 2 * buf, flag = inv + G::BM / 4, total = flag + 1;
    static constexpr size_t bytes = total * sizeof(uint4);
    static_assert(bytes <= 160 * 1024, "fits the CU's LDS");
};

struct GemmArgs {
    const uint8_t *w0, *w1;  // w1: the up matrix of kSwiGLU
    size_t rb;
    const void *x;           // f32 rows of k values, or Q8_1 rows of k / 32 blocks
    float *y;
    int n, m, k;
};

__device__ __forceinline__ f32x4 mfma(const uint4 &a, const uint4 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t h2u(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f16x2 u2h(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ f16x2 splat(float v) {
    const _Float16 h = static_cast<_Float16>(v);
    return f16x2{h, h};
}
// bytes (b0, 0x64, b1, 0x64) or (b2, .., b3, ..) of v: the fp16 pair 1024 + byte
__device__ __forceinline__ f16x2 bytes_lo(uint32_t v) { return u2h(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)); }
__device__ __forceinline__ f16x2 bytes_hi(uint32_t v) { return u2h(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)); }

// Consumes a row of sums: pure arithmetic is otherwise sunk below the next products, whose results then
// all stay live.
template <int NT>
__device__ __forceinline__ void pin(f32x4 (&v)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(v[t]));
}

// ---- activations ---------------------------------------------------------------------------------

// hi and lo parts of 8 values times sc (a power of two), or of 8 fp16 integers times sc: two
// mixed-precision fmas a value
template <class V>
__device__ __forceinline__ void split8(const V (&v)[8], float sc, uint4 &hi, uint4 &lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = static_cast<float>(v[2 * i]), b = static_cast<float>(v[2 * i + 1]);
        h[i] = h2u(f16x2{static_cast<_Float16>(fmaf(a, sc, 0.0f)), static_cast<_Float16>(fmaf(b, sc, 0.0f))});
        asm("" : "+v"(h[i]));  // one packed value (its halves would otherwise be formed twice)
        const f16x2 hp = u2h(h[i]);
        l[i] = h2u(f16x2{static_cast<_Float16>(fmaf(a, sc, -static_cast<float>(hp[0]))),
                         static_cast<_Float16>(fmaf(b, sc, -static_cast<float>(hp[1])))});
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// an infinite value has no lo part
__device__ __forceinline__ uint32_t finite_lo(uint32_t h, uint32_t l) {
    l = (h & 0x7fffu) == 0x7c00u ? l & 0xffff0000u : l;
    return (h & 0x7fff0000u) == 0x7c000000u ? l & 0x0000ffffu : l;
}
__device__ __forceinline__ void drop_inf(const uint4 &h, uint4 &l) {
    l = make_uint4(finite_lo(h.x, l.x), finite_lo(h.y, l.y), finite_lo(h.z, l.z), finite_lo(h.w, l.w));
}

// the largest of v over 8 lanes in a row (v >= 0, whose bits order as it does)
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_bits(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float max_of_8(float v) {
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    b = max(b, dpp_bits<0xb1>(b));
    b = max(b, dpp_bits<0x4e>(b));
    b = max(b, dpp_bits<0x141>(b));
    return __builtin_bit_cast(float, b);
}
// A token's scale 2^s, held as the magnitude 2^(15 - s) from which it has to change (0: no value yet).
struct Scale {
    float limit = 0.0f;
    // 2^s: the exponents of limit and 2^s add up to 15 (for no value yet some finite number, against zeros)
    __device__ __forceinline__ float sc() const {
        return __builtin_bit_cast(float, (269u << 23) - __builtin_bit_cast(uint32_t, limit));
    }
    // the factor by which the token's sums so far change for a step whose largest magnitude is am
    __device__ __forceinline__ float step(float am) {
        if (!(am > limit)) return 1.0f;
        if (!(am <= 3.4e38f)) {  // not finite: the result will not be either
            if (limit == 0.0f) limit = 32768.0f;
            return 1.0f;
        }
        int ex;
        (void)frexpf(am, &ex);
        const float was = limit;
        limit = ldexpf(1.0f, 15 - min(13 - ex, 120));
        return was > 0.0f ? was / limit : 1.0f;
    }
};
// max(|a|, |b|, c) in one instruction
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// ---- weights -------------------------------------------------------------------------------------

// The bytes of the 32-block at p, which a staging thread decodes.
template <int FMT> struct WRaw;
template <> struct WRaw<T_Q8_0> {
    static constexpr int bytes = 34;
    u32x4 q[2];
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *p) {
        d = ld_u16(p);
        q[0] = ld16_a2(p + 2);
        q[1] = ld16_a2(p + 18);
    }
};
template <> struct WRaw<T_Q5_0> {
    static constexpr int bytes = 22;
    u32x4 q;
    uint32_t d, qh;
    __device__ __forceinline__ void load(const uint8_t *p) {
        d = ld_u16(p);
        qh = ld4_a2(p + 2);
        q = ld16_a2(p + 6);
    }
};
template <> struct WRaw<T_Q4_0> {
    static constexpr int bytes = 18;
    u32x4 q;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *p) {
        d = ld_u16(p);
        q = ld16_a2(p + 2);
    }
};

// fp16 integers of 8 bytes less off
__device__ __forceinline__ uint4 minus8(uint32_t a, uint32_t b, f16x2 off) {
    return make_uint4(h2u(bytes_lo(a) + off), h2u(bytes_hi(a) + off), h2u(bytes_lo(b) + off), h2u(bytes_hi(b) + off));
}
// bits 0..3 of b to bit 4 of bytes 0..3
__device__ __forceinline__ uint32_t bit4_of_bytes(uint32_t b) { return (__umul24(b & 0xfu, 0x204081u) & 0x01010101u) << 4; }

// Elements 8g .. 8g+7 of the block for g = 0..3 through put(g, values).
template <int FMT, class Put>
__device__ __forceinline__ void decode(const WRaw<FMT> &r, Put put) {
    if constexpr (FMT == T_Q8_0) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
            put(g, minus8(r.q[g >> 1][2 * (g & 1)] ^ 0x80808080u, r.q[g >> 1][2 * (g & 1) + 1] ^ 0x80808080u, splat(-1152.0f)));
    } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // low nibbles: elements 0..15, high: 16..31
            uint32_t a = (r.q[2 * (g & 1)] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
            uint32_t b = (r.q[2 * (g & 1) + 1] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
            if constexpr (FMT == T_Q5_0) {
                a |= bit4_of_bytes(r.qh >> (8 * g));
                b |= bit4_of_bytes(r.qh >> (8 * g + 4));
            }
            put(g, minus8(a, b, splat(FMT == T_Q5_0 ? -1040.0f : -1032.0f)));
        }
    }
}

template <int FMT, bool Q81, int MODE, class G>
__global__ __launch_bounds__(kThreads, G::waves) void gemm_kernel(const GemmArgs a) {
    using L = Lds<G>;
    constexpr int MT = G::MT, NT = G::NT, BM = G::BM, BN = G::BN;
    constexpr int kOut = MODE == kSwiGLU ? BN / 2 : BN;  // output columns per workgroup
    static_assert(MODE != kSwiGLU || NT % 2 == 0, "gate and up tiles in pairs");
    extern __shared__ uint4 lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int wm = wave / G::WN, wn = wave % G::WN;
    int bx, by;
    gemm_tile((a.n + kOut - 1) / kOut, (a.m + BM - 1) / BM, bx, by);
    const int m0 = by * BM, o0 = bx * kOut;
    const int nblk = a.k / 32, nstep = (nblk + 1) / 2;
    const bool odd = nblk & 1;  // uniform: the last step has one block

    auto fbuf = [&](int at) { return reinterpret_cast<float *>(lds + at); };

    // ---- staging: activations.  Lane q of a token's 8 takes values 8q .. 8q+7 of the step.
    constexpr int XP = (BM * 8 + kThreads - 1) / kThreads;  // tokens per thread
    constexpr bool XAll = BM * 8 % kThreads == 0;
    constexpr int XB = Q81 ? 36 : 128;  // bytes of a block
    const int xq8 = tid & 7, xchunk = xq8 >> 2, xg = xq8 & 3;
    const bool xlive = XAll || tid < BM * 8;
    using XVec = std::conditional_t<Q81, uint2, float4>;
    XVec xv[XP][Q81 ? 1 : 2];
    uint32_t xds[Q81 ? XP : 1];  // a Q8_1 block's d and s
    Scale xs[XP];
    const uint8_t *xrow[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) {
        const int tok = min(m0 + p * (kThreads / 8) + (tid >> 3), a.m - 1);
        xrow[p] = static_cast<const uint8_t *>(a.x) + static_cast<size_t>(tok) * nblk * XB + XB * xchunk + (Q81 ? 0 : 32 * xg);
    }
    // loads past the last step read it again, those of a missing last block the one before it
    auto load_x = [&](int step) {
        if (!xlive) return;
        ptrdiff_t off = static_cast<ptrdiff_t>(min(step, nstep - 1)) * (2 * XB);
        if (odd && step >= nstep - 1) off -= xchunk * XB;
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            const uint8_t *b = xrow[p] + off;
            if constexpr (Q81) {
                __builtin_memcpy(&xv[p][0], __builtin_assume_aligned(b + 4 + 8 * xg, 4), 8);
                xds[p] = *reinterpret_cast<const uint32_t *>(b);
            } else {
                __builtin_memcpy(&xv[p][0], __builtin_assume_aligned(b, 4), 16);
                __builtin_memcpy(&xv[p][1], __builtin_assume_aligned(b + 16, 4), 16);
            }
        }
    };
    auto stage_x = [&](int step, uint4 *buf) {
        if (!xlive) return;
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            const int tok = p * (kThreads / 8) + (tid >> 3);
            const int at = ((tok >> 4) * 2 + xchunk) * 64 + xg * 16 + ((tok & 15) ^ (2 * xq8));
            if (odd && step == nstep - 1) {  // uniform
                asm volatile("");  // (a branch, not selects in every step)
                if (!xchunk) {
                } else if constexpr (Q81) {
                    xds[p] = 0u;
                } else {
                    xv[p][0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    xv[p][1] = xv[p][0];
                }
            }
            uint4 hi, lo;
            float am;
            if constexpr (Q81) {
                am = fabsf(f16_bits_to_f32(xds[p] & 0xffffu)) * 128.0f;
            } else {
                const float4 u = xv[p][0], v = xv[p][1];
                am = max3_abs(v.z, v.w, max3_abs(v.x, v.y, max3_abs(u.z, u.w, max3_abs(u.x, u.y, 0.0f))));
            }
            am = max_of_8(am);
            const float f = xs[p].step(am);
            const float sc = xs[p].sc();
            if constexpr (Q81) {
                const uint32_t q[2] = {xv[p][0].x ^ 0x80808080u, xv[p][0].y ^ 0x80808080u};
                const f16x2 off = splat(-1152.0f);
                const f16x2 e[4] = {bytes_lo(q[0]) + off, bytes_hi(q[0]) + off, bytes_lo(q[1]) + off, bytes_hi(q[1]) + off};
                const _Float16 v[8] = {e[0][0], e[0][1], e[1][0], e[1][1], e[2][0], e[2][1], e[3][0], e[3][1]};
                split8(v, f16_bits_to_f32(xds[p] & 0xffffu) * sc, hi, lo);
            } else {
                const float4 u = xv[p][0], v = xv[p][1];
                const float fv[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
                split8(fv, sc, hi, lo);
            }
            if (!(am <= 3.4e38f)) drop_inf(hi, lo);
            buf[L::hi + at] = hi;
            buf[L::lo + at] = lo;
            if (xq8 == 0) {
                reinterpret_cast<float *>(buf + L::fac)[tok] = f;
                if (f != 1.0f) reinterpret_cast<int *>(lds + L::flag)[step & 1] = step;
            }
        }
    };

    // ---- staging: weights.  A thread decodes one 32-block of one row per step.
    constexpr int WP = (BN * 2 + kThreads - 1) / kThreads;
    constexpr bool WAll = BN * 2 % kThreads == 0;
    constexpr int WB = WRaw<FMT>::bytes;
    const bool wlive = WAll || tid < BN * 2;
    const int whalf = tid & 1;
    WRaw<FMT> wr[2][WP];  // two steps ahead
    const uint8_t *wrow[WP];
#pragma unroll
    for (int p = 0; p < WP; ++p) {
        const int r = p * (kThreads / 2) + (tid >> 1);
        if constexpr (MODE == kSwiGLU) {
            // the rows of a wave column: NT / 2 gate tiles, then the same outputs' up tiles
            const int t = r / 16 % NT, o = o0 + (r / (16 * NT) * (NT / 2) + t % (NT / 2)) * 16 + r % 16;
            wrow[p] = (t < NT / 2 ? a.w0 : a.w1) + static_cast<size_t>(min(o, a.n - 1)) * a.rb;
        } else {
            wrow[p] = a.w0 + static_cast<size_t>(min(o0 + r, a.n - 1)) * a.rb;
        }
        wrow[p] += whalf * WB;
    }
    auto load_w = [&](WRaw<FMT> (&w)[WP], int step) {
        if (!wlive) return;
        ptrdiff_t off = static_cast<ptrdiff_t>(min(step, nstep - 1)) * (2 * WB);
        if (odd && step >= nstep - 1) off -= whalf * WB;
#pragma unroll
        for (int p = 0; p < WP; ++p) w[p].load(wrow[p] + off);
    };
    auto stage_w = [&](const WRaw<FMT> (&w)[WP], uint4 *buf) {
        if (!wlive) return;
#pragma unroll
        for (int p = 0; p < WP; ++p) {
            const int r = p * (kThreads / 2) + (tid >> 1);
            const int at = ((r >> 4) * 2 + whalf) * 64 + ((r & 15) ^ (8 * whalf));
            decode<FMT>(w[p], [&](int gg, const uint4 &v) { buf[L::w + at + 16 * gg] = v; });
            reinterpret_cast<float *>(buf + L::dw)[whalf * BN + r] = f16_bits_to_f32(w[p].d);
        }
    };
    // The next steps' loads go out behind a step's staging.  Past the last step it stages the last blocks
    // again, into a buffer that is not read any more.
    auto stage = [&](WRaw<FMT> (&w)[WP], int step) {
        uint4 *buf = lds + (step & 1) * L::buf;
        stage_w(w, buf);
        load_w(w, step + 2);
        stage_x(step, buf);
        load_x(step + 1);
    };

    // ---- products
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // One row of tiles at a time; the fragments of two rows on are read, and the row before's products
    // scaled, next to its MFMAs.
    auto multiply = [&](int step) {
        const uint4 *buf = lds + (step & 1) * L::buf;
        const int flag = reinterpret_cast<const int *>(lds + L::flag)[step & 1];
        struct Row {
            uint4 h, l;
        };
        auto load_row = [&](int c, int i) {
            const int at = ((wm * MT + i) * 2 + c) * 64 + g * 16 + (n ^ (8 * c + 2 * g));
            return Row{buf[L::hi + at], buf[L::lo + at]};
        };
        struct Cols {
            uint4 b[NT];
            float dw[NT];
        };
        auto load_cols = [&](int c) {
            Cols v;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                v.b[t] = buf[L::w + ((wn * NT + t) * 2 + c) * 64 + g * 16 + (n ^ (8 * c))];
                v.dw[t] = reinterpret_cast<const float *>(buf + L::dw)[c * BN + (wn * NT + t) * 16 + n];
            }
            return v;
        };
        Cols col = load_cols(0), col1;
        Row row[3] = {load_row(0, 0), load_row(MT > 1 ? 0 : 1, MT > 1 ? 1 : 0), Row{}};
        if (__builtin_amdgcn_readfirstlane(flag) == step) {  // uniform
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const f32x4 f = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(buf + L::fac) +
                                                                 (wm * MT + i) * 16 + 4 * g);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][t][r] *= f[r];
            }
        }
        f32x4 d[2][NT];
        float dwp[NT];  // the scales of the row before
        auto scale = [&](int i, const f32x4 (&v)[NT], const float (&dw)[NT]) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][t][r] = fmaf(dw[t], v[t][r], acc[i][t][r]);
            pin(acc[i]);
        };
#pragma unroll
        for (int u = 0; u < 2 * MT; ++u) {  // tile row u % MT of chunk u / MT
            const int i = u % MT;
            __builtin_amdgcn_sched_barrier(0);
            if (u == MT / 2) col1 = load_cols(1);
            if (u + 2 < 2 * MT) row[(u + 2) % 3] = load_row((u + 2) / MT, (u + 2) % MT);
            if (u == MT) {
#pragma unroll
                for (int t = 0; t < NT; ++t) dwp[t] = col.dw[t];
                col = col1;
            }
            const Row &x = row[u % 3];
#pragma unroll
            for (int t = 0; t < NT; ++t) d[u & 1][t] = mfma(x.h, col.b[t], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
            for (int t = 0; t < NT; ++t) d[u & 1][t] = mfma(x.l, col.b[t], d[u & 1][t]);
            if (u == MT) scale(MT - 1, d[(u - 1) & 1], dwp);
            else if (u > 0) scale(i - 1, d[(u - 1) & 1], col.dw);
        }
        scale(MT - 1, d[(2 * MT - 1) & 1], col.dw);
    };
    // nothing moves across a barrier
    auto sync = [&] {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    if (tid < 2) reinterpret_cast<int *>(lds + L::flag)[tid] = -1;
    load_w(wr[1], 0);
    load_x(0);
    load_w(wr[0], 1);
    sync();
    stage(wr[1], 0);
    sync();
    // the late half stages first: a step ahead of the early one from here on
    const int late = wave >= kWaves / 2 ? 1 : 0;
    if (late) {
        stage(wr[0], 1);
        load_w(wr[0], 2);
        load_w(wr[1], 3);
    }
    auto step = [&](WRaw<FMT> (&w)[WP], int k) {
        multiply(k);
        if (late) sync();
        stage(w, k + 1 + late);
        if (!late) sync();
    };
    for (int k = 0; k < nstep; k += 2) {
        step(wr[0], k);
        if (k + 1 < nstep) step(wr[1], k + 1);
    }
    if (xlive && xq8 == 0) {
#pragma unroll
        for (int p = 0; p < XP; ++p)
            fbuf(L::inv)[p * (kThreads / 8) + (tid >> 3)] = xs[p].limit > 0.0f ? xs[p].limit * 0x1p-15f : 1.0f;
    }
    __syncthreads();

    // lane (g, n) holds tokens 4g .. 4g+3 of each 16-token tile, weight row n of each 16-row tile
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int t0 = (wm * MT + i) * 16 + 4 * g;
        const f32x4 inv = *reinterpret_cast<const f32x4 *>(fbuf(L::inv) + t0);
#pragma unroll
        for (int t = 0; t < (MODE == kSwiGLU ? NT / 2 : NT); ++t) {
            const int o = o0 + (wn * (MODE == kSwiGLU ? NT / 2 : NT) + t) * 16 + n;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (o >= a.n || m0 + t0 + r >= a.m) continue;
                float *yp = a.y + static_cast<size_t>(m0 + t0 + r) * a.n + o;
                const float v = acc[i][t][r] * inv[r];
                if constexpr (MODE == kSwiGLU) {
                    const float u = acc[i][t + NT / 2][r] * inv[r];
                    *yp = v / (1.0f + expf(-v)) * u;
                } else if constexpr (MODE == kAdd) {
                    *yp += v;
                } else {
                    *yp = v;
                }
            }
        }
    }
}

template <int FMT, bool Q81, int MODE, class G>
hipError_t launch(const GemmArgs &a, hipStream_t s) {
    constexpr int out = MODE == kSwiGLU ? G::BN / 2 : G::BN;
    const dim3 grid = gemm_grid((a.n + out - 1) / out, (a.m + G::BM - 1) / G::BM);
    hipLaunchKernelGGL((gemm_kernel<FMT, Q81, MODE, G>), grid, dim3(kThreads), Lds<G>::bytes, s, a);
    return hipGetLastError();
}

using Large = Geo<4, 4, 2, 4>;  // 128 tokens x 256 rows
using Mid = Geo<2, 2, 2, 4>;    // 64 tokens x 128 rows

// Microseconds of a launch, measured: a step of a round of workgroups takes 2.5 us with the large tiles
// (matrix cores, vector ALU and LDS each about half busy); with the middle ones 1.35 us for one workgroup
// on a CU (a step's latency) and 1.75 us for two, which LDS and registers have room for (Q8_0 [14336, 4096] at
// 256 tokens 157 us with the large tiles, 117 with two of the middle ones; [28672, 1024] at 128 tokens 47 us
// with one middle one after the other, 35 with two at a time).  Filling and draining: 12 and 6 us.
struct GemmPlan {
    bool large;
    float us;
};
GemmPlan gemm_plan(int n, int k, int m, bool swiglu) {
    const int cus = device_info().cu_count > 0 ? device_info().cu_count : 256;
    const float steps = static_cast<float>((k / 32 + 1) / 2);
    auto groups = [&](int bm, int bn) {
        if (swiglu) bn /= 2;
        return static_cast<int64_t>((n + bn - 1) / bn) * ((m + bm - 1) / bm);
    };
    const int64_t lg = groups(Large::BM, Large::BN), mg = groups(Mid::BM, Mid::BN), rest = mg % (2 * cus);
    const float l = 12.0f + 2.5f * steps * static_cast<float>((lg + cus - 1) / cus);
    const float d = 6.0f + steps * (1.75f * static_cast<float>(mg / (2 * cus)) +
                                    (rest == 0 ? 0.0f : rest <= cus ? 1.35f : 1.75f));
    return l <= d ? GemmPlan{true, l} : GemmPlan{false, d};
}

template <int FMT, bool Q81, int MODE>
hipError_t by_size(const GemmArgs &a, hipStream_t s) {
    if (gemm_plan(a.n, a.k, a.m, MODE == kSwiGLU).large) return launch<FMT, Q81, MODE, Large>(a, s);
    return launch<FMT, Q81, MODE, Mid>(a, s);
}

template <int FMT>
hipError_t by_mode(const GemmArgs &a, bool q81, int mode, hipStream_t s) {
    if (q81) return by_size<FMT, true, kStore>(a, s);
    switch (mode) {
        case kStore: return by_size<FMT, false, kStore>(a, s);
        case kAdd: return by_size<FMT, false, kAdd>(a, s);
        case kSwiGLU: return by_size<FMT, false, kSwiGLU>(a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t run(int type, const GemmArgs &a, bool q81, int mode, hipStream_t s) {
    if (a.n == 0 || a.m == 0) return hipSuccess;
    switch (type) {
        case T_Q4_0: return by_mode<T_Q4_0>(a, q81, mode, s);
        case T_Q5_0: return by_mode<T_Q5_0>(a, q81, mode, s);
        case T_Q8_0: return by_mode<T_Q8_0>(a, q81, mode, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

float gemm_us(int n, int k, int m, bool swiglu) { return gemm_plan(n, k, m, swiglu).us; }

hipError_t gemm_f32(int type, const uint8_t *w0, const uint8_t *w1, size_t rb, const float *x, float *y, int n, int k,
                    int m, int mode, hipStream_t s) {
    return run(type, GemmArgs{w0, w1 ? w1 : w0, rb, x, y, n, m, k}, false, mode, s);
}

hipError_t gemm_q8_1(int type, const uint8_t *w, size_t rb, const uint8_t *xq, float *y, int n, int k, int m,
                     hipStream_t s) {
    return run(type, GemmArgs{w, w, rb, xq, y, n, m, k}, true, kStore, s);
}

}  // namespace qlin
