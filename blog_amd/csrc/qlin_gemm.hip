// qlin_gemm.hip -- the prefill GEMM of the 32-block formats: Q8_0, Q5_0 and Q4_0 weights times many rows of
// activations, f32 or Q8_1, on the matrix cores of gfx950.
//
//   y[r, o] (=|+=) sum_k w(o, k) x[r, k]                          (kernel.cu:1254-1279, quant_matmul_kernel)
//   y[r, o]  =     sum over 32-blocks of the Q8_1 block dots      (kernel.cu:2305-2402, quant_matmul_q8_1)
//   act[r, o] = g / (1 + expf(-g)) * u, g, u the rows of two matrices (SharedExperts.cpp:34-40)
//
// Operands, A the activations and B the weights, all products exact, f32 accumulation.
//   f32 activations: v_mfma_f32_16x16x32_bf16, x in its three bf16 parts (qlin_bf16x3.hpp), the weights as
//     integers; the block's d by one fma per output.  A workgroup that meets a value that does not fit the
//     parts computes its tile again at the end, as f32 values on v_mfma_f32_16x16x4_f32.
//   Q8_1 activations: v_mfma_f32_16x16x32_f16 on integers on both sides, so a block's dot is exact; its
//     scales d8 and d by a product and an fma per output.
//
// Tiling.  A workgroup of 8 waves computes BM tokens x BN weight rows in steps of 64 values of K.  Both
// operands of a step are staged in LDS once per workgroup, in the MFMA lane layout, two buffers: each weight
// decoded once for all BM tokens; f32 activations as they are (three parts would not fit beside the weights),
// split by the WN waves that read them.  The waves form a WM x WN grid, each MT x NT tiles of 16 x 16.  Between
// two barriers waves 0-3 (one per SIMD) multiply step k and then stage their share of step k + 1, while waves
// 4-7 stage theirs of step k + 1 and then multiply step k, so that one half's matrix instructions run beside the
// other's vector ones.  Global loads are one step ahead (activations, from L2) and two (weights).
//
// Slots of the LDS planes are permuted within a row group by an XOR with the k-group (A) or the chunk
// (B), so that the staging writes and the fragment reads both spread over the banks.
//
// Measured (f32 activations): Q8_0 [14336, 4096] at 512 tokens 1746 -> 181 us and Q4_0 [18944, 3584] at 203 tokens
// 618 -> 149 us against the f32 matrix cores with the weights decoded per 16 tokens (an fp16 pair of x under a
// scale per token: 155 and 132 us, but not exact); Q8_1 activations, Q8_0 [14336, 4096] at 512 tokens 303 -> 121 us
// against the 64-token tiles (155 with d8 q as an fp16 pair).  What bounds it: the step's chain (barrier, reads,
// splits, products, staging writes).  At [14336, 4096] x 512 vector instructions take 77% of an active SIMD's cycles
// and the matrix cores 54% (SQ_INSTS_VALU, SQ_VALU_MFMA_BUSY_CYCLES); 50 fewer of 450 vector instructions a step (Q4_0
// nibbles by v_cvt_off_f32_i4) and the splits spread between the MFMAs both left the times as they were.
//
// Blocks and rows are only 2-byte aligned in general; weights are read as wide loads at that alignment.
#include "qlin_bf16x3.hpp"
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_mfma.hpp"
#include "qlin_plan.hpp"
#include "qlin_values8.hpp"

#include <type_traits>

namespace qlin {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

enum : int { kStore = 0, kAdd = 1, kSwiGLU = 2 };

constexpr int kWaves = 8, kThreads = kWaves * 64;

template <int MT_, int NT_, int WM_, int WN_, int HT_>
struct Geo {
    static constexpr int HT = HT_;  // tiles multiplied before the ones before them are scaled
    static constexpr int MT = MT_, NT = NT_, WM = WM_, WN = WN_;
    static constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN;
    static constexpr int waves = MT * NT > 8 ? 2 : 4;  // per SIMD: two workgroups on a CU where LDS has room for them
    static_assert(WM * WN == kWaves, "8 waves");
};

// LDS, in uint4: two step buffers (activations: f32 values 0..3 and 4..7 of a lane's 8, or fp16 and the
// blocks' scales; weights; their block scales), then a flag.
template <class G, bool Q81>
struct Lds {
    static constexpr int a = G::BM / 16 * 2 * 64, b = G::BN / 16 * 2 * 64;
    static constexpr int x0 = 0, x1 = a, w = Q81 ? a : 2 * a, dw = w + b, dx = dw + 2 * G::BN / 4;
    static constexpr int buf = dx + (Q81 ? 2 * G::BM / 4 : 0);
    static constexpr int flag = 2 * buf, total = flag + 1;
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

__device__ __forceinline__ f32x4 mfma_h(const u32x4 &a, const u32x4 &b, const f32x4 &c) {
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
// fp16 integers of 8 bytes less off - 1024
__device__ __forceinline__ u32x4 minus8(uint32_t a, uint32_t b, f16x2 off) {
    return u32x4{h2u(bytes_lo(a) + off), h2u(bytes_hi(a) + off), h2u(bytes_lo(b) + off), h2u(bytes_hi(b) + off)};
}
__device__ __forceinline__ u32x4 f16_of_i8(uint32_t a, uint32_t b) {
    return minus8(a ^ 0x80808080u, b ^ 0x80808080u, splat(-1152.0f));
}

// Consumes a row of sums: pure arithmetic is otherwise sunk below the next products, whose results then
// all stay live.
template <int NT>
__device__ __forceinline__ void pin(f32x4 (&v)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(v[t]));
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

// Elements 8g .. 8g+7 of the block for g = 0..3 through put(g, values): fp16 beside Q8_1 activations, else bf16.
template <int FMT, bool F16, class Put>
__device__ __forceinline__ void decode(const WRaw<FMT> &r, Put put) {
    if constexpr (FMT == T_Q8_0) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t a = r.q[g >> 1][2 * (g & 1)], b = r.q[g >> 1][2 * (g & 1) + 1];
            put(g, F16 ? f16_of_i8(a, b) : bf16_of_i8(a, b));
            if constexpr (!F16) __builtin_amdgcn_sched_barrier(0);  // (8 floats live at a time)
        }
    } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // low nibbles: elements 0..15, high: 16..31
            uint32_t a = (r.q[2 * (g & 1)] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
            uint32_t b = (r.q[2 * (g & 1) + 1] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
            if constexpr (FMT == T_Q5_0) {
                a |= bit4_of_bytes(r.qh >> (8 * g));
                b |= bit4_of_bytes(r.qh >> (8 * g + 4));
            }
            constexpr float off = FMT == T_Q5_0 ? 16.0f : 8.0f;
            put(g, F16 ? minus8(a, b, splat(-1024.0f - off)) : bf16_of_u8(a, b, off));
            if constexpr (!F16) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int FMT, bool Q81, int MODE, class G>
__global__ __launch_bounds__(kThreads, G::waves) void gemm_kernel(const GemmArgs a) {
    using L = Lds<G, Q81>;
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

    int *const again = reinterpret_cast<int *>(lds + L::flag);  // some value does not fit the parts

    // ---- staging: activations.  Lane q of a token's 8 takes values 8q .. 8q+7 of the step.
    constexpr int XP = (BM * 8 + kThreads - 1) / kThreads;  // tokens per thread
    constexpr bool XAll = BM * 8 % kThreads == 0;
    constexpr int XB = Q81 ? 36 : 128;  // bytes of a block
    const int xq8 = tid & 7, xchunk = xq8 >> 2, xg = xq8 & 3;
    const bool xlive = XAll || tid < BM * 8;
    using XVec = std::conditional_t<Q81, uint2, f32x4>;
    XVec xv[XP][Q81 ? 1 : 2];
    uint32_t xds[Q81 ? XP : 1];  // a Q8_1 block's d and s
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
        const bool none = odd && step == nstep - 1 && xchunk;  // the missing last block: zeros
#pragma unroll
        for (int p = 0; p < XP; ++p) {
            const int tok = p * (kThreads / 8) + (tid >> 3);
            const int at = ((tok >> 4) * 2 + xchunk) * 64 + xg * 16 + ((tok & 15) ^ (2 * xq8));
            if constexpr (Q81) {
                buf[L::x0 + at] = __builtin_bit_cast(uint4, f16_of_i8(xv[p][0].x, xv[p][0].y));
                if (xg == 0)
                    reinterpret_cast<float *>(buf + L::dx)[xchunk * BM + tok] = none ? 0.0f : f16_bits_to_f32(xds[p] & 0xffffu);
            } else {
                if (odd && step == nstep - 1) {  // uniform
                    asm volatile("");            // (a branch, not selects in every step)
                    if (none) xv[p][0] = xv[p][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
                const f32x4 u = xv[p][0], v = xv[p][1];
                const float am = max3_abs(v[2], v[3], max3_abs(v[0], v[1], max3_abs(u[2], u[3], max3_abs(u[0], u[1], 0.0f))));
                if (out_of_range(am)) *again = 1;
                buf[L::x0 + at] = __builtin_bit_cast(uint4, u);
                buf[L::x1 + at] = __builtin_bit_cast(uint4, v);
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
    auto stage_w = [&](const WRaw<FMT> (&w)[WP], int step, uint4 *buf) {
        if (!wlive) return;
#pragma unroll
        for (int p = 0; p < WP; ++p) {
            const int r = p * (kThreads / 2) + (tid >> 1);
            const int at = ((r >> 4) * 2 + whalf) * 64 + ((r & 15) ^ (8 * whalf));
            decode<FMT, Q81>(w[p], [&](int gg, const u32x4 &v) { buf[L::w + at + 16 * gg] = __builtin_bit_cast(uint4, v); });
            // (the missing last block: 0, as its activations)
            reinterpret_cast<float *>(buf + L::dw)[whalf * BN + r] =
                odd && step == nstep - 1 && whalf ? 0.0f : f16_bits_to_f32(w[p].d);
            if (!Q81 && (w[p].d & 0x7c00u) == 0x7c00u) *again = 1;
        }
    };
    // The next steps' loads go out behind a step's staging.  Past the last step it stages the last blocks
    // again, into a buffer that is not read any more.
    auto stage = [&](WRaw<FMT> (&w)[WP], int step) {
        uint4 *buf = lds + (step & 1) * L::buf;
        stage_w(w, step, buf);
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
    // A row of HT tiles (of one chunk) at a time: the operands of the next one are read or split, and the row
    // before's products scaled, next to its MFMAs.
    constexpr int HT = G::HT, H = NT / HT;
    static_assert(NT % HT == 0, "whole groups of tiles");
    struct Raw {  // a lane's values of a tile row, and its Q8_1 tokens' scales
        u32x4 v[Q81 ? 1 : 2];
        f32x4 dx;
    };
    struct Operands {
        u32x4 part[Q81 ? 1 : 3];  // largest first
        f32x4 dx;
    };
    auto load_raw = [&](const uint4 *buf, int c, int i) {
        const int at = ((wm * MT + i) * 2 + c) * 64 + g * 16 + (n ^ (8 * c + 2 * g));
        Raw r{};
        r.v[0] = __builtin_bit_cast(u32x4, buf[L::x0 + at]);
        if constexpr (Q81)
            r.dx = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(buf + L::dx) + c * BM + (wm * MT + i) * 16 + 4 * g);
        else
            r.v[1] = __builtin_bit_cast(u32x4, buf[L::x1 + at]);
        return r;
    };
    auto operands = [&](const Raw &r) {
        Operands o;
        if constexpr (Q81) {
            o.part[0] = r.v[0];
            o.dx = r.dx;
        } else {
            split3(__builtin_bit_cast(f32x4, r.v[0]), __builtin_bit_cast(f32x4, r.v[1]), o.part[0], o.part[1], o.part[2]);
        }
        return o;
    };
    struct Cols {
        u32x4 b[HT];
        float dw[HT];
    };
    auto load_cols = [&](const uint4 *buf, int c, int h) {
        Cols v;
#pragma unroll
        for (int t = 0; t < HT; ++t) {
            const int tile = wn * NT + h * HT + t;
            v.b[t] = __builtin_bit_cast(u32x4, buf[L::w + (tile * 2 + c) * 64 + g * 16 + (n ^ (8 * c))]);
            v.dw[t] = reinterpret_cast<const float *>(buf + L::dw)[c * BN + tile * 16 + n];
        }
        return v;
    };
    auto multiply = [&](int step) {
        const uint4 *buf = lds + (step & 1) * L::buf;
        constexpr int N = 2 * H * MT;  // rows: row v is tile row v % MT of column group v / MT % H of chunk v / MT / H
        Raw raw[MT];
        Operands x[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) raw[i] = load_raw(buf, 0, i);
        Cols col = load_cols(buf, 0, 0), next = col;
        x[0] = operands(raw[0]);
        f32x4 d[2][HT], dxp = {};
        float dwp[HT] = {};  // the scales of the row before
        auto scale = [&](int v) {
            const int i = v % MT, h = v / MT % H;
            f32x4 s[HT];
#pragma unroll
            for (int t = 0; t < HT; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = Q81 ? d[v & 1][t][r] * dxp[r] : d[v & 1][t][r];
                    s[t][r] = fmaf(dwp[t], p, acc[i][h * HT + t][r]);
                }
            }
            pin(s);
#pragma unroll
            for (int t = 0; t < HT; ++t) acc[i][h * HT + t] = s[t];
        };
#pragma unroll
        for (int v = 0; v < N; ++v) {
            const int i = v % MT;
            __builtin_amdgcn_sched_barrier(0);
            if (i == 0 && v + MT < N) next = load_cols(buf, (v + MT) / MT / H, (v + MT) / MT % H);
            const Operands xi = x[i];
            f32x4 *dv = d[v & 1];
#pragma unroll
            for (int t = 0; t < HT; ++t)
                dv[t] = Q81 ? mfma_h(xi.part[0], col.b[t], f32x4{0.0f, 0.0f, 0.0f, 0.0f})
                            : mfma(xi.part[0], col.b[t], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
            if constexpr (!Q81) {
#pragma unroll
                for (int p = 1; p < 3; ++p)
#pragma unroll
                    for (int t = 0; t < HT; ++t) dv[t] = mfma(xi.part[p], col.b[t], dv[t]);
            }
            if (v > 0) scale(v - 1);
            // the next row's operands, if it is the first that uses them; its values two rows on
            if (v + 1 < N && (v + 1) / MT % H == 0) {
                const int i1 = (v + 1) % MT;
                x[i1] = operands(raw[i1]);
                if ((v + 1) / MT / H == 0) raw[i1] = load_raw(buf, 1, i1);
            }
            if (v == 0) raw[0] = load_raw(buf, 1, 0);
#pragma unroll
            for (int t = 0; t < HT; ++t) dwp[t] = col.dw[t];
            if constexpr (Q81) dxp = xi.dx;
            if (i == MT - 1) col = next;
        }
        scale(N - 1);
    };
    // nothing moves across a barrier
    auto sync = [&] {
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    if (tid == 0) *again = 0;
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
    if constexpr (!Q81) {
        __syncthreads();
        if (*again) {  // uniform, rare: the tile once more, as f32 values
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int o = MODE == kSwiGLU ? o0 + (wn * (NT / 2) + t % (NT / 2)) * 16 + n : o0 + (wn * NT + t) * 16 + n;
                const uint8_t *wr = (MODE == kSwiGLU && t >= NT / 2 ? a.w1 : a.w0) + static_cast<size_t>(min(o, a.n - 1)) * a.rb;
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const float *xr = static_cast<const float *>(a.x) +
                                      static_cast<size_t>(min(m0 + (wm * MT + i) * 16 + n, a.m - 1)) * a.k;
                    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
                    for (int kb = 0; kb < a.k; kb += 128) {  // (sums of 128 values first: a short chain of roundings)
                        f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
                        for (int k0 = kb + 8 * g; k0 < min(kb + 128, a.k); k0 += 32) {
                            Raw8<FMT> r;
                            raw8<FMT>(wr, k0, r);
                            float xe[8], v[8];
                            __builtin_memcpy(xe, __builtin_assume_aligned(xr + k0, 4), sizeof(xe));
                            values8<FMT>(r, k0, v);
#pragma unroll
                            for (int e = 0; e < 8; ++e) d = mfma_f32(xe[e], v[e], d);
                        }
                        sum += d;
                    }
                    acc[i][t] = sum;
                }
            }
        }
    }

    // lane (g, n) holds tokens 4g .. 4g+3 of each 16-token tile, weight row n of each 16-row tile
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int t0 = (wm * MT + i) * 16 + 4 * g;
#pragma unroll
        for (int t = 0; t < (MODE == kSwiGLU ? NT / 2 : NT); ++t) {
            const int o = o0 + (wn * (MODE == kSwiGLU ? NT / 2 : NT) + t) * 16 + n;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (o >= a.n || m0 + t0 + r >= a.m) continue;
                float *yp = a.y + static_cast<size_t>(m0 + t0 + r) * a.n + o;
                const float v = acc[i][t][r];
                if constexpr (MODE == kSwiGLU) {
                    const float u = acc[i][t + NT / 2][r];
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
    hipLaunchKernelGGL((gemm_kernel<FMT, Q81, MODE, G>), grid, dim3(kThreads), (Lds<G, Q81>::bytes), s, a);
    return hipGetLastError();
}

// Two and one tiles a row: no register spilled.  Four and two: 20-28 and 0-9 spilled, 223-273 us for [14336, 4096] at
// 512 tokens against 178-181.
using Large = Geo<2, 8, 4, 2, 2>;  // 128 tokens x 256 rows
using Mid = Geo<1, 4, 4, 2, 1>;    // 64 tokens x 128 rows
static_assert(Large::BM == plan::kGemmLarge.bm && Large::BN == plan::kGemmLarge.bn && Mid::BM == plan::kGemmMid.bm &&
                  Mid::BN == plan::kGemmMid.bn,
              "the plan's tiles");

template <int FMT, bool Q81, int MODE>
hipError_t by_size(const GemmArgs &a, hipStream_t s) {
    if (plan::gemm(FMT, Q81, a.n, a.k, a.m, MODE == kSwiGLU, cu_count()).large) return launch<FMT, Q81, MODE, Large>(a, s);
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

hipError_t gemm_f32(int type, const uint8_t *w0, const uint8_t *w1, size_t rb, const float *x, float *y, int n, int k,
                    int m, int mode, hipStream_t s) {
    return run(type, GemmArgs{w0, w1 ? w1 : w0, rb, x, y, n, m, k}, false, mode, s);
}

hipError_t gemm_q8_1(int type, const uint8_t *w, size_t rb, const uint8_t *xq, float *y, int n, int k, int m,
                     hipStream_t s) {
    return run(type, GemmArgs{w, w, rb, xq, y, n, m, k}, true, kStore, s);
}

}  // namespace qlin
