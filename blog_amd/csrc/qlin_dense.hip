// qlin_dense.hip -- quantized matmul over a few rows of f32 activations on the matrix cores, gfx950.
//
//   y[r, o] = sum_k w(o, k) * x[r, k]          (kernel.cu:1254-1279, quant_matmul_kernel; m > 1)
//   y[r, o] += ...                              (the gemm + add of SharedExperts.cpp:42-48)
//   act[r, o] = g / (1 + expf(-g)) * u,  g, u the rows of the gate and up matrices
//                                               (the gemm, gemm, silu_mul of SharedExperts.cpp:34-40)
//
// Q4_K (the shared experts) on v_mfma_f32_16x16x32_bf16 with the tokens as the MFMA rows
// (q4k_rows_dot, qlin_rows.hpp): the nibble q enters as the exact bf16 128 + q and x as the bf16 pair
// hi = bf16(x), lo = bf16(x - hi), so every product is exact and accumulates in f32; per sub-block
// and 16-token tile one MFMA pair gives sum x (128 + q) for 16 weight rows and another pair sum x,
// and two fmas per output apply the scales.  The other formats: rows_kernel, below.
//
// Layout (Q4_K).  A workgroup owns a tile of 16 output rows and all of K; its 8 waves take the
// super-blocks in turn (wave w: w, w + 8, ...).  Lane l supplies output row l % 16 and token l % 16 of the
// current 16-token tile, and elements 8g .. 8g+7 of each sub-block (g = l / 16).  D holds tokens 4g ..
// 4g+3 of row l % 16.  The waves' partials meet in LDS and are summed in wave order.  A grid row per 64
// tokens.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_mfma.hpp"
#include "qlin_rows.hpp"
#include "qlin_values8.hpp"
#include <type_traits>

namespace qlin {
namespace {

constexpr int kDWaves = 8, kDThreads = kDWaves * 64;
constexpr int kDTokens = 64;  // tokens per grid row (4 tiles of 16)

enum : int { kStore = 0, kAdd = 1, kSwiGLU = 2 };

struct DenseArgs {
    const uint8_t *w0, *w1;  // w1: the up matrix of kSwiGLU
    size_t rb;
    const float *x;
    float *y;
    int n, k, m;
    RouteCombine c;  // kAdd: a batched MoE decode's deferred combine (c.yr non-null), added before the product
};

// The deferred combine's routed total of (token t, row h): the routes in route order from 0, as the
// combine launch forms it (qlin_moe_grouped.hip).
__device__ __forceinline__ float routed_total(const RouteCombine &c, int t, int h, int hidden) {
    constexpr int kLoadsFirst = 16;
    float total = 0.0f;
    if (c.k <= kLoadsFirst) {  // uniform
        // every route's id, weight and result requested at once (one round trip), then the same sum
        // (a route without an expert has no result written; its value is read but not used)
        int e[kLoadsFirst];
        float y[kLoadsFirst], w[kLoadsFirst];
#pragma unroll
        for (int r = 0; r < kLoadsFirst; ++r) {
            if (r < c.k) {
                const int route = t * c.k + r;
                e[r] = c.ids[route];
                w[r] = c.rw[route];
                y[r] = c.yr[static_cast<size_t>(route) * hidden + h];
            }
        }
#pragma unroll
        for (int r = 0; r < kLoadsFirst; ++r)
            if (r < c.k && e[r] >= 0 && e[r] < c.n_experts) total = fmaf(y[r], w[r], total);
        return total;
    }
    for (int r = 0; r < c.k; ++r) {
        const int route = t * c.k + r, e = c.ids[route];
        if (e < 0 || e >= c.n_experts) continue;
        total = fmaf(c.yr[static_cast<size_t>(route) * hidden + h], c.rw[route], total);
    }
    return total;
}
// y = (y + routed total) + v: the combine launch's y += total, then the plain add
__device__ __forceinline__ void add_out(const DenseArgs &a, float *yo, int t, int h, float v) {
    float y = *yo;
    if (a.c.yr) y += routed_total(a.c, t, h, a.n);  // uniform
    *yo = y + v;
}

template <int MODE>
__global__ __launch_bounds__(kDThreads) void q4k_dense_kernel(const DenseArgs a) {
    constexpr int NW = MODE == kSwiGLU ? 2 : 1;
    __shared__ f32x4 part[kDWaves][NW][4][64];  // [wave][matrix][token tile][lane]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int K = a.k, nsb = K / 256;
    const int row0 = blockIdx.x * 16;
    const int row = min(row0 + n, a.n - 1);
    const int t0 = blockIdx.y * kDTokens;
    const int ntt = min(4, (a.m - t0 + 15) / 16);  // token tiles of this grid row
    const uint8_t *rp[2] = {a.w0 + static_cast<size_t>(row) * a.rb, a.w1 + static_cast<size_t>(row) * a.rb};
    const int rows = min(16, a.n - row0);

    // kAdd over at most two token tiles (thread i writes output i alone): what is added before the
    // product -- the output's current value and a batched MoE decode's routed results with their
    // ids and weights -- depends on nothing this launch computes, so it is requested here, ahead of
    // the weights, and the same adds in the same order run at the end (one round trip fewer after the
    // sums)
    constexpr int kPreRoutes = MODE == kAdd ? 8 : 1;
    const bool pre = MODE == kAdd && ntt <= 2 && a.c.k <= kPreRoutes;  // uniform
    const int ptl = tid >> 4, po = tid & 15, pt = t0 + ptl;
    const bool pown = pre && tid < ntt * 256 && po < rows && pt < a.m;
    float pre_y = 0.0f, pre_v[kPreRoutes], pre_w[kPreRoutes];
    int pre_e[kPreRoutes];
    if constexpr (MODE == kAdd) {
        if (pown) {
            pre_y = a.y[static_cast<size_t>(pt) * a.n + row0 + po];
            if (a.c.yr) {  // uniform
#pragma unroll
                for (int r = 0; r < kPreRoutes; ++r) {
                    if (r < a.c.k) {
                        const int route = pt * a.c.k + r;
                        pre_e[r] = a.c.ids[route];
                        pre_w[r] = a.c.rw[route];
                        pre_v[r] = a.c.yr[static_cast<size_t>(route) * a.n + row0 + po];
                    }
                }
            }
        }
    }

    // one 16-token tile at a time (a tile's weights come again from the cache for the next one)
    for (int tt = 0; tt < ntt; ++tt) {
        // token of this lane's A row (tokens past m read the last one; their D rows are dropped)
        const int tok = min(t0 + tt * 16 + n, a.m - 1);
        const float *xrow = a.x + static_cast<size_t>(tok) * K + 8 * g;
        f32x4 D[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) D[w] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // wave w takes super-blocks w, w + 8, ...
        q4k_rows_dot<NW>(rp, xrow, wave, kDWaves, nsb, g, D);
#pragma unroll
        for (int w = 0; w < NW; ++w) part[wave][w][tt][lane] = D[w];
    }
    __syncthreads();

    // outputs: row o = row0 + (i % 16), token t0 + i / 16; D element r of lane l is token 4(l/16) + r
    for (int i = tid; i < ntt * 256; i += kDThreads) {
        const int tl = i >> 4, o = i & 15;  // token within the grid row, row within the tile
        const int t = t0 + tl;
        if (o >= rows || t >= a.m) continue;
        const int tt = tl >> 4, l = ((tl & 15) >> 2) * 16 + o, r = tl & 3;
        float v0 = 0.0f, v1 = 0.0f;
        for (int wv = 0; wv < kDWaves; ++wv) {
            v0 += part[wv][0][tt][l][r];
            if constexpr (NW == 2) v1 += part[wv][NW - 1][tt][l][r];
        }
        float *yo = a.y + static_cast<size_t>(t) * a.n + row0 + o;
        if constexpr (MODE == kSwiGLU) {
            *yo = v0 / (1.0f + expf(-v0)) * v1;
        } else if constexpr (MODE == kAdd) {
            if (pre) {  // (then i == tid)
                float y = pre_y;
                if (a.c.yr) {
                    float total = 0.0f;  // routed_total's sum from the preloaded values
#pragma unroll
                    for (int r = 0; r < kPreRoutes; ++r)
                        if (r < a.c.k && pre_e[r] >= 0 && pre_e[r] < a.c.n_experts) total = fmaf(pre_v[r], pre_w[r], total);
                    y += total;
                }
                *yo = y + v0;
            } else {
                add_out(a, yo, t, row0 + o, v0);
            }
        } else {
            *yo = v0;
        }
    }
}

// ---- the other formats (Q4_0, Q5_0, Q8_0, Q6_K) --------------------------------------------------
//
// v_mfma_f32_16x16x32_f16 with the tokens as the MFMA rows, the operands of the prefill GEMM
// (qlin_gemm.hip): B = q less its offset (Q6_K: sc (q - 32) in two exact parts), A = x 2^s split into fp16
// hi and lo, s per token from its largest magnitude so far (rescaled when a value 8 times that comes).
// Nothing is shared between waves: each takes whole units of four 32-blocks of K in turn (wave w: w, w + 8,
// ...) for all of the workgroup's rows and tokens, straight from memory, one unit's weights and one token
// tile's x ahead, so short and narrow products need no barrier per step; the waves' sums meet in LDS.
// What bounds it: a tile's chain (x turned in LDS, its scale, 64 split and 16-32 scaling instructions
// around 8-16 MFMAs) with two waves on a SIMD.  A request whose lanes lie in different rows costs the
// address path a cycle per lane, which is why x is read along its rows and a lane group reads a whole
// block.  Against f32 matrix cores (v_mfma_f32_16x16x4_f32) on decoded values with the layout's own
// 8-byte pieces: Q6_K [3584, 18944] at 12 rows 78 -> 33 us, Q5_0 [4096, 4096] at 6 rows 19 -> 10 us, Q8_0
// [4096, 4096] at 100 rows 108 -> 38 us, Q5_0 [30000, 1024] at 40 rows 92 -> 26 us.

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma_h(const uint4 &a, const uint4 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t h2u(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f16x2 u2h(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ f16x2 splat(float v) {
    const _Float16 h = static_cast<_Float16>(v);
    return f16x2{h, h};
}
// the fp16 pairs 1024 + byte of bytes 0, 1 and 2, 3
__device__ __forceinline__ f16x2 bytes_lo(uint32_t v) { return u2h(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)); }
__device__ __forceinline__ f16x2 bytes_hi(uint32_t v) { return u2h(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)); }
__device__ __forceinline__ uint4 minus8(uint32_t a, uint32_t b, f16x2 off) {
    return make_uint4(h2u(bytes_lo(a) + off), h2u(bytes_hi(a) + off), h2u(bytes_lo(b) + off), h2u(bytes_hi(b) + off));
}
__device__ __forceinline__ uint32_t bit4_of_bytes(uint32_t b) { return (__umul24(b & 0xfu, 0x204081u) & 0x01010101u) << 4; }

constexpr int kUnit = 4;  // 32-blocks of a unit

// Lane moves between the four groups of 16 lanes (rows) of a wave.
// swap32(a, b): a = {a's rows 0, 1, b's rows 0, 1}, b = {a's rows 2, 3, b's rows 2, 3}
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = static_cast<uint32_t>(s[0]);
    b = static_cast<uint32_t>(s[1]);
}
// swap16(a, b): a = {a0, b0, a2, b2}, b = {a1, b1, a3, b3} by rows
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = static_cast<uint32_t>(s[0]);
    b = static_cast<uint32_t>(s[1]);
}
// o[j] = group j's v, in every group
__device__ __forceinline__ void all_groups(uint32_t v, uint32_t (&o)[4]) {
    uint32_t lo = v, hi = v;
    swap32(lo, hi);
    o[0] = o[1] = lo;
    swap16(o[0], o[1]);
    o[2] = o[3] = hi;
    swap16(o[2], o[3]);
}

// A unit of one row, loaded with a whole block per lane group (as few, wide requests as the layout of one
// row per lane allows: each costs the address path a cycle per lane), then exchanged between the groups
// so that group g holds elements 8g .. 8g+7 of every block.  blk: the unit's first block; last: the row's
// last block (a unit cut short reads it again).
template <int T>
struct Unit {
    static constexpr int W = T == T_Q8_0 ? 8 : 4;
    uint32_t q[W], d, qh;
    __device__ __forceinline__ void load(const uint8_t *row, int blk, int last, int g) {
        const uint8_t *b = row + static_cast<size_t>(min(blk + g, last)) * Block<T>::bytes;
        d = ld_u16(b);
        if constexpr (T == T_Q5_0) qh = ld4_a2(b + 2);
#pragma unroll
        for (int i = 0; i < W; i += 4) {
            const u32x4 v = ld16_a2(b + (T == T_Q5_0 ? 6 : 2) + 4 * i);
            q[i] = v.x;
            q[i + 1] = v.y;
            q[i + 2] = v.z;
            q[i + 3] = v.w;
        }
    }
    // the operands and scales of the unit's blocks
    __device__ __forceinline__ void operands(int g, uint4 (&b)[kUnit], uint4 (&)[1], float (&dw)[kUnit]) const {
        uint32_t ds[4], o[kUnit][2];
        all_groups(d, ds);
#pragma unroll
        for (int e = 0; e < 2; ++e) {  // the dwords of a lane's 8 bytes
            if constexpr (T == T_Q8_0) {
                uint32_t m0 = q[e], m1 = q[2 + e], m2 = q[4 + e], m3 = q[6 + e];
                swap32(m0, m2);
                swap32(m1, m3);
                swap16(m0, m1);
                swap16(m2, m3);
                o[0][e] = m0;
                o[1][e] = m1;
                o[2][e] = m2;
                o[3][e] = m3;
            } else {  // bytes 8 (g & 1) .. + 7 of every block
                uint32_t m0 = q[e], m1 = q[2 + e];
                swap16(m0, m1);
                uint32_t a0 = m0, a2 = m0, a1 = m1, a3 = m1;
                swap32(a0, a2);
                swap32(a1, a3);
                o[0][e] = a0;
                o[1][e] = a1;
                o[2][e] = a2;
                o[3][e] = a3;
            }
        }
        [[maybe_unused]] uint32_t h[4];
        if constexpr (T == T_Q5_0) all_groups(qh, h);
#pragma unroll
        for (int j = 0; j < kUnit; ++j) {
            dw[j] = f16_bits_to_f32(ds[j]);
            if constexpr (T == T_Q8_0) {
                b[j] = minus8(o[j][0] ^ 0x80808080u, o[j][1] ^ 0x80808080u, splat(-1152.0f));
            } else {  // low nibbles: elements 0..15, high: 16..31
                uint32_t u = (o[j][0] >> (4 * (g >> 1))) & 0x0f0f0f0fu, v = (o[j][1] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
                if constexpr (T == T_Q5_0) {
                    const uint32_t hb = h[j] >> (8 * g);
                    u |= bit4_of_bytes(hb);
                    v |= bit4_of_bytes(hb >> 4);
                }
                b[j] = minus8(u, v, splat(T == T_Q5_0 ? -1040.0f : -1032.0f));
            }
        }
    }
};
template <>
struct Unit<T_Q6_K> {  // half a super-block
    uint2 l[2], h, sc;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *row, int blk, int, int g) {
        const uint8_t *sb = row + static_cast<size_t>(blk >> 3) * 210;
        const int half = (blk >> 2) & 1;
        l[0] = ld8_a2(sb + 64 * half + 8 * g);
        l[1] = ld8_a2(sb + 64 * half + 32 + 8 * g);
        h = ld8_a2(sb + 128 + 32 * half + 8 * g);
        sc = ld8_a2(sb + 192 + 8 * half);
        d = ld_u16(sb + 208);
    }
    __device__ __forceinline__ void operands(int g, uint4 (&b1)[kUnit], uint4 (&b2)[kUnit], float (&dw)[kUnit]) const {
        dw[0] = f16_bits_to_f32(d);
#pragma unroll
        for (int j = 0; j < kUnit; ++j) operand(j, g, b1[j], b2[j]);
    }
    __device__ __forceinline__ void operand(int j, int g, uint4 &b1, uint4 &b2) const {
        const uint32_t s = (((j < 2 ? sc.x : sc.y) >> (8 * (2 * (j & 1) + (g >> 1)))) & 0xffu) ^ 0x80u;
        const f16x2 s2 = u2h(0x64006400u | s | (s << 16)) + splat(-1152.0f);
        const uint2 lw = l[j & 1];
        const uint32_t u = ((lw.x >> (4 * (j >> 1))) & 0x0f0f0f0fu) | (((h.x >> (2 * j)) & 0x03030303u) << 4);
        const uint32_t v = ((lw.y >> (4 * (j >> 1))) & 0x0f0f0f0fu) | (((h.y >> (2 * j)) & 0x03030303u) << 4);
        const uint4 q = minus8(u, v, splat(-1056.0f));
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        uint32_t p1[4], p2[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const f16x2 p = u2h(w[e]) * s2;
            p1[e] = h2u(p);
            p2[e] = h2u(__builtin_elementwise_fma(u2h(w[e]), s2, -p));
        }
        b1 = make_uint4(p1[0], p1[1], p1[2], p1[3]);
        b2 = make_uint4(p2[0], p2[1], p2[2], p2[3]);
    }
};

// max over the four lane groups of v (>= 0, whose bits order as it does): every lane gets its token's
__device__ __forceinline__ float max_over_groups(float v) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto s = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const uint32_t c = max(static_cast<uint32_t>(s[0]), static_cast<uint32_t>(s[1]));
    const auto t = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return __builtin_bit_cast(float, max(static_cast<uint32_t>(t[0]), static_cast<uint32_t>(t[1])));
}
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// hi and lo fp16 parts of 8 values times sc (a power of two)
__device__ __forceinline__ void split8(const f32x4 &a, const f32x4 &b, float sc, uint4 &hi, uint4 &lo) {
    const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = h2u(f16x2{static_cast<_Float16>(fmaf(v[2 * i], sc, 0.0f)), static_cast<_Float16>(fmaf(v[2 * i + 1], sc, 0.0f))});
        asm("" : "+v"(h[i]));  // one packed value (its halves would otherwise be formed twice)
        const f16x2 hp = u2h(h[i]);
        l[i] = h2u(f16x2{static_cast<_Float16>(fmaf(v[2 * i], sc, -static_cast<float>(hp[0]))),
                         static_cast<_Float16>(fmaf(v[2 * i + 1], sc, -static_cast<float>(hp[1])))});
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

template <int T, int MODE, int NT, int TT>
__global__ __launch_bounds__(kDThreads) void rows_kernel(const DenseArgs a) {
    static_assert(MODE != kSwiGLU || NT % 2 == 0, "gate and up tiles in pairs");
    constexpr int OT = MODE == kSwiGLU ? NT / 2 : NT;  // output row tiles
    constexpr bool Q6 = T == T_Q6_K;
    extern __shared__ f32x4 part[];  // [wave][row tile][token tile][lane]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int K = a.k, nblk = K / 32, nunit = (nblk + kUnit - 1) / kUnit;
    int bx, by;
    gemm_tile((a.n + 16 * OT - 1) / (16 * OT), (a.m + 16 * TT - 1) / (16 * TT), bx, by);
    const int row0 = bx * 16 * OT, t0 = by * 16 * TT;

    const uint8_t *rp[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const size_t row = min(row0 + (t % OT) * 16 + n, a.n - 1);
        rp[t] = (t < OT ? a.w0 : a.w1) + row * a.rb;
    }
    f32x4 acc[TT][NT];
    float limit[TT];  // 2^(15 - s) of the lane's token in each tile (0: no value yet)
#pragma unroll
    for (int i = 0; i < TT; ++i) {
        limit[i] = 0.0f;
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }

    // x of a token tile's unit: read along the tokens' rows (32 lanes of a token, two tokens a request),
    // turned in the wave's own LDS (slot c of token t at c ^ t) into lane (token n, elements 8g .. 8g+7 of
    // every block).  A wave's LDS accesses complete in order, so it needs no waits of its own.
    f32x4 *turn = part + wave * (16 * 8 * kUnit);
    const int lt = lane >> 5, lc = lane & 31;
    auto load_x = [&](f32x4 (&x)[2 * kUnit], int i, int u) {
        // a unit cut short reads the row's last block again
        const int c = min(8 * kUnit * u + lc, 8 * nblk - 8 + (lc & 7));
#pragma unroll
        for (int p = 0; p < 2 * kUnit; ++p)
            x[p] = reinterpret_cast<const f32x4 *>(a.x + static_cast<size_t>(min(t0 + 16 * i + 2 * p + lt, a.m - 1)) * K)[c];
    };
    auto turn_x = [&](const f32x4 (&x)[2 * kUnit], f32x4 (&r)[2 * kUnit]) {
#pragma unroll
        for (int p = 0; p < 2 * kUnit; ++p) turn[(2 * p + lt) * 32 + (lc ^ (2 * p + lt))] = x[p];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int e = 0; e < 2 * kUnit; ++e) r[e] = turn[n * 32 + ((8 * (e >> 1) + 2 * g + (e & 1)) ^ n)];
        __builtin_amdgcn_wave_barrier();
    };
    Unit<T> raw[NT];
    f32x4 ahead[2 * kUnit];
    int u = wave;
    if (u < nunit) {
#pragma unroll
        for (int t = 0; t < NT; ++t) raw[t].load(rp[t], kUnit * u, nblk - 1, g);
        load_x(ahead, 0, u);
    }
    for (; u < nunit; u += kDWaves) {  // uniform
        uint4 B[NT][kUnit], B2[NT][Q6 ? kUnit : 1];
        float dw[NT][kUnit];
#pragma unroll
        for (int t = 0; t < NT; ++t) raw[t].operands(g, B[t], B2[t], dw[t]);
        const int next = u + kDWaves;
        auto tile = [&](int i) {
            f32x4 x[2 * kUnit];
            turn_x(ahead, x);
            // the next tile's x (of this unit or the next); the next unit's weights behind the first tile's
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < TT) load_x(ahead, i + 1, u);
            else if (next < nunit) load_x(ahead, 0, next);
            if (i == 0 && next < nunit) {
#pragma unroll
                for (int t = 0; t < NT; ++t) raw[t].load(rp[t], kUnit * next, nblk - 1, g);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!Q6 && kUnit * u + kUnit > nblk) {  // uniform: a unit cut short
                asm volatile("");
#pragma unroll
                for (int j = 1; j < kUnit; ++j)
                    if (kUnit * u + j >= nblk) x[2 * j] = x[2 * j + 1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            float am = 0.0f;
#pragma unroll
            for (int e = 0; e < 2 * kUnit; ++e) am = max3_abs(x[e][2], x[e][3], max3_abs(x[e][0], x[e][1], am));
            am = max_over_groups(am);
            const bool inf = !(am <= 3.4e38f);
            if (__any(am > limit[i])) {  // uniform, rare: new scales, the sums so far brought to them
                asm volatile("");
                float f = 1.0f;
                if (am > limit[i]) {
                    if (inf) {
                        if (limit[i] == 0.0f) limit[i] = 32768.0f;
                    } else {
                        int ex;
                        (void)frexpf(am, &ex);
                        const float was = limit[i];
                        limit[i] = ldexpf(1.0f, 15 - min(13 - ex, 120));
                        if (was > 0.0f) f = was / limit[i];
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float fr = __shfl(f, 4 * g + r, 64);
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[i][t][r] *= fr;
                }
            }
            // 2^s: the exponents of limit and 2^s add up to 15 (no value yet: some finite number, against zeros)
            const float sc = __builtin_bit_cast(float, (269u << 23) - __builtin_bit_cast(uint32_t, limit[i]));
            auto blocks = [&](auto with_inf) {
                [[maybe_unused]] f32x4 D6[NT];
#pragma unroll
                for (int j = 0; j < kUnit; ++j) {
                    uint4 hi, lo;
                    split8(x[2 * j], x[2 * j + 1], sc, hi, lo);
                    uint4 hi2 = hi;  // against B2, which may be 0 where the weight is not: no infinite values
                    if constexpr (decltype(with_inf)::value) {
                        drop_inf(hi, lo);
                        drop_inf(hi, hi2);
                    }
                    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (Q6) {  // d is the unit's: its blocks add up first
#pragma unroll
                        for (int t = 0; t < NT; ++t) D6[t] = mfma_h(hi, B[t][j], j ? D6[t] : zero);
#pragma unroll
                        for (int t = 0; t < NT; ++t) D6[t] = mfma_h(hi2, B2[t][j], D6[t]);
#pragma unroll
                        for (int t = 0; t < NT; ++t) D6[t] = mfma_h(lo, B[t][j], D6[t]);
                    } else {
                        f32x4 D[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t) D[t] = mfma_h(hi, B[t][j], zero);
#pragma unroll
                        for (int t = 0; t < NT; ++t) D[t] = mfma_h(lo, B[t][j], D[t]);
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[i][t][r] = fmaf(dw[t][j], D[t][r], acc[i][t][r]);
                    }
                }
                if constexpr (Q6) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][t][r] = fmaf(dw[t][0], D6[t][r], acc[i][t][r]);
                }
            };
            if (__any(inf)) blocks(std::true_type{});  // uniform
            else blocks(std::false_type{});
#pragma unroll
            for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(acc[i][t]));  // (not sunk below the next tile)
        };
        tile(0);
        if constexpr (TT > 1) tile(1);
        if constexpr (TT > 2) tile(2);
        if constexpr (TT > 3) tile(3);
    }
    __syncthreads();  // (the sums below take the LDS of the tiles)

    // each wave's sums at their true scale; lane (row, g) of D holds tokens 4g .. 4g+3
#pragma unroll
    for (int i = 0; i < TT; ++i) {
        const float inv = limit[i] > 0.0f ? limit[i] * 0x1p-15f : 1.0f;
        f32x4 iv;
#pragma unroll
        for (int r = 0; r < 4; ++r) iv[r] = __shfl(inv, 4 * g + r, 64);
#pragma unroll
        for (int t = 0; t < NT; ++t) part[((wave * NT + t) * TT + i) * 64 + lane] = acc[i][t] * iv;
    }
    __syncthreads();
    const int rows = min(16 * OT, a.n - row0), toks = min(16 * TT, a.m - t0);
    for (int e = tid; e < 16 * OT * 16 * TT; e += kDThreads) {
        const int tl = e / (16 * OT), o = e % (16 * OT);
        if (o >= rows || tl >= toks) continue;
        const int i = tl >> 4, t = o >> 4, l = ((tl & 15) >> 2) * 16 + (o & 15), r = tl & 3;
        float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
        for (int w = 0; w < kDWaves; ++w) {
            v0 += part[((w * NT + t) * TT + i) * 64 + l][r];
            if constexpr (MODE == kSwiGLU) v1 += part[((w * NT + OT + t) * TT + i) * 64 + l][r];
        }
        float *yo = a.y + static_cast<size_t>(t0 + tl) * a.n + row0 + o;
        if constexpr (MODE == kSwiGLU) *yo = v0 / (1.0f + expf(-v0)) * v1;
        else if constexpr (MODE == kAdd) add_out(a, yo, t0 + tl, row0 + o, v0);
        else *yo = v0;
    }
}

template <int T, int MODE, int NT, int TT>
hipError_t launch_rows(const DenseArgs &a, hipStream_t s) {
    constexpr int OT = MODE == kSwiGLU ? NT / 2 : NT;
    const auto max = [](int a, int b) { return a > b ? a : b; };
    const dim3 grid = gemm_grid((a.n + 16 * OT - 1) / (16 * OT), (a.m + 16 * TT - 1) / (16 * TT));
    hipLaunchKernelGGL((rows_kernel<T, MODE, NT, TT>), grid, dim3(kDThreads), sizeof(f32x4) * kDWaves * max(NT * TT * 64, 16 * 8 * kUnit), s, a);
    return hipGetLastError();
}

// The tiles of a launch: NT row tiles (of a SwiGLU: NT / 2 outputs') by TT token tiles per workgroup, one
// workgroup on a CU at a time.  Measured, a round of workgroups takes about 2 us plus, per unit of a wave,
// 2.1 (1 x 1), 3.3 (2 x 1), 3.2 (1 x 2), 4.6 (2 x 2), 6.6 (2 x 3) and 8.8 us (2 x 4): larger tiles split x and read the
// weights for more products, smaller ones fill the chip.  The cheapest total is taken (Q8_0 [896, 4864] at 384
// tokens: 168 workgroups of 2 x 4 tiles 44 us, 224 of 2 x 3 32 us).
struct RowsPlan {
    int nt, tt;
    float us;
};
RowsPlan rows_plan(int n, int k, int m, bool swiglu) {
    static constexpr struct {
        int nt, tt;
        float unit;
    } kinds[] = {{1, 1, 2.1f}, {2, 1, 3.3f}, {1, 2, 3.2f}, {2, 2, 4.6f}, {2, 3, 6.6f}, {2, 4, 8.8f}};
    const int cus = device_info().cu_count > 0 ? device_info().cu_count : 256;
    const float units = static_cast<float>((k / 32 + kUnit * kDWaves - 1) / (kUnit * kDWaves));
    RowsPlan best{0, 0, 0.0f};
    for (const auto &c : kinds) {
        if (swiglu && c.nt == 1) continue;
        const int rows = 16 * c.nt / (swiglu ? 2 : 1), toks = 16 * c.tt;
        const int64_t wgs = static_cast<int64_t>((n + rows - 1) / rows) * ((m + toks - 1) / toks);
        const float us = static_cast<float>((wgs + cus - 1) / cus) * (2.0f + units * c.unit);
        if (!best.nt || us < best.us) best = RowsPlan{c.nt, c.tt, us};
    }
    return best;
}

template <int T, int MODE>
hipError_t by_shape(const DenseArgs &a, hipStream_t s) {
    const RowsPlan p = rows_plan(a.n, a.k, a.m, MODE == kSwiGLU);
    if constexpr (MODE != kSwiGLU) {
        if (p.nt == 1) return p.tt == 1 ? launch_rows<T, MODE, 1, 1>(a, s) : launch_rows<T, MODE, 1, 2>(a, s);
    }
    switch (p.tt) {
        case 1: return launch_rows<T, MODE, 2, 1>(a, s);
        case 2: return launch_rows<T, MODE, 2, 2>(a, s);
        case 3: return launch_rows<T, MODE, 2, 3>(a, s);
        default: return launch_rows<T, MODE, 2, 4>(a, s);
    }
}

template <int T>
hipError_t launch_dense(const DenseArgs &a, int mode, hipStream_t s) {
    switch (mode) {
        case kStore: return by_shape<T, kStore>(a, s);
        case kAdd: return by_shape<T, kAdd>(a, s);
        case kSwiGLU: return by_shape<T, kSwiGLU>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool dense_ok(int type, const uint8_t *w0, const uint8_t *w1, size_t rb, const float *x, int k) {
    const auto al = [](const void *p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & (m - 1)) == 0; };
    if (type == T_Q4_K) return k % 256 == 0 && rb % 16 == 0 && al(w0, 16) && (!w1 || al(w1, 16)) && al(x, 16);
    if (type != T_Q4_0 && type != T_Q5_0 && type != T_Q8_0 && type != T_Q6_K) return false;
    // the per-element decoder reads 16-bit fields: 2-byte aligned blocks
    return k % 32 == 0 && rb % 2 == 0 && al(w0, 2) && (!w1 || al(w1, 2)) && al(x, 16);
}

float dense_us(int n, int k, int m, bool swiglu) { return rows_plan(n, k, m, swiglu).us; }

hipError_t dense_matmul(int type, const uint8_t *w0, const uint8_t *w1, size_t rb, const float *x, float *y, int n,
                        int k, int m, int mode, hipStream_t s, const RouteCombine *combine) {
    if (n == 0 || m == 0) return hipSuccess;
    DenseArgs a{w0, w1 ? w1 : w0, rb, x, y, n, k, m, RouteCombine{}};
    if (combine && mode == kAdd) a.c = *combine;
    const dim3 grid((n + 15) / 16, (m + kDTokens - 1) / kDTokens);
    switch (type) {
        case T_Q4_K: break;
        case T_Q4_0: return launch_dense<T_Q4_0>(a, mode, s);
        case T_Q5_0: return launch_dense<T_Q5_0>(a, mode, s);
        case T_Q8_0: return launch_dense<T_Q8_0>(a, mode, s);
        case T_Q6_K: return launch_dense<T_Q6_K>(a, mode, s);
        default: return hipErrorInvalidValue;
    }
    switch (mode) {
        case kStore: hipLaunchKernelGGL(q4k_dense_kernel<kStore>, grid, dim3(kDThreads), 0, s, a); break;
        case kAdd: hipLaunchKernelGGL(q4k_dense_kernel<kAdd>, grid, dim3(kDThreads), 0, s, a); break;
        case kSwiGLU: hipLaunchKernelGGL(q4k_dense_kernel<kSwiGLU>, grid, dim3(kDThreads), 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace qlin
