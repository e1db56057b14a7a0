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
#include "qlin_bf16x3.hpp"
#include "qlin_internal.hpp"
#include "qlin_mfma.hpp"
#include "qlin_plan.hpp"
#include "qlin_rows.hpp"
#include "qlin_values8.hpp"

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
// The tokens are the MFMA rows; x enters in its three exact bf16 parts and the weights as integers
// (qlin_bf16x3.hpp).  32-block formats: v_mfma_f32_16x16x32_bf16, one scale per block.  Q6_K, whose scales
// are per 16 values: v_mfma_f32_16x16x16_bf16, one scale d sc (exact in f32) per MFMA sum.
// Nothing is shared between waves: each takes whole units of four 32-blocks of K in turn (wave w: w, w + 8,
// ...) for all of the workgroup's rows and tokens, straight from memory, one unit's weights and one token
// tile's x ahead, so short and narrow products need no barrier per step; the waves' sums meet in LDS.
// A request whose lanes lie in different rows costs the address path a cycle per lane, which is why x is read
// along its rows and a lane group reads a whole block.
// What bounds it: a tile's chain (x turned in LDS, 176 instructions to split its 32 values a lane, 12-24 MFMAs and
// their scaling) with two or three waves on a SIMD.  Against f32 matrix cores (v_mfma_f32_16x16x4_f32) on decoded
// values: Q6_K [3584, 18944] at 12 rows 78 -> 33 us, Q5_0 [4096, 4096] at 6 rows 18.4 -> 9.2 us, Q8_0 [4096, 4096]
// at 100 rows 107 -> 32 us; 2-norm error against f64 over N(0, 1) x 2.1e-7 .. 8.6e-7 -> 0.7e-7 .. 1.2e-7 (0.9e-7 .. 1.6e-7
// as an fp16 pair under a scale per token, at the same times).  149 registers (1 x 1) to 256 (2 x 4: 0 to 6 of them
// spilled, Q6_K's 2 x 3 up to 6; the measured costs in qlin_plan.hpp include them).

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
    static constexpr int kScales = kUnit;  // the unit's scales
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
    __device__ __forceinline__ void operands(int g, u32x4 (&b)[kUnit], float (&dw)[kScales]) const {
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
                b[j] = bf16_of_i8(o[j][0], o[j][1]);
            } else {  // low nibbles: elements 0..15, high: 16..31
                uint32_t u = (o[j][0] >> (4 * (g >> 1))) & 0x0f0f0f0fu, v = (o[j][1] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
                if constexpr (T == T_Q5_0) {
                    const uint32_t hb = h[j] >> (8 * g);
                    u |= bit4_of_bytes(hb);
                    v |= bit4_of_bytes(hb >> 4);
                }
                b[j] = bf16_of_u8(u, v, T == T_Q5_0 ? 16.0f : 8.0f);
            }
        }
    }
    // x's slot (f32x4) e of the unit for lane group g: elements 8g + 4 (e & 1) .. + 3 of block e / 2
    static __device__ __forceinline__ int x_slot(int e, int g) { return 8 * (e >> 1) + 2 * g + (e & 1); }
};
// Half a super-block.  A lane reads bytes 8g .. 8g+7 of each 32, of one 16-value group for lanes of groups 0
// and 1, of the other for 2 and 3; after the swap every lane has 4 values of each 16-group: group g of
// 16-group s has its elements 8 (g & 1) + 4 (g >> 1) .. + 3.  b[j]: those of 16-groups 2j and 2j + 1.
template <>
struct Unit<T_Q6_K> {
    static constexpr int kScales = 2 * kUnit;
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
    __device__ __forceinline__ void operands(int, u32x4 (&b)[kUnit], float (&dw)[kScales]) const {
        const float df = f16_bits_to_f32(d);
        uint2 lo[2] = {l[0], l[1]}, hi = h;
        swap32(lo[0].x, lo[0].y);
        swap32(lo[1].x, lo[1].y);
        swap32(hi.x, hi.y);
#pragma unroll
        for (int j = 0; j < kUnit; ++j) {
            const uint2 lw = lo[j & 1];
            const uint32_t u = ((lw.x >> (4 * (j >> 1))) & 0x0f0f0f0fu) | (((hi.x >> (2 * j)) & 0x03030303u) << 4);
            const uint32_t v = ((lw.y >> (4 * (j >> 1))) & 0x0f0f0f0fu) | (((hi.y >> (2 * j)) & 0x03030303u) << 4);
            b[j] = bf16_of_u8(u, v, 32.0f);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                dw[2 * j + s] = mul_rn(df, static_cast<float>(static_cast<int8_t>((j < 2 ? sc.x : sc.y) >> (8 * (2 * (j & 1) + s)))));
        }
    }
    static __device__ __forceinline__ int x_slot(int e, int g) { return 4 * e + 2 * (g & 1) + (g >> 1); }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 mfma16(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, make_uint2(a0, a1)),
                                                     __builtin_bit_cast(s16x4, make_uint2(b0, b1)), c, 0, 0, 0);
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
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // x of a token tile's unit: read along the tokens' rows (32 lanes of a token, two tokens a request),
    // turned in the wave's own LDS (slot c of token t at c ^ t) into lane (token n, the lane group's slots).
    // A wave's LDS accesses complete in order, so it needs no waits of its own.
    f32x4 *turn = part + wave * (16 * 8 * kUnit);
    const int lt = lane >> 5, lc = lane & 31;
    auto load_x = [&](f32x4 (&x)[2 * kUnit], int i, int u) {
        // a unit cut short reads the row's last block again
        const int c = min(8 * kUnit * u + lc, 8 * nblk - 8 + (lc & 7));
#pragma unroll
        for (int p = 0; p < 2 * kUnit; ++p)
            __builtin_memcpy(&x[p], __builtin_assume_aligned(a.x + static_cast<size_t>(min(t0 + 16 * i + 2 * p + lt, a.m - 1)) * K + 4 * c, 4), 16);
    };
    auto turn_x = [&](const f32x4 (&x)[2 * kUnit], f32x4 (&r)[2 * kUnit]) {
#pragma unroll
        for (int p = 0; p < 2 * kUnit; ++p) turn[(2 * p + lt) * 32 + (lc ^ (2 * p + lt))] = x[p];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int e = 0; e < 2 * kUnit; ++e) r[e] = turn[n * 32 + (Unit<T>::x_slot(e, g) ^ n)];
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
        u32x4 B[NT][kUnit];
        float dw[NT][Unit<T>::kScales];
        float dmax = 0.0f;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            raw[t].operands(g, B[t], dw[t]);
            // (the packed values, not the floats they were made from, stay live)
#pragma unroll
            for (int j = 0; j < kUnit; ++j) asm("" : "+v"(B[t][j]));
#pragma unroll
            for (int j = 0; j < Unit<T>::kScales; j += 2) dmax = max3_abs(dw[t][j], dw[t][j + 1], dmax);
        }
        const bool winf = !(dmax <= 3.4e38f);  // (a scale that is NaN makes NaN either way)
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
            if (__any(out_of_range(am) || winf)) {  // uniform, rare: as f32 values
#pragma unroll
                for (int j = 0; j < kUnit; ++j) {
                    if (!Q6 && kUnit * u + j >= nblk) break;  // uniform (its weights are not the row's)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        u32x4 b = B[t][j];
                        asm volatile("" : "+v"(b));  // (the f32 values are not kept from tile to tile)
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            acc[i][t] = mfma_f32(x[2 * j + (e >> 2)][e & 3],
                                                 mul_rn(dw[t][Q6 ? 2 * j + (e >> 2) : j], bf16_at(b, e)), acc[i][t]);
                    }
                }
                return;
            }
            // (the unit's own sum, then added: a shorter chain of roundings)
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            f32x4 sum[NT];
#pragma unroll
            for (int j = 0; j < kUnit; ++j) {
                u32x4 hi, mid, lo;
                split3(x[2 * j], x[2 * j + 1], hi, mid, lo);
                auto scaled = [&](const f32x4 (&D)[NT], int scale) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            sum[t][r] = scale ? fmaf(dw[t][scale], D[t][r], sum[t][r]) : dw[t][0] * D[t][r];
                };
                if constexpr (Q6) {
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        f32x4 D[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t) D[t] = mfma16(hi[2 * s], hi[2 * s + 1], B[t][j][2 * s], B[t][j][2 * s + 1], zero);
#pragma unroll
                        for (int t = 0; t < NT; ++t) D[t] = mfma16(mid[2 * s], mid[2 * s + 1], B[t][j][2 * s], B[t][j][2 * s + 1], D[t]);
#pragma unroll
                        for (int t = 0; t < NT; ++t) D[t] = mfma16(lo[2 * s], lo[2 * s + 1], B[t][j][2 * s], B[t][j][2 * s + 1], D[t]);
                        scaled(D, 2 * j + s);
                    }
                } else {
                    // the small parts' sum apart from hi's: 0.7e-7 .. 0.9e-7 from f64 instead of 1.0e-7 .. 1.1e-7, for 1-3%
                    // of the time (Q6_K's sums are half as long: 1.2e-7 either way, and 4%)
                    f32x4 D[NT], E[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) D[t] = mfma(hi, B[t][j], zero);
#pragma unroll
                    for (int t = 0; t < NT; ++t) E[t] = mfma(mid, B[t][j], zero);
#pragma unroll
                    for (int t = 0; t < NT; ++t) E[t] = mfma(lo, B[t][j], E[t]);
#pragma unroll
                    for (int t = 0; t < NT; ++t) D[t] += E[t];
                    scaled(D, j);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                acc[i][t] += sum[t];
                asm volatile("" : "+v"(acc[i][t]));  // (not sunk below the next tile)
            }
        };
        tile(0);
        if constexpr (TT > 1) tile(1);
        if constexpr (TT > 2) tile(2);
        if constexpr (TT > 3) tile(3);
    }
    __syncthreads();  // (the sums below take the LDS of the tiles)

    // lane (row, g) of D holds tokens 4g .. 4g+3
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) part[((wave * NT + t) * TT + i) * 64 + lane] = acc[i][t];
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

template <int T, int MODE>
hipError_t by_shape(const DenseArgs &a, hipStream_t s) {
    const plan::Rows p = plan::rows(T, a.n, a.k, a.m, MODE == kSwiGLU, cu_count());
    if constexpr (MODE != kSwiGLU) {
        if constexpr (T == T_Q6_K) {
            if (p.nt == 1 && p.tt == 2) return launch_rows<T, MODE, 1, 2>(a, s);
        }
        if (p.nt == 1) return launch_rows<T, MODE, 1, 1>(a, s);
    }
    if constexpr (T != T_Q6_K) {
        if (p.tt == 4) return launch_rows<T, MODE, 2, 4>(a, s);
    }
    switch (p.tt) {
        case 1: return launch_rows<T, MODE, 2, 1>(a, s);
        case 2: return launch_rows<T, MODE, 2, 2>(a, s);
        default: return launch_rows<T, MODE, 2, 3>(a, s);
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

bool dense_ok(int type, const uint8_t *w0, const uint8_t *w1, size_t rb, const float *x, int n, int k) {
    const auto at = [](const void *p) { return reinterpret_cast<uintptr_t>(p); };
    if (type == T_Q4_K) return k % 256 == 0 && rb % 16 == 0 && (at(w0) | at(w1) | at(x)) % 16 == 0;
    return plan::rows_layout_ok(type, at(w0), at(w1), rb, at(x), n, k);
}

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
