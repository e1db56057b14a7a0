// qlin_plan.hpp -- launch planning of the matrix-core streaming kernels: host-only arithmetic, no
// HIP calls, so the same code is checked on the CPU (tests/plan_check.cpp).
//
// A plan gives the workgroup count and the dynamic LDS of a launch.  The kernels' own (static) LDS
// is an input: the callers read it from the compiled kernels (hipFuncGetAttributes), and a plan is
// accepted only when static + dynamic LDS fits the CU's 160 KB.  A shape no plan fits takes the
// per-element kernels instead, so a call that passes validation never fails at launch for LDS.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace qlin {
namespace plan {

constexpr size_t kMaxLds = 160 * 1024;  // LDS per CU on gfx950
// Padding of each staged x part (bf16 hi or lo, int8 digit plane) past its K values, in bytes: an
// A-operand read gathers one offset of several parts, and a part length that is a multiple of the
// LDS bank row (256 bytes) would put them all in the same banks.  16 bytes (one b128 read) shifts
// each part by 4 banks.  Staging of a route (one x) takes 4K + 2 kXPad bytes as bf16 parts.
constexpr int kXPad = 16;

// The decode GEMV (qlin_mfma_gemv.hip): one workgroup per CU over `total` rows of nsb chunks of
// k / nsb weights.  Dynamic LDS: x in the bf16 layout (4K + 2 kXPad bytes, which the int8 digit
// planes, 3 (K + kXPad) bytes and their sums, never exceed), the x sums (one float per sum_elems elements) and one partial per (row,
// matrix, chunk) of the workgroup's rows.  interleave: workgroup b takes 16-row tiles b, b + G, ...
struct Gemv {
    int grid = 0;
    size_t lds = 0;
    bool magic_exact = false;  // every step index c of a workgroup has c * nsb < 2^32
};
inline Gemv gemv(int total, int k, int nsb, bool swiglu, int sum_elems, int cu_count, bool interleave) {
    Gemv p;
    p.grid = std::max(1, std::min(cu_count, (total + 15) / 16));
    const int rows = interleave ? ((total + 15) / 16 + p.grid - 1) / p.grid * 16 : (total + p.grid - 1) / p.grid;
    const uint64_t steps = static_cast<uint64_t>((rows + 15) / 16) * (swiglu ? 2 : 1) * static_cast<uint64_t>(nsb);
    p.magic_exact = steps * static_cast<uint64_t>(nsb) < (uint64_t{1} << 32);
    const size_t K = static_cast<size_t>(k);
    p.lds = 4 * K + 2 * kXPad + (K / static_cast<size_t>(sum_elems)) * sizeof(float) +
            static_cast<size_t>(rows) * (swiglu ? 2 : 1) * static_cast<size_t>(nsb) * sizeof(float);
    return p;
}
inline bool gemv_fits(const Gemv &p, size_t static_lds) {
    return p.magic_exact && static_lds <= kMaxLds && p.lds <= kMaxLds - static_lds;
}

// The grouped MoE streaming kernels (qlin_moe_grouped.hip): routes per pass nq (4, else 2), and the
// tiles whose partials fit in LDS at once.  Dynamic LDS: the pass's routes' staged x (Q4_K 4K +
// 2 kXPad bytes; the 32-weight formats tpb 16-byte slot vectors per block and hi / lo part, each part
// kXPad bytes longer), one x sum
// per 32 elements and route, and per tile nw * nq * nchunk * 16 partials.  The selected experts are
// only known on the device, so a piece is sized for twice an even share of min(E, R) of them.
struct StreamFmt {
    int ce;     // weights per chunk
    bool q4k;   // Q4_K staging (otherwise slot vectors)
    int tpb;    // 16-byte slot vectors per block (32-weight formats)
};
struct Stream {
    bool ok = false;
    int nq = 0, grid = 0, piece = 0;
    size_t lds = 0;
};
inline Stream stream(const StreamFmt &f, bool swiglu, int rows, int K, int E, int R, int cu_count,
                     size_t static_nq4, size_t static_nq2) {
    Stream p;
    const int nw = swiglu ? 2 : 1;
    const int nblk = K / 32, nchunk = K / f.ce, tpe = (rows + 15) / 16;
    const int grid = std::max(1, cu_count);
    const int64_t share = (static_cast<int64_t>(std::min(E, R)) * tpe + grid - 1) / grid;
    for (int nq = 4; nq >= 2; nq -= 2) {
        const size_t st = nq == 4 ? static_nq4 : static_nq2;
        if (st >= kMaxLds) continue;
        const size_t budget = kMaxLds - st;
        const size_t stage = f.q4k ? static_cast<size_t>(nq) * (4 * K + 2 * kXPad)
                                   : static_cast<size_t>(nq) * 2 * (nblk * f.tpb * 16 + kXPad);
        const size_t fixed = stage + static_cast<size_t>(nq) * nblk * sizeof(float);
        const size_t per_tile = static_cast<size_t>(nw) * nq * nchunk * 16 * sizeof(float);
        if (fixed + per_tile > budget) continue;
        const int64_t cap = static_cast<int64_t>((budget - fixed) / per_tile);
        p.ok = true;
        p.nq = nq;
        p.grid = grid;
        p.piece = static_cast<int>(std::min<int64_t>(cap, std::max<int64_t>(1, 2 * share)));
        p.lds = fixed + static_cast<size_t>(p.piece) * per_tile;
        return p;
    }
    return p;
}

// Several rows of activations: the formats' order in the tables below (ggml types Q4_0, Q5_0, Q8_0, Q6_K).
inline int rows_format(int type) { return type == 2 ? 0 : type == 6 ? 1 : type == 8 ? 2 : type == 14 ? 3 : -1; }
inline int64_t tiles(int n, int bn, int m, int bm) {
    return static_cast<int64_t>((n + bn - 1) / bn) * ((m + bm - 1) / bm);
}

// The row products of qlin_dense.hip (rows_kernel): nt row tiles (of a SwiGLU: nt / 2 outputs') by tt token tiles
// of 16 per workgroup, one workgroup on a CU at a time, whose 8 waves take units of 128 values of K in turn.
// us is base plus, per round of workgroups, round + unit x (the units of K / 8: a tenth of it rounded up to whole
// turns of the waves), by least squares of the logarithm over the tiles of 61 shapes of each format (36 of n 512 ..
// 32768, k 512 .. 16384, m 2 .. 700; full rounds of k 1024 .. 16384; 13 of k 32 .. 512, not of Q6_K): 5-7% off in
// the mean; the kernel and tiles it picks are 0.1-0.2% slower in the mean than the fastest, 10% at worst.  Larger
// tiles split x and read the weights for more products, smaller ones fill the chip.  Q6_K has no 2 x 4 tiles (they
// spill: 8.2 us a unit, as much per product as 2 x 3's 6.0), the others no 1 x 2 (the cheapest for 6 of 10000 shapes).
struct Rows {
    int nt = 0, tt = 0;
    float us = 0.0f;
};
inline Rows rows(int type, int n, int k, int m, bool swiglu, int cus) {
    static constexpr int nt[6] = {1, 2, 1, 2, 2, 2}, tt[6] = {1, 1, 2, 2, 3, 4};
    static constexpr struct {
        float base, round[6], unit[6];
    } costs[4] = {{1.15f, {1.3f, 1.85f, 0.0f, 2.75f, 3.7f, 4.55f}, {1.51f, 2.13f, 0.0f, 3.36f, 4.38f, 5.4f}},
                  {1.0f, {1.4f, 2.0f, 0.0f, 2.95f, 3.95f, 5.0f}, {1.65f, 2.46f, 0.0f, 3.68f, 4.76f, 5.81f}},
                  {1.1f, {1.3f, 1.7f, 0.0f, 2.6f, 3.55f, 4.6f}, {1.68f, 2.65f, 0.0f, 3.95f, 5.0f, 6.24f}},
                  {1.3f, {1.35f, 1.85f, 1.9f, 2.45f, 3.55f, 0.0f}, {1.93f, 3.34f, 2.96f, 4.69f, 5.98f, 0.0f}}};
    const int f = rows_format(type);
    Rows best;
    if (f < 0) return best;
    const int all = (k / 32 + 3) / 4;
    const float units = 0.1f * static_cast<float>((all + 7) / 8) + 0.1125f * static_cast<float>(all);
    for (int i = 0; i < 6; ++i) {
        if (i == (f == 3 ? 5 : 2) || (swiglu && nt[i] == 1)) continue;
        const int64_t wgs = tiles(n, 16 * nt[i] / (swiglu ? 2 : 1), m, 16 * tt[i]);
        const float us = costs[f].base + static_cast<float>((wgs + cus - 1) / cus) * (costs[f].round[i] + units * costs[f].unit[i]);
        if (!best.nt || us < best.us) {
            best.nt = nt[i];
            best.tt = tt[i];
            best.us = us;
        }
    }
    return best;
}

// The prefill GEMM (qlin_gemm.hip): its tiles (bm tokens x bn rows) and the microseconds of a launch, fill + K steps
// of 64 x the cost of one, fitted as above (5-9% off in the mean): with the large tiles a step per round of
// workgroups; with the middle ones a step of one workgroup on a CU, or of two at a time, which LDS and registers
// have room for.
struct Tile {
    int bm, bn;
};
constexpr Tile kGemmLarge{128, 256}, kGemmMid{64, 128};
struct Gemm {
    bool large = false;
    float us = 0.0f;
};
inline Gemm gemm(int type, bool q81, int n, int k, int m, bool swiglu, int cus) {
    static constexpr struct {
        float fill, step, mid_fill, mid_two, mid_one;
    } costs[2][3] = {{{6.3f, 2.56f, 3.35f, 2.15f, 1.4f}, {6.8f, 2.65f, 3.35f, 2.28f, 1.55f}, {7.0f, 2.54f, 3.3f, 2.27f, 1.51f}},
                     {{7.5f, 1.67f, 1.85f, 1.3f, 0.86f}, {7.6f, 1.71f, 2.6f, 1.41f, 0.99f}, {7.1f, 1.69f, 1.75f, 1.17f, 1.07f}}};
    const int f = rows_format(type);
    if (f < 0 || f > 2) return Gemm{};
    const auto &c = costs[q81 ? 1 : 0][f];
    const float steps = static_cast<float>((k / 32 + 1) / 2);
    const int64_t lg = tiles(n, kGemmLarge.bn / (swiglu ? 2 : 1), m, kGemmLarge.bm);
    const int64_t mg = tiles(n, kGemmMid.bn / (swiglu ? 2 : 1), m, kGemmMid.bm), rest = mg % (2 * cus);
    const float l = c.fill + c.step * steps * static_cast<float>((lg + cus - 1) / cus);
    const float d = c.mid_fill + steps * (c.mid_two * static_cast<float>(mg / (2 * cus)) +
                                          (rest == 0 ? 0.0f : rest <= cus ? c.mid_one : c.mid_two));
    Gemm g;
    g.large = l <= d;
    g.us = g.large ? l : d;
    return g;
}

// The Q8_1 GEMM of 64-token tiles (qlin_qblk_gemm.hip), for the 32-block formats: the default tiles, the small ones
// where those would leave more than half the CUs idle, and the microseconds of a launch, fill + units of 256
// values x the cost of one per round of workgroups, fitted as above (4-9% off).
constexpr Tile kQblkLarge{64, 256}, kQblkSmall{32, 128};
inline bool qblk_small(int n, int m, int cus) { return tiles(n, kQblkLarge.bn, m, kQblkLarge.bm) * 2 < cus; }
inline float qblk_us(int type, int n, int k, int m, int cus) {
    static constexpr float fill[3] = {3.9f, 3.75f, 4.15f}, small[3] = {2.89f, 3.03f, 2.97f}, large[3] = {6.8f, 6.65f, 6.55f};
    const int f = rows_format(type);
    if (f < 0 || f > 2) return 0.0f;
    const bool s = qblk_small(n, m, cus);
    const Tile t = s ? kQblkSmall : kQblkLarge;
    return fill[f] + static_cast<float>((tiles(n, t.bn, m, t.bm) + cus - 1) / cus) * (s ? small[f] : large[f]) *
                         static_cast<float>((k + 255) / 256);
}

// The block dots of matmul_q8_1_kernel (qlin_q8_1.hip, any layout): a wave per output, 64 blocks of K at a time.
// Measured per output and 64 blocks: Q8_0 [512, 18976] at 64 rows 117 us, [2048, 352] at 8 rows 7.9.
inline float block_dots_us(int type, int n, int k, int m) {
    static constexpr float dot[3] = {3.75e-4f, 4.3e-4f, 3.5e-4f};
    const int f = rows_format(type);
    const float rounds = static_cast<float>((k / 32 + 63) / 64);
    return 2.0f + rounds * (0.3f + dot[f < 0 || f > 2 ? 1 : f] * static_cast<float>(m) * static_cast<float>(n));
}
// The kernel of a 32-block product with Q8_1 activations: the cheaper GEMM where the 64-token one takes the layout
// (qblk_ok), else the other GEMM against the block dots (Q8_0 [512, 18976] at 2 rows: 270 us against 9.7; from 16
// rows of [4096, 4128] on the GEMM).
enum class Q81 { kGemm, kQblk, kBlockDots };
inline Q81 q8_1_route(int type, int n, int k, int m, bool qblk_ok, bool gemm_ok, int cus) {
    const float other = qblk_ok ? qblk_us(type, n, k, m, cus) : block_dots_us(type, n, k, m);
    if (gemm_ok && gemm(type, true, n, k, m, false, cus).us < other) return Q81::kGemm;
    return qblk_ok ? Q81::kQblk : Q81::kBlockDots;
}

// The layouts that rows_kernel reads: blocks at 2-byte and x at 4-byte alignment (a 16-byte load on a dword
// boundary runs as an aligned one), a lone row at any stride.
inline bool rows_layout_ok(int type, uintptr_t w0, uintptr_t w1, size_t row_bytes, uintptr_t x, int n, int k) {
    return rows_format(type) >= 0 && k % (type == 14 ? 256 : 32) == 0 && (n <= 1 || row_bytes % 2 == 0) && w0 % 2 == 0 &&
           w1 % 2 == 0 && x % 4 == 0;
}

// The prefill GEMM of the super-block formats (qlin_f32_gemm.hip): the default tiles, unless they would leave more
// than half the CUs idle, and the microseconds of a Q6_K launch (a round of workgroups takes about 6.8 us per
// super-block on the default tiles and 3.2 on the small ones).
constexpr Tile kSuperLarge{64, 256}, kSuperSmall{32, 128};
inline bool super_block_small(int n, int m, int cus) { return tiles(n, kSuperLarge.bn, m, kSuperLarge.bm) * 2 < cus; }
inline float super_block_us(int n, int k, int m, int cus) {
    const bool s = super_block_small(n, m, cus);
    const Tile t = s ? kSuperSmall : kSuperLarge;
    return 4.0f + static_cast<float>((tiles(n, t.bn, m, t.bm) + cus - 1) / cus) * (s ? 3.2f : 6.8f) * static_cast<float>(k / 256);
}

// The kernel of a product with m > 1 rows of f32 activations, as dense_matmul (kDense: rows_kernel, Q4_K's own) and the
// GEMMs take the layout: the GEMM of the 32-block formats where its tiles fill the chip or x is long enough to be
// staged once per tile (below that the waves of a workgroup split K), that of the super-block formats from min_rows
// rows on (Q6_K: where it is the cheaper one; Q4_K's dense_matmul holds less of x).
enum class Product { kPerElement, kDense, kGemm, kSuperBlockGemm };
inline Product product(int type, int n, int k, int m, bool dense_ok, bool super_block_ok, int min_rows, int cus) {
    const int f = rows_format(type);
    if (f >= 0 && f < 3)
        return !dense_ok || gemm(type, false, n, k, m, false, cus).us < rows(type, n, k, m, false, cus).us ? Product::kGemm
                                                                                                       : Product::kDense;
    if (m >= min_rows && super_block_ok &&
        (f < 0 || !dense_ok || super_block_us(n, k, m, cus) <= rows(type, n, k, m, false, cus).us))
        return Product::kSuperBlockGemm;
    return dense_ok ? Product::kDense : Product::kPerElement;
}
// The same of a SwiGLU over m > 1 rows (no GEMM of the super-block formats has that mode).
inline Product swiglu_product(int type, int ffn, int k, int m, bool dense_ok, int cus) {
    const int f = rows_format(type);
    if (f >= 0 && f < 3 && (!dense_ok || gemm(type, false, ffn, k, m, true, cus).us < rows(type, ffn, k, m, true, cus).us))
        return Product::kGemm;
    return dense_ok ? Product::kDense : Product::kPerElement;
}

// Workgroups of the Q8_1 quantizer (8 lanes per block, 32 blocks at a time): at most kQuantizeGroups, which then take
// further blocks in turn, since a launch's threads have to stay below 2^32 (2^29 blocks, 64 GiB of x).
constexpr int64_t kQuantizeGroups = int64_t{1} << 16;
inline int64_t quantize_groups(int64_t blocks) { return std::min(kQuantizeGroups, (blocks + 31) / 32); }

}  // namespace plan
}  // namespace qlin
