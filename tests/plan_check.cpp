// CPU check of the launch planners' LDS arithmetic (blog_amd/csrc/qlin_plan.hpp), built and run by
// tests/test_plan.py: every accepted plan fits the CU's 160 KB together with the kernel's static
// LDS, the edge shapes land on the right side of it, and a shape no plan fits is refused (so the
// caller takes the per-element kernels rather than a launch that would fail).
#include <cstdio>
#include <cstdlib>

#include "qlin_plan.hpp"

using namespace qlin::plan;

static int failures = 0;
#define CHECK(c)                                                          \
    do {                                                                  \
        if (!(c)) {                                                       \
            std::printf("FAIL line %d: %s\n", __LINE__, #c);              \
            ++failures;                                                   \
        }                                                                 \
    } while (0)

int main() {
    // decode GEMV: over shapes, sum sizes and static LDS, an accepted plan always fits
    const size_t statics[] = {0, 256, 512, 4096};
    long accepted = 0, refused = 0;
    for (int k = 256; k <= 65536; k += 256)
        for (int total : {1, 16, 300, 3584, 18944, 152064, 1 << 20})
            for (int se : {16, 32})
                for (bool sw : {false, true})
                    for (size_t st : statics) {
                        const Gemv p = gemv(total, k, k / 256, sw, se, 256, true);
                        if (gemv_fits(p, st)) {
                            ++accepted;
                            CHECK(p.lds + st <= kMaxLds);
                            CHECK(p.grid >= 1 && p.grid <= 256);
                        } else {
                            ++refused;
                        }
                    }
    CHECK(accepted > 0 && refused > 0);
    // the edge: one row (grid 1, one 16-row tile), K = 256 n: 4K + 2 pads + K/32 * 4 + 16 n * 4 =
    // 1120 n + 2 kXPad bytes
    {
        const size_t pad = 2 * kXPad;
        const int n_edge = static_cast<int>((kMaxLds - pad) / 1120);
        const Gemv e = gemv(1, 256 * n_edge, n_edge, false, 32, 256, true);
        CHECK(e.lds == 1120u * n_edge + pad);
        CHECK(gemv_fits(e, kMaxLds - 1120 * n_edge - pad));
        CHECK(!gemv_fits(e, kMaxLds - 1120 * n_edge - pad + 1));
        CHECK(!gemv_fits(gemv(1, 256 * (n_edge + 1), n_edge + 1, false, 32, 256, true), 0));
    }
    CHECK(!gemv_fits(gemv(16, 256, 1, false, 32, 256, true), kMaxLds));  // a kernel that cannot be read
    // the grouped MoE streaming plans: Q4_K SwiGLU, Q5_0 / Q8_0 / Q4_K down
    const StreamFmt q4k{256, true, 0}, q50{128, false, 4}, q80{128, false, 8};
    struct Case { StreamFmt f; bool sw; };
    const Case cases[] = {{q4k, true}, {q4k, false}, {q50, false}, {q80, false}};
    for (const Case &c : cases)
        for (int K = c.f.ce; K <= 24576; K += c.f.ce)
            for (int rows : {16, 1408, 2048, 2816, 7168})
                for (int R : {1, 6, 96, 4096})
                    for (size_t st : statics) {
                        const Stream p = stream(c.f, c.sw, rows, K, 64, R, 256, st, st);
                        if (!p.ok) continue;
                        CHECK(p.nq == 4 || p.nq == 2);
                        CHECK(p.piece >= 1);
                        CHECK(p.lds + st <= kMaxLds);
                    }
    // Q4_K SwiGLU at the edge of four routes per pass: fixed = 4*(4K + 2 pads) + 4*K/32*4, per tile
    // 2*4*nchunk*64
    {
        auto need4 = [](int K) { return 16L * K + 8L * kXPad + K / 2 + 2L * 4 * (K / 256) * 64; };
        int K = 256;
        while (need4(K + 256) <= static_cast<long>(kMaxLds)) K += 256;
        const size_t st_fit = kMaxLds - need4(K);
        const Stream a = stream(q4k, true, 16, K, 64, 6, 256, st_fit, st_fit);
        CHECK(a.ok && a.nq == 4 && a.lds + st_fit <= kMaxLds);
        const Stream b = stream(q4k, true, 16, K, 64, 6, 256, st_fit + 1, st_fit + 1);  // four no longer fit
        CHECK(b.ok && b.nq == 2 && b.lds + st_fit + 1 <= kMaxLds);
        const Stream c = stream(q4k, true, 16, 4 * K, 64, 6, 256, 0, 0);  // not even two routes
        CHECK(!c.ok);
        CHECK(!stream(q4k, true, 16, 256, 64, 6, 256, kMaxLds, kMaxLds).ok);  // unreadable kernels
    }
    // the quantizer's launch: a group per 32 blocks, its threads below 2^32 however many blocks there are
    for (int64_t blocks : {int64_t{1}, int64_t{33}, int64_t{1} << 20, int64_t{1} << 29, int64_t{1} << 31, int64_t{1} << 40}) {
        const int64_t g = quantize_groups(blocks);
        CHECK(g >= 1 && g <= (blocks + 31) / 32 && g * 256 < (int64_t{1} << 32));
        CHECK(g == (blocks + 31) / 32 || g == kQuantizeGroups);
    }
    // Q8_1 products in layouts that the 64-token GEMM does not take: few outputs stay with the block dots,
    // however long their rows; enough of them take the other GEMM.  (Q4_0 2, Q5_0 6, Q8_0 8)
    for (int type : {2, 6, 8}) {
        for (int m : {1, 2, 8, 64}) CHECK(q8_1_route(type, 512, 18976, m, false, true, 256) == Q81::kBlockDots);
        CHECK(q8_1_route(type, 300, 1056, 66, false, true, 256) == Q81::kBlockDots);
        CHECK(q8_1_route(type, 64, 96, 2, false, true, 256) == Q81::kBlockDots);
        CHECK(q8_1_route(type, 14336, 4128, 64, false, true, 256) == Q81::kGemm);
        CHECK(q8_1_route(type, 14336, 4128, 64, false, false, 256) == Q81::kBlockDots);  // 2-byte aligned activations
        CHECK(q8_1_route(type, 14336, 4096, 512, true, true, 256) == Q81::kGemm);
        CHECK(q8_1_route(type, 14336, 4096, 8, true, true, 256) == Q81::kQblk);
    }
    // the smallest products stay with rows_kernel (2.5 us for [16, 32] at 2 rows; the GEMM takes 3.7)
    for (int type : {2, 6, 8})
        CHECK(rows(type, 16, 32, 2, false, 256).us < gemm(type, false, 16, 32, 2, false, 256).us);
    // and short K: [512, 96] at 288 rows 4.7 against 6.6 us, [2304, 160] at 128 6.5 against 8.2
    for (int type : {2, 6, 8}) {
        CHECK(rows(type, 512, 96, 288, false, 256).us < gemm(type, false, 512, 96, 288, false, 256).us);
        CHECK(rows(type, 2304, 160, 128, false, 256).us < gemm(type, false, 2304, 160, 128, false, 256).us);
        CHECK(rows(type, 8300, 224, 130, false, 256).us > gemm(type, false, 8300, 224, 130, false, 256).us);
    }
    // rows_kernel takes what the entry points accept: x on any float, blocks on any 2 bytes, a lone row at an odd
    // stride (Q6_K 14; Q4_K 12 has a kernel of its own)
    for (int type : {2, 6, 8, 14}) {
        for (uintptr_t x : {0, 4, 8, 12}) CHECK(rows_layout_ok(type, 2, 6, 210, 64 + x, 100, 256));
        CHECK(rows_layout_ok(type, 16, 0, 211, 64, 1, 256));
        CHECK(!rows_layout_ok(type, 16, 0, 211, 64, 2, 256));
        CHECK(!rows_layout_ok(type, 16, 0, 210, 66, 100, 256));
    }
    CHECK(!rows_layout_ok(12, 16, 0, 144, 64, 100, 256));
    std::printf("%s: %ld gemv plans accepted, %ld refused\n", failures ? "FAILED" : "ok", accepted, refused);
    return failures ? 1 : 0;
}
