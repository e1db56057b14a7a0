// The kernels that products with several rows of f32 activations take at 256 CUs (blog_amd/csrc/qlin_plan.hpp):
// for each input line "type n k m swiglu", the name that the case lists of tests/test_gpu_parity.py give it.
// Layouts as the tests have them: every kernel takes the activations, the super-block GEMM rows on dwords.
#include <iostream>

#include "qlin_plan.hpp"

using namespace qlin::plan;

int main() {
    int type, n, k, m, swiglu;
    while (std::cin >> type >> n >> k >> m >> swiglu) {
        const bool super_ok = type == 12 || (type == 14 && k / 256 * 210 % 4 == 0);
        const Product p = swiglu ? swiglu_product(type, n, k, m, true, 256) : product(type, n, k, m, true, super_ok, 64, 256);
        const Rows r = rows(type, n, k, m, swiglu != 0, 256);
        if (p == Product::kGemm) std::cout << (gemm(type, false, n, k, m, swiglu != 0, 256).large ? "large" : "mid") << '\n';
        else if (p == Product::kSuperBlockGemm) std::cout << (super_block_small(n, m, 256) ? "super small" : "super") << '\n';
        else if (p == Product::kDense && r.nt) std::cout << r.nt << 'x' << r.tt << '\n';
        else std::cout << (p == Product::kDense ? "q4k" : "per element") << '\n';
    }
    return 0;
}
