// qlin_q8_1.hip -- Q8_1 activation quantizer and the quantized-weight x Q8_1 matmul (prefill), gfx950.
// The block quantizer and the per-type block dots (kernel.cu:1679-1720, 2305-2402) are in qlin_q8_1.hpp.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_plan.hpp"
#include "qlin_q8_1.hpp"

namespace qlin {
namespace {

// 8 lanes per 32-block: a wave reads 1 KB of a row and writes 8 blocks.  With one
// thread per block, its 32 values in turn, quantizing 512 rows of 4096 and multiplying them by Q4_K
// [14336, 4096] took 151 us; now 147, 5.0 of them here.
__global__ __launch_bounds__(256) void quantize_q8_1_kernel(const float *__restrict__ x, uint8_t *__restrict__ xq,
                                                            int in_dim, int64_t blocks, int bpr, int raw) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 32;
    const int j = threadIdx.x & 7;
    for (int64_t gb = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) >> 3; gb < blocks; gb += stride) {  // (whole groups of 8 lanes)
        const int64_t r = gb / bpr;
        const int b = static_cast<int>(gb - r * bpr);
        // 36-byte blocks: 4-aligned
        quantize_block_q8_1_lanes(x + r * in_dim, 32 * b + 4 * j, in_dim, j, reinterpret_cast<uint32_t *>(xq + gb * 36), raw != 0);
    }
}

// One wave per (activation row, output row); lanes over 32-wide blocks.
template <int T>
__global__ __launch_bounds__(256) void matmul_q8_1_kernel(const uint8_t *__restrict__ w, size_t rb,
                                                          const uint8_t *__restrict__ xq, float *__restrict__ y,
                                                          int out_dim, int in_dim, int m) {
    const int64_t wave = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave >= static_cast<int64_t>(m) * out_dim) return;
    const int r = static_cast<int>(wave / out_dim), o = static_cast<int>(wave - static_cast<int64_t>(r) * out_dim);
    const int bpr = in_dim / 32;
    const uint8_t *row = w + static_cast<size_t>(o) * rb;
    const uint8_t *xr = xq + static_cast<size_t>(r) * bpr * 36;
    float acc = 0.0f;
    for (int qb = lane; qb < bpr; qb += 64) acc += block_dot_q8_1<T>(row, qb, xr + static_cast<size_t>(qb) * 36);
    acc = wave_sum(acc);
    if (lane == 0) y[static_cast<size_t>(r) * out_dim + o] = acc;
}

}  // namespace

hipError_t quantize_q8_1(const float *x, uint8_t *xq, int in_dim, int m, bool raw_sum, hipStream_t s) {
    const int bpr = (in_dim + 31) / 32;
    const int64_t nblk = static_cast<int64_t>(m) * bpr;
    if (nblk == 0) return hipSuccess;
    hipLaunchKernelGGL(quantize_q8_1_kernel, dim3(static_cast<unsigned>(plan::quantize_groups(nblk))), dim3(256), 0, s, x, xq,
                       in_dim, nblk, bpr, raw_sum ? 1 : 0);
    return hipGetLastError();
}

hipError_t matmul_q8_1(int type, const uint8_t *w, size_t rb, const uint8_t *xq, float *y, int out_dim,
                       int in_dim, int m, hipStream_t s) {
    const int64_t waves = static_cast<int64_t>(m) * out_dim;
    if (waves == 0) return hipSuccess;
    if (type == T_Q4_K && q4k_gemm_ok(w, rb, xq, in_dim)) return q4k_gemm_q8_1(w, rb, xq, y, out_dim, in_dim, m, s);
    if (type == T_Q4_0 || type == T_Q5_0 || type == T_Q8_0) {
        const plan::Q81 route = plan::q8_1_route(type, out_dim, in_dim, m, qblk_gemm_ok(type, w, rb, xq, in_dim),
                                                 (reinterpret_cast<uintptr_t>(xq) & 3u) == 0, cu_count());
        if (route == plan::Q81::kGemm) return gemm_q8_1(type, w, rb, xq, y, out_dim, in_dim, m, s);
    }
    if (qblk_gemm_ok(type, w, rb, xq, in_dim)) return qblk_gemm_q8_1(type, w, rb, xq, y, out_dim, in_dim, m, s);
    const dim3 grid(static_cast<unsigned>((waves + 3) / 4));
    switch (type) {
        case T_Q4_0: hipLaunchKernelGGL((matmul_q8_1_kernel<T_Q4_0>), grid, dim3(256), 0, s, w, rb, xq, y, out_dim, in_dim, m); break;
        case T_Q5_0: hipLaunchKernelGGL((matmul_q8_1_kernel<T_Q5_0>), grid, dim3(256), 0, s, w, rb, xq, y, out_dim, in_dim, m); break;
        case T_Q8_0: hipLaunchKernelGGL((matmul_q8_1_kernel<T_Q8_0>), grid, dim3(256), 0, s, w, rb, xq, y, out_dim, in_dim, m); break;
        case T_Q4_K: hipLaunchKernelGGL((matmul_q8_1_kernel<T_Q4_K>), grid, dim3(256), 0, s, w, rb, xq, y, out_dim, in_dim, m); break;
        case T_Q6_K: hipLaunchKernelGGL((matmul_q8_1_kernel<T_Q6_K>), grid, dim3(256), 0, s, w, rb, xq, y, out_dim, in_dim, m); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace qlin
