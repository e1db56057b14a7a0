// qlin_dequant.hip -- whole-stream dequantization to f32 or f16, gfx950.
//
// Semantics of the reference's dequantize_{q4k,q80,q50,q6k}_to_f16_kernel
// (AI/codes/local-llm/src/backend/cuda/ops/kernel.cu:954-1063): every element is the canonical
// non-contracted f32 value of its block (qlin_device.hpp), and the f16 output is that value rounded
// to nearest-even (scalar v_cvt_f16_f32 under the default round-to-nearest mode, f16 subnormals
// preserved).  Results are bit-exact
// against any correct evaluation of the formulas.  Q4_0 is added from the ggml format.
//
// Layout: one thread per 8 consecutive elements (one block, one scale): its 8 or so quant bytes in one
// request, its 16 (f16) or 32 (f32) output bytes in one or two, consecutive threads on consecutive
// groups; the block's scale is one request that the threads of a block share.  Bound by the output
// (2 or 4 bytes per 0.56..1.06 bytes in).  One thread per element, each decoding its block's scale for
// itself from byte loads, took 154 us for Q4_K [14336, 4096] to f16 (975 GB/s).
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_values8.hpp"

namespace qlin {
namespace {

template <int T, bool F16>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t *__restrict__ src,
                                                      void *__restrict__ out, int64_t groups) {
    constexpr int BE = Block<T>::elems, BB = Block<T>::bytes, G = BE / 8;  // groups of 8 per block
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < groups; i += stride) {
        const int64_t b = i / G;
        const int k0 = 8 * static_cast<int>(i - b * G);
        Raw8<T> r;
        raw8<T>(src + b * BB, k0, r);
        float v[8];
        values8<T>(r, k0, v);
        if constexpr (F16) {
            uint32_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = f32_to_f16_bits(v[2 * e]) | (f32_to_f16_bits(v[2 * e + 1]) << 16);
            __builtin_memcpy(__builtin_assume_aligned(static_cast<uint16_t *>(out) + 8 * i, 2), h, sizeof(h));
        } else {
            __builtin_memcpy(__builtin_assume_aligned(static_cast<float *>(out) + 8 * i, 4), v, sizeof(v));
        }
    }
}

template <int T>
hipError_t launch_t(const uint8_t *src, void *out, int64_t n, bool f16, hipStream_t s) {
    const int64_t groups = n / 8, want = (groups + 255) / 256;  // (n is whole blocks)
    const int blocks = static_cast<int>(want < (1 << 20) ? want : (1 << 20));
    if (f16)
        hipLaunchKernelGGL((dequant_kernel<T, true>), dim3(blocks), dim3(256), 0, s, src, out, groups);
    else
        hipLaunchKernelGGL((dequant_kernel<T, false>), dim3(blocks), dim3(256), 0, s, src, out, groups);
    return hipGetLastError();
}

}  // namespace

hipError_t dequant(int type, const uint8_t *src, void *out, int64_t n, bool to_f16, hipStream_t s) {
    if (n == 0) return hipSuccess;
    switch (type) {
        case T_Q4_0: return launch_t<T_Q4_0>(src, out, n, to_f16, s);
        case T_Q5_0: return launch_t<T_Q5_0>(src, out, n, to_f16, s);
        case T_Q8_0: return launch_t<T_Q8_0>(src, out, n, to_f16, s);
        case T_Q4_K: return launch_t<T_Q4_K>(src, out, n, to_f16, s);
        case T_Q6_K: return launch_t<T_Q6_K>(src, out, n, to_f16, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qlin
