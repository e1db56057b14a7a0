// qlin_embed_mla.hip -- the remaining quantized-weight consumers of the DeepSeek layer, gfx950:
// the quantized embedding lookup and the three MLA latent-absorption products over kv_b.
//
//   embedding  out[t, k] = w(ids[t], k)                  (kernel.cu:2678-2693, quant_embedding_kernel)
//   q_nope     q_abs[h, l] = sum_{d < qk_nope} w(r_h + d, l) * q[h, d]        (kernel.cu:3018-3045)
//   xsum_delta delta[h, b] = sum_{d < qk_nope} q[h, d] * (-dmin * m)(r_h + d, b)  (Q4_K, 3052-3075)
//   v          attn[h, v] = sum_k w(r_h + qk_nope + v, k) * latent[h, k]
//                           (+ for Q4_K: sum_b (-dmin * m)(row, b) * xsum_delta[h, b])   (3417-3453)
// with r_h = h * (qk_nope + v_head) the first kv_b row of head h, q rows of qk_nope + qk_rope, and
// w(row, k) the canonical dequantized element.  These are small (DeepSeek-V2-Lite: 16 heads, kv_b
// [4096, 512]) and latency-bound.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_values8.hpp"

namespace qlin {
namespace {

template <int T>
__global__ __launch_bounds__(256) void embedding_kernel(const int *__restrict__ ids, float *__restrict__ out,
                                                        const uint8_t *__restrict__ table, size_t rb, int hidden) {
    constexpr int BE = Block<T>::elems, BB = Block<T>::bytes;
    const int t = blockIdx.x;
    const uint8_t *row = table + static_cast<size_t>(ids[t]) * rb;
    float *o = out + static_cast<size_t>(t) * hidden;
    for (int k = blockIdx.y * 256 + threadIdx.x; k < hidden; k += gridDim.y * 256)
        o[k] = block_value<T>(row + static_cast<size_t>(k / BE) * BB, k % BE);
}

// The three absorptions are small (DeepSeek-V2-Lite: 16 heads, kv_b [4096, 512], 1.2 MB) and bound by
// latency, so each spreads its rows over enough threads that every byte is requested in one or two
// rounds.  With one thread per output and the rows in turn (128 dependent rounds of byte loads) q_nope
// took 64 us and xsum_delta, one workgroup in all, 77 us; v, a wave per output with one element per
// lane and round, 9.6 us.

constexpr int kQCols = 64, kQThreads = 1024;

// A workgroup per (head, 64 latent columns): thread (cg, ds) takes columns 8cg .. 8cg+7 of the head's
// rows ds, ds + 128, ...; the rows' sums meet by lane shuffles, then in LDS in wave order.
template <int T>
__global__ __launch_bounds__(kQThreads) void absorb_q_nope_kernel(const float *__restrict__ q,
                                                                  const uint8_t *__restrict__ w, size_t rb,
                                                                  float *__restrict__ q_abs, int qk_nope, int qk_rope,
                                                                  int v_head, int kv_lora, int tiles) {
    __shared__ float part[kQThreads / 64][kQCols];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x / tiles, l0 = (blockIdx.x - h * tiles) * kQCols;
    const int cg = tid & 7, ds = tid >> 3, k0 = l0 + 8 * cg;
    const float *qh = q + static_cast<size_t>(h) * (qk_nope + qk_rope);
    const uint8_t *rows = w + static_cast<size_t>(h) * (qk_nope + v_head) * rb;
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    if (k0 < kv_lora) {
        for (int d = ds; d < qk_nope; d += kQThreads / 8) {
            Raw8<T> r;
            raw8<T>(rows + static_cast<size_t>(d) * rb, k0, r);
            const float qd = qh[d];
            float v[8];
            values8<T>(r, k0, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = fmaf(v[i], qd, acc[i]);
        }
    }
#pragma unroll
    for (int off = 8; off < 64; off <<= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += __shfl_xor(acc[i], off, 64);
    if (lane < 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) part[wave][8 * cg + i] = acc[i];
    }
    __syncthreads();
    if (tid < kQCols && l0 + tid < kv_lora) {
        float v = 0.0f;
#pragma unroll
        for (int u = 0; u < kQThreads / 64; ++u) v += part[u][tid];
        q_abs[static_cast<size_t>(h) * kv_lora + l0 + tid] = v;
    }
}

// -dmin * m of sub-block j from a Q4_K super-block's first 16 bytes (the min term of every element of
// that 32-block)
__device__ __forceinline__ float q4k_min_coeff(const u32x4 &hdr, int j) {
    int sc, m;
    q4k_scale_min(j, hdr.y, hdr.z, hdr.w, sc, m);
    return -mul_rn(f16_bits_to_f32(hdr.x >> 16), static_cast<float>(m));
}

constexpr int kDThreads = 128;

// A workgroup per (head, super-block): a thread per row, the super-block's 8 sums over the rows by
// wave sums and LDS.
__global__ __launch_bounds__(kDThreads) void absorb_xsum_delta_kernel(const float *__restrict__ q,
                                                                      const uint8_t *__restrict__ w, size_t rb,
                                                                      float *__restrict__ delta, int qk_nope,
                                                                      int qk_rope, int v_head, int nsb) {
    __shared__ float part[kDThreads / 64][8];
    const int tid = threadIdx.x, h = blockIdx.x / nsb, s = blockIdx.x - h * nsb;
    const float *qh = q + static_cast<size_t>(h) * (qk_nope + qk_rope);
    const uint8_t *rows = w + static_cast<size_t>(h) * (qk_nope + v_head) * rb + static_cast<size_t>(s) * 144;
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
    for (int d = tid; d < qk_nope; d += kDThreads) {
        const u32x4 hdr = ld16_a2(rows + static_cast<size_t>(d) * rb);
        const float qd = qh[d];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = fmaf(qd, q4k_min_coeff(hdr, j), acc[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = wave_sum(acc[j]);
    if ((tid & 63) == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) part[tid >> 6][j] = acc[j];
    }
    __syncthreads();
    if (tid < 8) delta[static_cast<size_t>(blockIdx.x) * 8 + tid] = part[0][tid] + part[1][tid];
}

// A wave per output row, 8 consecutive elements per lane: one round for kv_lora up to 512.
template <int T>
__global__ __launch_bounds__(256) void absorb_v_kernel(const uint8_t *__restrict__ w, size_t rb,
                                                       const float *__restrict__ latent,
                                                       const float *__restrict__ delta, float *__restrict__ attn,
                                                       int n_heads, int qk_nope, int v_head, int kv_lora) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n_heads * v_head) return;  // whole waves
    const int h = i / v_head, v = i - h * v_head;
    const uint8_t *row = w + (static_cast<size_t>(h) * (qk_nope + v_head) + qk_nope + v) * rb;
    const float *x = latent + static_cast<size_t>(h) * kv_lora;
    float acc = 0.0f;
    for (int k0 = 8 * lane; k0 < kv_lora; k0 += 512) {
        Raw8<T> r;
        raw8<T>(row, k0, r);
        float xv[8], wv[8];
        __builtin_memcpy(xv, x + k0, sizeof(xv));
        values8<T>(r, k0, wv);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = fmaf(wv[e], xv[e], acc);
        if constexpr (T == T_Q4_K) {
            if ((k0 & 31) == 0) {
                const int b = k0 >> 5;
                acc = fmaf(q4k_min_coeff(r.hdr, b & 7), delta[static_cast<size_t>(h) * (kv_lora / 32) + b], acc);
            }
        }
    }
    acc = wave_sum(acc);
    if (lane == 0) attn[i] = acc;
}

template <template <int> class K, typename... Args>
bool by_type(int type, Args... args) {
    switch (type) {
        case T_Q4_K: K<T_Q4_K>::run(args...); return true;
        case T_Q6_K: K<T_Q6_K>::run(args...); return true;
        case T_Q5_0: K<T_Q5_0>::run(args...); return true;
        case T_Q8_0: K<T_Q8_0>::run(args...); return true;
        default: return false;
    }
}

template <int T> struct Embed {
    static void run(const int *ids, float *out, const uint8_t *table, size_t rb, int hidden, int n, hipStream_t s) {
        const dim3 grid(n, (hidden + 255) / 256 < 8 ? (hidden + 255) / 256 : 8);
        hipLaunchKernelGGL(embedding_kernel<T>, grid, dim3(256), 0, s, ids, out, table, rb, hidden);
    }
};
template <int T> struct QNope {
    static void run(const float *q, const uint8_t *w, size_t rb, float *q_abs, int nh, int qn, int qr, int vh, int kl,
                    hipStream_t s) {
        const int tiles = (kl + kQCols - 1) / kQCols;
        hipLaunchKernelGGL(absorb_q_nope_kernel<T>, dim3(nh * tiles), dim3(kQThreads), 0, s, q, w, rb, q_abs, qn, qr,
                           vh, kl, tiles);
    }
};
template <int T> struct AbsorbV {
    static void run(const uint8_t *w, size_t rb, const float *latent, const float *delta, float *attn, int nh, int qn,
                    int vh, int kl, hipStream_t s) {
        hipLaunchKernelGGL(absorb_v_kernel<T>, dim3((nh * vh + 3) / 4), dim3(256), 0, s, w, rb, latent, delta, attn,
                           nh, qn, vh, kl);
    }
};

}  // namespace

hipError_t quant_embedding(int type, const int *ids, float *out, const uint8_t *table, size_t rb, int hidden,
                           int n, hipStream_t s) {
    if (n == 0 || hidden == 0) return hipSuccess;
    if (!by_type<Embed>(type, ids, out, table, rb, hidden, n, s)) return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t mla_absorb_q_nope(int type, const float *q, const uint8_t *w, size_t rb, float *q_abs, int n_heads,
                             int qk_nope, int qk_rope, int v_head, int kv_lora, hipStream_t s) {
    if (n_heads == 0 || kv_lora == 0) return hipSuccess;
    if (!by_type<QNope>(type, q, w, rb, q_abs, n_heads, qk_nope, qk_rope, v_head, kv_lora, s))
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t mla_absorb_q4_xsum_delta(const float *q, const uint8_t *w, size_t rb, float *delta, int n_heads,
                                    int qk_nope, int qk_rope, int v_head, int kv_lora, hipStream_t s) {
    const int nsb = kv_lora / 256;
    if (n_heads == 0 || nsb == 0) return hipSuccess;
    hipLaunchKernelGGL(absorb_xsum_delta_kernel, dim3(n_heads * nsb), dim3(kDThreads), 0, s, q, w, rb, delta, qk_nope,
                       qk_rope, v_head, nsb);
    return hipGetLastError();
}

hipError_t mla_absorb_v(int type, const uint8_t *w, size_t rb, const float *latent, const float *delta, float *attn,
                        int n_heads, int qk_nope, int v_head, int kv_lora, hipStream_t s) {
    if (n_heads == 0 || v_head == 0) return hipSuccess;
    if (!by_type<AbsorbV>(type, w, rb, latent, delta, attn, n_heads, qk_nope, v_head, kv_lora, s))
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace qlin
