// qlin_mla_latent.hip -- the MLA decode kernels over the Q8_1 latent cache, gfx950.
//
// The latent cache holds one Q8_1 row (kernel.cu:1679-1720 blocks, 36 bytes per 32 values) per
// position: the RMS-normed latent of kv_a.  With pos = *d_pos (device memory, as the reference's
// device-pos launchers read it) and L(t, k) = d * q the dequantized latent element k of row t:
//
//   store      cache[pos] = Q8_1(kv_cache[pos, 0 .. kv_lora))             (kernel.cu:2945-2978)
//   scores     s[h, t] = scale * ( sum_k q_abs[h, k] L(t, k) + sum_r q_rope[h, r] k_rope(t, r)
//                        + sum_b delta[h, b] (S(t, b) - sum_l L(t, 32b + l)) ),  t <= pos
//                                                                            (kernel.cu:3157-3196)
//   context    p[h, t] = exp(s[h, t] - max_t s[h]) / (sum_t exp(...) + 1e-9);
//              latent[h, k] = sum_t p[h, t] L(t, k);  delta[h, b] = sum_t p[h, t] (S(t, b) - ...)
//                                                                            (kernel.cu:3198-3257)
//   attend     scores, softmax (fast exp, no 1e-9) and context in one launch   (kernel.cu:3078-3155)
//   project_v  kv_b_cache[pos, v row r of head h] = W_kv_b[r] . cache[pos] with the Q8_1 block-dot
//              semantics of quant_matmul_q8_1                               (kernel.cu:3259-3361)
//   context_v  attn[h, v] = sum_t p[h, t] kv_b_cache[t, v row of head h]   (kernel.cu:3368-3415)
//
// S(t, b) is the block's stored f16 sum and the inner sum is the block's dequantized values added in
// order.  The products run on v_mfma_f32_16x16x4_f32 where heads meet positions (scores: heads x
// positions; context: heads x latent columns over positions); operands are the reference's f32 values
// and only the summation order differs.
#include "qlin_device.hpp"
#include "qlin_internal.hpp"
#include "qlin_mfma.hpp"
#include "qlin_q8_1.hpp"

namespace qlin {
namespace {

// The block sum correction S(t, b) - sum_l L(t, 32b + l).  The sum in order is d times the integer sum of
// the q's exactly: d has 11 significant bits and |sum q| < 2^12, so every partial sum is exact in f32.
__device__ __forceinline__ float sum_correction(uint32_t ds, int qsum) {
    return __fsub_rn(f16_bits_to_f32(ds >> 16), __fmul_rn(f16_bits_to_f32(ds & 0xffffu), static_cast<float>(qsum)));
}
__device__ __forceinline__ int sum4(uint32_t q, int acc) {
    return __builtin_amdgcn_sdot4(static_cast<int>(q), 0x01010101, acc, false);
}
// the sum over the lane's group of 4, or of 8, lanes
template <int CTRL>
__device__ __forceinline__ int dpp_add(int v) {
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ int sum_of_4(int v) { return dpp_add<0x4e>(dpp_add<0xb1>(v)); }  // quad_perm
__device__ __forceinline__ int sum_of_8(int v) { return dpp_add<0x141>(sum_of_4(v)); }      // row_half_mirror
// 0xff in the bytes below n of a dword (n <= 0: none, n >= 4: all)
__device__ __forceinline__ uint32_t byte_mask(int n) { return n >= 4 ? ~0u : (n <= 0 ? 0u : (1u << (8 * n)) - 1u); }
// S(t, b) - sum of the block at blk (l over the kv_lora - 32b valid values).
__device__ __forceinline__ float block_sum_delta(const uint8_t *blk, int valid) {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(blk);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = sum4(w[1 + i] & byte_mask(valid - 4 * i), sum);
    return sum_correction(w[0], sum);
}

__global__ __launch_bounds__(256) void store_latent_kernel(const float *__restrict__ kv_cache, uint8_t *cache,
                                                           int kv_lora, int qk_rope, size_t row_bytes, int nblk,
                                                           const int *__restrict__ d_pos) {
    const int i = blockIdx.x * 256 + threadIdx.x, b = i >> 3, j = i & 7;  // 8 lanes per block
    const int pos = *d_pos;
    if (b >= nblk || pos < 0) return;  // (whole groups of 8 lanes)
    const float *src = kv_cache + static_cast<size_t>(pos) * (kv_lora + qk_rope);
    quantize_block_q8_1_lanes(src, 32 * b + 4 * j, kv_lora, j,
                              reinterpret_cast<uint32_t *>(cache + static_cast<size_t>(pos) * row_bytes + b * 36), false);
}

struct ScoreArgs {
    const float *q_abs, *q;
    const uint8_t *cache;
    size_t crb;
    const float *delta, *kv_cache;
    float *scores;
    int n_heads, qk_nope, qk_rope, kv_lora, max_seq;
    const int *d_pos;
    float scale;
};

// 8 floats at p, those at index `valid` and past it 0 and not read
__device__ __forceinline__ void load8(float (&v)[8], const float *p, int valid) {
    if (valid >= 8) {
        __builtin_memcpy(v, p, sizeof(v));
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = e < valid ? p[e] : 0.0f;
    }
}

constexpr int kSWaves = 9, kSThreads = kSWaves * 64;

// A workgroup per (16 positions, 16 heads): lane l supplies head l % 16 (A) and position l % 16 (B); the
// 8 MFMAs of a 32-value block take its values 8g .. 8g+7 in k-slot g = l / 16, a ninth its sum
// correction.  The waves take the latent blocks and the rope chunks of 32 in turn (DeepSeek-V2-Lite: 16
// blocks and 2 chunks, two rounds of loads) and their sums meet in LDS in wave order.  Bound by the
// rounds' latency: with one wave per tile walking the 18 in turn the launch took 33 us at position 1500.
__global__ __launch_bounds__(kSThreads) void scores_kernel(const ScoreArgs a) {
    __shared__ f32x4 part[kSWaves][64];
    const int pos = min(*a.d_pos, a.max_seq - 1);
    const int t0 = blockIdx.x * 16;
    if (t0 > pos) return;  // uniform (also pos < 0)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    const int h0 = blockIdx.y * 16;
    const int hn = min(h0 + n, a.n_heads - 1), tn = min(t0 + n, pos);
    const int nb = (a.kv_lora + 31) / 32, nr = (a.qk_rope + 31) / 32;
    const float *qa = a.q_abs + static_cast<size_t>(hn) * a.kv_lora;
    const float *dl = a.delta + static_cast<size_t>(hn) * nb;
    const uint8_t *row = a.cache + static_cast<size_t>(tn) * a.crb;
    const float *qr = a.q + static_cast<size_t>(hn) * (a.qk_nope + a.qk_rope) + a.qk_nope;
    const float *kr = a.kv_cache + static_cast<size_t>(tn) * (a.kv_lora + a.qk_rope) + a.kv_lora;

    f32x4 D = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = wave; i < nb + nr; i += kSWaves) {  // uniform
        float av[8], bv[8];
        if (i < nb) {
            const uint8_t *blk = row + static_cast<size_t>(i) * 36;
            const uint32_t ds = *reinterpret_cast<const uint32_t *>(blk);
            const uint2 q = ld8_a4(blk + 4 + 8 * g);
            const int k0 = i * 32 + 8 * g, valid = a.kv_lora - k0;
            const float dh = dl[i];
            load8(av, qa + k0, valid);
            const uint32_t w[2] = {q.x & byte_mask(valid), q.y & byte_mask(valid - 4)};
            const float d = f16_bits_to_f32(ds & 0xffffu);
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = __fmul_rn(d, static_cast<float>(static_cast<int8_t>(w[e >> 2] >> (8 * (e & 3)))));
            int sum = sum4(w[1], sum4(w[0], 0));
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
#pragma unroll
            for (int e = 0; e < 8; ++e) D = mfma_f32(av[e], bv[e], D);
            D = mfma_f32(g == 0 ? dh : 0.0f, g == 0 ? sum_correction(ds, sum) : 0.0f, D);
        } else {
            const int r0 = (i - nb) * 32 + 8 * g;
            load8(av, qr + r0, a.qk_rope - r0);
            load8(bv, kr + r0, a.qk_rope - r0);
#pragma unroll
            for (int e = 0; e < 8; ++e) D = mfma_f32(av[e], bv[e], D);
        }
    }
    part[wave][lane] = D;
    __syncthreads();
    if (tid >= 256) return;
    // thread (head hl, position tl) of the tile; lane (position, g) of D holds heads 4g .. 4g+3
    const int hl = tid >> 4, tl = tid & 15, h = h0 + hl, t = t0 + tl;
    if (h >= a.n_heads || t > pos) return;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kSWaves; ++w) v += part[w][(hl >> 2) * 16 + tl][hl & 3];
    a.scores[static_cast<size_t>(h) * a.max_seq + t] = __fmul_rn(v, a.scale);
}

constexpr int kCWaves = 16, kCThreads = kCWaves * 64;

struct ContextArgs {
    const float *scores;
    const uint8_t *cache;
    size_t crb;
    float *delta_out, *latent_out;
    int n_heads, kv_lora, max_seq;
    const int *d_pos;
};

// A workgroup per (a quarter of the columns of 2 latent blocks, 16 heads).  Each wave first takes one
// head's largest score; then the waves take 16 positions at a time in turn: lane (n, g) reads dword
// n % 8 of block n / 8 at positions 4g .. 4g+3 and its head n's scores there, so that MFMA i adds
// position 4g + i in k-slot g with byte c of the dwords as its 16 columns (column 4 (n % 8) + c of
// block n / 8, c the workgroup's); the workgroup of byte 3 takes a second MFMA per position for the
// blocks' sum corrections.  exp(s - max) goes in unnormalized and its sums divide the result.  Bound by
// the latency of its rounds and the exponentials, which every workgroup takes for itself: with a byte
// and a score per lane, position and column tile, two passes of statistics and the corrections' bytes
// summed in turn, the launch took 166 us at position 1500.
__global__ __launch_bounds__(kCThreads) void context_kernel(const ContextArgs a) {
    static_assert(kCWaves == 16, "one head per wave in the maxima");
    constexpr int kHalf = kCWaves / 2;
    __shared__ float s_max[16], s_den[kCWaves][16];
    __shared__ f32x4 part[kHalf][2][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    const int pos = min(*a.d_pos, a.max_seq - 1);
    const int h0 = blockIdx.y * 16;
    const int nb = (a.kv_lora + 31) / 32;
    const int bc = min(2 * static_cast<int>(blockIdx.x >> 2) + (n >> 3), nb - 1);
    const int c0 = blockIdx.x & 3;
    const bool corr = c0 == 3;  // one of the pair's workgroups also sums the corrections
    const uint32_t qmask = byte_mask(a.kv_lora - 32 * bc - 4 * (n & 7));

    // 16 positions a step; two steps' words requested ahead
    struct Step {
        uint32_t ds[4], q[4];
        float s[4];
    };
    const float *sh = a.scores + static_cast<size_t>(min(h0 + n, a.n_heads - 1)) * a.max_seq;
    const uint8_t *base = a.cache + static_cast<size_t>(bc) * 36;
    const uint32_t crb = static_cast<uint32_t>(a.crb);  // (15 rows stay below 4 GiB)
    auto load = [&](Step &st, int t0) {  // past the end: the last position again
        t0 = min(t0, pos);  // uniform
        const uint8_t *row = base + static_cast<size_t>(t0) * a.crb;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t dt = min(4 * g + i, pos - t0);
            const uint8_t *blk = row + dt * crb;
            st.ds[i] = *reinterpret_cast<const uint32_t *>(blk);
            st.q[i] = *reinterpret_cast<const uint32_t *>(blk + 4 + 4 * (n & 7));
            st.s[i] = sh[t0 + dt];
        }
    };
    Step s0{}, s1{};
    int t0 = 16 * wave;
    constexpr int kStride = 16 * kCWaves;
    if (t0 <= pos) {
        load(s0, t0);
        load(s1, t0 + kStride);
    }
    {  // heads past n_heads repeat the last one (their outputs are not stored)
        constexpr int U = 32;
        const float *shw = a.scores + static_cast<size_t>(min(h0 + wave, a.n_heads - 1)) * a.max_seq;
        float m = -INFINITY;
        for (int t = lane; t <= pos; t += 64 * U) {
            float v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = shw[min(t + 64 * u, pos)];
#pragma unroll
            for (int u = 0; u < U; ++u) m = fmaxf(m, v[u]);
        }
        m = wave_max(m);
        if (lane == 0) s_max[wave] = m;
    }
    __syncthreads();
    const float mx = s_max[n];

    f32x4 D[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) D[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
    auto add = [&](const Step &cur) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = t0 + 4 * g + i <= pos;
            const float e = in ? expf(cur.s[i] - mx) : 0.0f;
            den += e;
            const uint32_t q = cur.q[i] & qmask;
            const float d = f16_bits_to_f32(cur.ds[i] & 0xffffu);
            D[0] = mfma_f32(e, __fmul_rn(d, static_cast<float>(static_cast<int8_t>(q >> (8 * c0)))), D[0]);
            if (corr) D[1] = mfma_f32(e, sum_correction(cur.ds[i], sum_of_8(sum4(q, 0))), D[1]);  // uniform
        }
    };
    for (; t0 <= pos; t0 += kStride) {  // uniform
        Step s2;
        load(s2, t0 + 2 * kStride);
        add(s0);
        s0 = s1;
        s1 = s2;
    }
    den += __shfl_xor(den, 16, 64);
    den += __shfl_xor(den, 32, 64);
    if (lane < 16) s_den[wave][n] = den;
    if (wave >= kHalf) {
#pragma unroll
        for (int c = 0; c < 2; ++c) part[wave - kHalf][c][lane] = D[c];
    }
    __syncthreads();
    if (wave < kHalf) {
#pragma unroll
        for (int c = 0; c < 2; ++c) part[wave][c][lane] += D[c];
    }
    __syncthreads();
    // thread (head hl, column lane cl): lane (column lane, g) of D holds heads 4g .. 4g+3
    const int hl = tid >> 4, cl = tid & 15, h = h0 + hl;
    if (hl >= 16 || h >= a.n_heads) return;
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < kCWaves; ++w) s += s_den[w][hl];
    s += 1e-9f;
    const int cb = 2 * (blockIdx.x >> 2) + (cl >> 3), k = 32 * cb + 4 * (cl & 7) + c0;
    const int src = (hl >> 2) * 16 + cl;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kHalf; ++w) v += part[w][0][src][hl & 3];
    if (k < a.kv_lora) a.latent_out[static_cast<size_t>(h) * a.kv_lora + k] = v / s;
    if (corr && (cl & 7) == 0 && cb < nb) {
        float dv = 0.0f;
#pragma unroll
        for (int w = 0; w < kHalf; ++w) dv += part[w][1][src][hl & 3];
        a.delta_out[static_cast<size_t>(h) * nb + cb] = dv / s;
    }
}

// One wave per (head, v row): kv_b row h * (qk_nope + v_head) + qk_nope + v against the latent row.
template <int T>
__global__ __launch_bounds__(256) void project_v_kernel(const uint8_t *__restrict__ w, size_t rb,
                                                        const uint8_t *__restrict__ cache, size_t crb,
                                                        float *__restrict__ kvb_cache, int n_heads, int qk_nope,
                                                        int v_head, int kv_lora, const int *__restrict__ d_pos) {
    const int wv = static_cast<int>((blockIdx.x * 256 + threadIdx.x) >> 6), lane = threadIdx.x & 63;
    const int pos = *d_pos;
    if (wv >= n_heads * v_head || pos < 0) return;  // whole waves
    const int h = wv / v_head, v = wv - h * v_head;
    const int r = h * (qk_nope + v_head) + qk_nope + v;
    const uint8_t *wr = w + static_cast<size_t>(r) * rb;
    const uint8_t *xr = cache + static_cast<size_t>(pos) * crb;
    float acc = 0.0f;
    for (int qb = lane; qb < kv_lora / 32; qb += 64) acc += block_dot_q8_1<T>(wr, qb, xr + static_cast<size_t>(qb) * 36);
    acc = wave_sum(acc);
    if (lane == 0) kvb_cache[static_cast<size_t>(pos) * n_heads * (qk_nope + v_head) + r] = acc;
}

constexpr int kVMax = 4;  // v_head <= 64 * kVMax

// A workgroup per head: wave w takes positions w, w + 16, ...; lane l columns l, l + 64, ...
__global__ __launch_bounds__(kCThreads) void context_v_kernel(const float *__restrict__ scores,
                                                              const float *__restrict__ kvb_cache,
                                                              float *__restrict__ attn, int n_heads, int qk_nope,
                                                              int v_head, const int *__restrict__ d_pos,
                                                              int max_seq) {
    __shared__ float s_part[2][kCWaves];
    __shared__ float s_acc[kCWaves][64 * kVMax];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x;
    const int pos = min(*d_pos, max_seq - 1);
    const float *sh = scores + static_cast<size_t>(h) * max_seq;
    // statistics over the whole workgroup: per-wave max, then per-wave sums of exp(s - max)
    float m = -INFINITY;
    for (int t = tid; t <= pos; t += kCThreads) m = fmaxf(m, sh[t]);
    m = wave_max(m);
    if (lane == 0) s_part[0][wave] = m;
    __syncthreads();
    m = -INFINITY;
    for (int w = 0; w < kCWaves; ++w) m = fmaxf(m, s_part[0][w]);
    float s = 0.0f;
    for (int t = tid; t <= pos; t += kCThreads) s += expf(sh[t] - m);
    s = wave_sum(s);
    if (lane == 0) s_part[1][wave] = s;
    __syncthreads();
    s = 0.0f;
    for (int w = 0; w < kCWaves; ++w) s += s_part[1][w];
    const float den = s + 1e-9f;

    const int stride = n_heads * (qk_nope + v_head);
    const float *vbase = kvb_cache + static_cast<size_t>(h) * (qk_nope + v_head) + qk_nope;
    float acc[kVMax] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = wave; t <= pos; t += kCWaves) {
        const float p = expf(sh[t] - m) / den;
        const float *vr = vbase + static_cast<size_t>(t) * stride;
#pragma unroll
        for (int c = 0; c < kVMax; ++c)
            if (lane + 64 * c < v_head) acc[c] = fmaf(p, vr[lane + 64 * c], acc[c]);
    }
#pragma unroll
    for (int c = 0; c < kVMax; ++c) s_acc[wave][lane + 64 * c] = acc[c];
    __syncthreads();
    for (int v = tid; v < v_head; v += kCThreads) {
        float o = 0.0f;
        for (int w = 0; w < kCWaves; ++w) o += s_acc[w][v];
        attn[static_cast<size_t>(h) * v_head + v] = o;
    }
}

constexpr int kAMaxSeq = 32768;  // attend: scores of every position in LDS
constexpr size_t kMaxLds = 160 * 1024;

// Scores, softmax and context of one head in one workgroup (the fused form): the scores of all
// positions stay in LDS.  exp is the fast __expf and the denominator has no 1e-9 term, as in
// kernel.cu:3078-3155.
__global__ __launch_bounds__(kCThreads) void attend_kernel(const ScoreArgs a, float *delta_out, float *latent_out) {
    extern __shared__ float s_sc[];  // [max_seq] scores, then q_abs [kv_lora], q_rope [qk_rope], delta [nb]
    __shared__ float s_red[2][kCWaves];
    __shared__ float s_out[kCWaves][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x;
    const int pos = min(*a.d_pos, a.max_seq - 1);
    const int nb = (a.kv_lora + 31) / 32;
    float *s_qa = s_sc + a.max_seq, *s_qr = s_qa + a.kv_lora, *s_dl = s_qr + a.qk_rope;
    for (int i = tid; i < a.kv_lora; i += kCThreads) s_qa[i] = a.q_abs[static_cast<size_t>(h) * a.kv_lora + i];
    for (int i = tid; i < a.qk_rope; i += kCThreads)
        s_qr[i] = a.q[static_cast<size_t>(h) * (a.qk_nope + a.qk_rope) + a.qk_nope + i];
    for (int i = tid; i < nb; i += kCThreads) s_dl[i] = a.delta[static_cast<size_t>(h) * nb + i];
    __syncthreads();

    // scores: a wave per position, lanes over the latent values, the rope pair and the block sums
    float m = -INFINITY;
    for (int t = wave; t <= pos; t += kCWaves) {
        const uint8_t *row = a.cache + static_cast<size_t>(t) * a.crb;
        const float *kr = a.kv_cache + static_cast<size_t>(t) * (a.kv_lora + a.qk_rope) + a.kv_lora;
        float dot = 0.0f;
        for (int k = lane; k < a.kv_lora; k += 64) {
            const uint8_t *blk = row + static_cast<size_t>(k >> 5) * 36;
            dot = fmaf(s_qa[k], __fmul_rn(f16_bits_to_f32(ld_u16(blk)),
                                          static_cast<float>(reinterpret_cast<const int8_t *>(blk + 4)[k & 31])), dot);
        }
        for (int r = lane; r < a.qk_rope; r += 64) dot = fmaf(s_qr[r], kr[r], dot);
        for (int b = lane; b < nb; b += 64)
            dot = fmaf(s_dl[b], block_sum_delta(row + static_cast<size_t>(b) * 36, a.kv_lora - 32 * b), dot);
        dot = wave_sum(dot);
        const float sc = __fmul_rn(dot, a.scale);
        if (lane == 0) s_sc[t] = sc;
        m = fmaxf(m, sc);
    }
    if (lane == 0) s_red[0][wave] = m;
    __syncthreads();
    m = -INFINITY;
    for (int w = 0; w < kCWaves; ++w) m = fmaxf(m, s_red[0][w]);
    float den = 0.0f;
    for (int t = tid; t <= pos; t += kCThreads) {
        const float e = __expf(s_sc[t] - m);
        s_sc[t] = e;
        den += e;
    }
    den = wave_sum(den);
    if (lane == 0) s_red[1][wave] = den;
    __syncthreads();
    den = 0.0f;
    for (int w = 0; w < kCWaves; ++w) den += s_red[1][w];

    // context: a column per lane, the positions split over the waves, wave partials added in order
    const int ncol = a.kv_lora + nb;
    for (int c0 = 0; c0 < ncol; c0 += 64) {
        const int c = c0 + lane;
        float acc = 0.0f;
        if (c < ncol)
            for (int t = wave; t <= pos; t += kCWaves) {
                const uint8_t *row = a.cache + static_cast<size_t>(t) * a.crb;
                float v;
                if (c < a.kv_lora) {
                    const uint8_t *blk = row + static_cast<size_t>(c >> 5) * 36;
                    v = __fmul_rn(f16_bits_to_f32(ld_u16(blk)),
                                  static_cast<float>(reinterpret_cast<const int8_t *>(blk + 4)[c & 31]));
                } else {
                    const int b = c - a.kv_lora;
                    v = block_sum_delta(row + static_cast<size_t>(b) * 36, a.kv_lora - 32 * b);
                }
                acc = fmaf(s_sc[t] / den, v, acc);
            }
        s_out[wave][lane] = acc;
        __syncthreads();
        if (tid < 64 && c < ncol) {
            float o = 0.0f;
            for (int w = 0; w < kCWaves; ++w) o += s_out[w][tid];
            if (c < a.kv_lora) latent_out[static_cast<size_t>(h) * a.kv_lora + c] = o;
            else delta_out[static_cast<size_t>(h) * nb + (c - a.kv_lora)] = o;
        }
        __syncthreads();
    }
}

// The same for kv_lora a multiple of 32 up to 512 and qk_rope a multiple of 4 up to 64: a wave scores four
// positions at a time, 16 lanes each, lane b of a position taking latent block b (its 32 q_abs values
// stay in registers) and rope values 4b .. 4b+3; for the context a lane takes 8 columns (the quarter
// of a block) and the waves take the positions in turn, eight requested at once.  Bound by the 16 waves'
// arithmetic on one CU per head.
constexpr int kFBlocks = 16, kFCols = kFBlocks * 33;  // latent columns and sum corrections, at most

__global__ __launch_bounds__(kCThreads) void attend_blocks_kernel(const ScoreArgs a, float *delta_out,
                                                                  float *latent_out) {
    extern __shared__ float s_sc[];  // [max_seq] scores; afterwards the waves' sums [kCWaves][kFCols]
    __shared__ float s_red[2][kCWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x;
    const int pos = min(*a.d_pos, a.max_seq - 1);
    const int nb = a.kv_lora / 32;

    float m = -INFINITY;
    {
        const int p = lane >> 4, b = lane & 15;
        const bool live = b < nb, rlive = 4 * b < a.qk_rope;
        float qa[32], qr[4] = {0.0f, 0.0f, 0.0f, 0.0f}, dl = 0.0f;
#pragma unroll
        for (int e = 0; e < 32; ++e) qa[e] = 0.0f;
        if (live) {
            __builtin_memcpy(qa, a.q_abs + static_cast<size_t>(h) * a.kv_lora + 32 * b, sizeof(qa));
            dl = a.delta[static_cast<size_t>(h) * nb + b];
        }
        if (rlive)
            __builtin_memcpy(qr, a.q + static_cast<size_t>(h) * (a.qk_nope + a.qk_rope) + a.qk_nope + 4 * b, sizeof(qr));
        struct Row {
            uint32_t w[9];
            float r[4];
        };
        auto load = [&](Row &x, int t) {
            t = min(t, pos);
            if (live) {
                const uint32_t *blk = reinterpret_cast<const uint32_t *>(a.cache + static_cast<size_t>(t) * a.crb + 36 * b);
#pragma unroll
                for (int i = 0; i < 9; ++i) x.w[i] = blk[i];
            }
            if (rlive)
                __builtin_memcpy(x.r, a.kv_cache + static_cast<size_t>(t) * (a.kv_lora + a.qk_rope) + a.kv_lora + 4 * b,
                                 sizeof(x.r));
        };
        Row cur{}, nxt{};
        int t = 4 * wave + p;
        if (4 * wave <= pos) load(cur, t);
        for (int t0 = 4 * wave; t0 <= pos; t0 += 4 * kCWaves, t += 4 * kCWaves) {  // uniform
            load(nxt, t + 4 * kCWaves);
            const float d = f16_bits_to_f32(cur.w[0] & 0xffffu);
            float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            int sum = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sum = sum4(cur.w[1 + i], sum);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    dot[c] = fmaf(qa[4 * i + c],
                                  __fmul_rn(d, static_cast<float>(static_cast<int8_t>(cur.w[1 + i] >> (8 * c)))), dot[c]);
            }
            float v = (dot[0] + dot[1]) + (dot[2] + dot[3]);
#pragma unroll
            for (int c = 0; c < 4; ++c) v = fmaf(qr[c], cur.r[c], v);
            if (live) v = fmaf(dl, sum_correction(cur.w[0], sum), v);
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            const float sc = __fmul_rn(v, a.scale);
            if (t <= pos) {
                if (b == 0) s_sc[t] = sc;
                m = fmaxf(m, sc);
            }
            cur = nxt;
        }
        m = wave_max(m);
    }
    if (lane == 0) s_red[0][wave] = m;
    __syncthreads();
    m = -INFINITY;
#pragma unroll
    for (int w = 0; w < kCWaves; ++w) m = fmaxf(m, s_red[0][w]);
    float den = 0.0f;
    for (int t = tid; t <= pos; t += kCThreads) {
        const float e = __expf(s_sc[t] - m);
        s_sc[t] = e;
        den += e;
    }
    den = wave_sum(den);
    if (lane == 0) s_red[1][wave] = den;
    __syncthreads();
    den = 0.0f;
#pragma unroll
    for (int w = 0; w < kCWaves; ++w) den += s_red[1][w];

    // context: columns 8 lane .. 8 lane + 7, and the block's correction in the first of its 4 lanes
    float acc[8], dacc = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
    const int b = min(lane >> 2, nb - 1), part8 = 8 * (lane & 3);
    constexpr int U = 8;
    for (int t0 = wave; t0 <= pos; t0 += U * kCWaves) {  // uniform
        uint32_t ds[U];
        uint2 q[U];
        float e[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = t0 + u * kCWaves;
            const uint8_t *blk = a.cache + static_cast<size_t>(min(t, pos)) * a.crb + 36 * b;
            ds[u] = *reinterpret_cast<const uint32_t *>(blk);
            __builtin_memcpy(&q[u], __builtin_assume_aligned(blk + 4 + part8, 4), 8);
            e[u] = t <= pos ? s_sc[t] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t0 + u * kCWaves > pos) break;  // uniform
            const float d = f16_bits_to_f32(ds[u] & 0xffffu);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                acc[c] = fmaf(e[u], __fmul_rn(d, static_cast<float>(static_cast<int8_t>((c < 4 ? q[u].x : q[u].y) >> (8 * (c & 3))))),
                              acc[c]);
            dacc = fmaf(e[u], sum_correction(ds[u], sum_of_4(sum4(q[u].y, sum4(q[u].x, 0)))), dacc);
        }
    }
    __syncthreads();  // (the scores are no longer read: their LDS takes the waves' sums)
    float *mine = s_sc + wave * kFCols;
#pragma unroll
    for (int c = 0; c < 8; ++c) mine[8 * lane + c] = acc[c];
    if ((lane & 3) == 0) mine[32 * kFBlocks + (lane >> 2)] = dacc;
    __syncthreads();
    if (tid >= kFCols) return;
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < kCWaves; ++w) o += s_sc[w * kFCols + tid];
    o = pos < 0 ? 0.0f : o / den;
    if (tid < a.kv_lora) latent_out[static_cast<size_t>(h) * a.kv_lora + tid] = o;
    else if (tid >= 32 * kFBlocks && tid - 32 * kFBlocks < nb) delta_out[static_cast<size_t>(h) * nb + tid - 32 * kFBlocks] = o;
}

// LDS of the block form; the shapes it takes are those of the general form with room for the waves' sums.
size_t attend_blocks_lds(int max_seq) {
    constexpr int sums = kCWaves * kFCols;
    return sizeof(float) * static_cast<size_t>(max_seq > sums ? max_seq : sums);
}
bool attend_blocks_ok(int max_seq, int kv_lora, int qk_rope) {
    return kv_lora % 32 == 0 && kv_lora <= 32 * kFBlocks && qk_rope % 4 == 0 && qk_rope <= 4 * kFBlocks &&
           attend_blocks_lds(max_seq) + sizeof(float) * 2 * kCWaves <= kMaxLds;
}

template <int T> struct ProjectV {
    static void run(const uint8_t *w, size_t rb, const uint8_t *cache, size_t crb, float *kvb, int nh, int qn, int vh,
                    int kl, const int *d_pos, hipStream_t s) {
        hipLaunchKernelGGL(project_v_kernel<T>, dim3((nh * vh + 3) / 4), dim3(256), 0, s, w, rb, cache, crb, kvb, nh,
                           qn, vh, kl, d_pos);
    }
};

}  // namespace

hipError_t mla_store_latent_q8_1(const float *kv_cache, uint8_t *cache, int kv_lora, int qk_rope, size_t row_bytes,
                                 const int *d_pos, hipStream_t s) {
    const int nblk = static_cast<int>(row_bytes / 36);
    if (nblk == 0) return hipSuccess;
    hipLaunchKernelGGL(store_latent_kernel, dim3((nblk + 31) / 32), dim3(256), 0, s, kv_cache, cache, kv_lora, qk_rope,
                       row_bytes, nblk, d_pos);
    return hipGetLastError();
}

hipError_t mla_absorb_scores(const float *q_abs, const float *q, const uint8_t *cache, size_t crb,
                             const float *delta, const float *kv_cache, float *scores, int n_heads, int qk_nope,
                             int qk_rope, int kv_lora, const int *d_pos, int max_seq, float scale, hipStream_t s) {
    if (n_heads == 0 || max_seq == 0) return hipSuccess;
    const ScoreArgs a{q_abs, q, cache, crb, delta, kv_cache, scores, n_heads, qk_nope, qk_rope, kv_lora, max_seq,
                      d_pos, scale};
    hipLaunchKernelGGL(scores_kernel, dim3((max_seq + 15) / 16, (n_heads + 15) / 16), dim3(kSThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t mla_absorb_context(const float *scores, const uint8_t *cache, size_t crb, float *delta_out,
                              float *latent_out, int n_heads, int kv_lora, const int *d_pos, int max_seq,
                              hipStream_t s) {
    if (n_heads == 0 || kv_lora == 0) return hipSuccess;
    const ContextArgs a{scores, cache, crb, delta_out, latent_out, n_heads, kv_lora, max_seq, d_pos};
    const dim3 grid(4 * ((kv_lora + 63) / 64), (n_heads + 15) / 16);
    hipLaunchKernelGGL(context_kernel, grid, dim3(kCThreads), 0, s, a);
    return hipGetLastError();
}

size_t mla_attend_lds(int max_seq, int kv_lora, int qk_rope) {
    return sizeof(float) * (static_cast<size_t>(max_seq) + kv_lora + qk_rope + (kv_lora + 31) / 32);
}

bool mla_attend_ok(int max_seq, int kv_lora, int qk_rope) {
    return max_seq <= kAMaxSeq && mla_attend_lds(max_seq, kv_lora, qk_rope) + sizeof(float) * 2 * kCWaves +
                                          sizeof(float) * kCWaves * 64 <= kMaxLds;
}

hipError_t mla_absorb_attend(const float *q_abs, const float *q, const uint8_t *cache, size_t crb, const float *delta,
                             float *delta_out, const float *kv_cache, float *latent_out, int n_heads, int qk_nope,
                             int qk_rope, int kv_lora, const int *d_pos, int max_seq, float scale, hipStream_t s) {
    if (n_heads == 0) return hipSuccess;
    const ScoreArgs a{q_abs, q, cache, crb, delta, kv_cache, nullptr, n_heads, qk_nope, qk_rope, kv_lora, max_seq,
                      d_pos, scale};
    if (attend_blocks_ok(max_seq, kv_lora, qk_rope)) {
        hipLaunchKernelGGL(attend_blocks_kernel, dim3(n_heads), dim3(kCThreads), attend_blocks_lds(max_seq), s, a,
                           delta_out, latent_out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(attend_kernel, dim3(n_heads), dim3(kCThreads), mla_attend_lds(max_seq, kv_lora, qk_rope), s, a,
                       delta_out, latent_out);
    return hipGetLastError();
}

hipError_t mla_project_v(int type, const uint8_t *w, size_t rb, const uint8_t *cache, size_t crb, float *kvb_cache,
                         int n_heads, int qk_nope, int v_head, int kv_lora, const int *d_pos, hipStream_t s) {
    if (n_heads == 0 || v_head == 0) return hipSuccess;
    switch (type) {
        case T_Q4_K: ProjectV<T_Q4_K>::run(w, rb, cache, crb, kvb_cache, n_heads, qk_nope, v_head, kv_lora, d_pos, s); break;
        case T_Q6_K: ProjectV<T_Q6_K>::run(w, rb, cache, crb, kvb_cache, n_heads, qk_nope, v_head, kv_lora, d_pos, s); break;
        case T_Q5_0: ProjectV<T_Q5_0>::run(w, rb, cache, crb, kvb_cache, n_heads, qk_nope, v_head, kv_lora, d_pos, s); break;
        case T_Q8_0: ProjectV<T_Q8_0>::run(w, rb, cache, crb, kvb_cache, n_heads, qk_nope, v_head, kv_lora, d_pos, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t mla_absorb_context_v(const float *scores, const float *kvb_cache, float *attn, int n_heads, int qk_nope,
                                int v_head, const int *d_pos, int max_seq, hipStream_t s) {
    if (n_heads == 0 || v_head == 0) return hipSuccess;
    hipLaunchKernelGGL(context_v_kernel, dim3(n_heads), dim3(kCThreads), 0, s, scores, kvb_cache, attn, n_heads,
                       qk_nope, v_head, d_pos, max_seq);
    return hipGetLastError();
}

}  // namespace qlin
