// The operations between the linears of a decoder layer for a whole prompt of T rows (the one-row forms of a token step
// are in cq_decode.hip): residual + RMSNorm, rotary embedding + cache write, causal attention.
//
// Semantics follow the reference's model code (llama/modeling_llama_quant.py): RMSNorm :75-89, rotary embedding :95-210,
// attention :391-402 and :671-696.  fp16 storage, fp32 arithmetic inside a kernel, roundings where the
// reference's fp16 tensors are materialised; scores stay in fp32 (the reference's are rounded to fp16 twice).
//
// All of them are bound by latency at prompt lengths of a few hundred: what counts is the number of launches.  As
// tensor operations they were some 35 launches a layer; now they are five (7B, 128 tokens, whole prompt: 11.5 -> 6.1 ms;
// norm 3.9, keys and values 3.3, attention 5.3 us).  In the native pass over plain layers the norms, SiLU * up (cq_prompt.hip) and the
// attention write the next product's operands too.
#include "cq_device.h"
#include "cq_kernels.h"

// products and sums of the rotary embedding are rounded one by one
#pragma clang fp contract(off)

namespace cq {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// ---- h <- h + delta (none: as it is);  y <- weight * fp16(h * rsqrt(mean(h^2) + eps)), row by row ------------
// A workgroup owns a row and keeps it in registers between the two passes.  H % 8 == 0, H <= 8192.
constexpr int kNormChunks = kPrefillMaxHidden / (256 * 8);

__global__ __launch_bounds__(256) void prefill_norm_kernel(__half *__restrict__ h, const __half *__restrict__ delta,
                                                           const __half *__restrict__ weight, __half *__restrict__ y, int H,
                                                           float eps) {
    __shared__ float s_part[4];
    const int t = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * H;
    half8_t v[kNormChunks], w[kNormChunks];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < kNormChunks; c++) {
        const int i = 8 * (t + 256 * c);
        if (i >= H) break;
        v[c] = *reinterpret_cast<const half8_t *>(h + row + i);
        w[c] = *reinterpret_cast<const half8_t *>(weight + i);
        if (delta) {
            v[c] += *reinterpret_cast<const half8_t *>(delta + row + i);
            *reinterpret_cast<half8_t *>(h + row + i) = v[c];
        }
#pragma unroll
        for (int e = 0; e < 8; e++) ss += (float)v[c][e] * (float)v[c][e];
    }
    ss = wave_sum_all(ss);
    if ((t & 63) == 0) s_part[t >> 6] = ss;
    __syncthreads();
    const float rs = rsqrtf((s_part[0] + s_part[1] + s_part[2] + s_part[3]) / (float)H + eps);
#pragma unroll
    for (int c = 0; c < kNormChunks; c++) {
        const int i = 8 * (t + 256 * c);
        if (i >= H) break;
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = w[c][e] * (_Float16)((float)v[c][e] * rs);
        *reinterpret_cast<half8_t *>(y + row + i) = o;
    }
}

// ---- rotary embedding ----------------------------------------------------------------------------------------
// a: dimensions i .. i + 7 of a head, b: the same + 64; c, s: cosine and sine of their angles
__device__ __forceinline__ void rotate(half8_t &a, half8_t &b, const half8_t c, const half8_t s) {
    const half8_t x1 = a, x2 = b;
    a = x1 * c + (-x2) * s;
    b = x2 * c + x1 * s;
}

// ---- keys and values into the cache and into the order the attention kernel reads ------------------------------
// Fragments of v_mfma_f32_16x16x32_f16: a lane holds 8 consecutive k-indices of one row (or column).
//   kf[((head * 2 VB + key / 16) * 4 + dim / 32) * 64 + (dim % 32) / 8 * 16 + key % 16]: 8 dimensions of a key
//   vf[((head * VB + key / 32) * 8 + dim / 16) * 64 + q * 16 + dim % 16]: the 8 keys 4 q + 0..3 and 16 + 4 q + 0..3 of 32
// (VB = ceil(T / 32); the second is the key order in which the product of keys and queries leaves its results in a
// lane, so that probabilities need no exchange between lanes).  Positions T and above of the last block are zeros.
__global__ __launch_bounds__(256) void prefill_kv_kernel(const __half *__restrict__ k, const __half *__restrict__ v,
                                                         const __half *__restrict__ cos_t, const __half *__restrict__ sin_t,
                                                         __half *__restrict__ k_cache, __half *__restrict__ v_cache,
                                                         half8_t *__restrict__ kf, half8_t *__restrict__ vf, int T, int max_len) {
    __shared__ __attribute__((aligned(16))) _Float16 s_v[32][128 + 8];
    const int t = threadIdx.x, r = t >> 3, c = t & 7, block = blockIdx.x, head = blockIdx.y, VB = gridDim.x;
    const int pos = 32 * block + r;
    const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    half8_t k0 = zero, k1 = zero, v0 = zero, v1 = zero;
    if (pos < T) {
        const size_t src = ((size_t)pos * gridDim.y + head) * 128 + 8 * c, dst = ((size_t)head * max_len + pos) * 128 + 8 * c;
        k0 = *reinterpret_cast<const half8_t *>(k + src), k1 = *reinterpret_cast<const half8_t *>(k + src + 64);
        v0 = *reinterpret_cast<const half8_t *>(v + src), v1 = *reinterpret_cast<const half8_t *>(v + src + 64);
        rotate(k0, k1, *reinterpret_cast<const half8_t *>(cos_t + (size_t)pos * 64 + 8 * c),
               *reinterpret_cast<const half8_t *>(sin_t + (size_t)pos * 64 + 8 * c));
        *reinterpret_cast<half8_t *>(k_cache + dst) = k0, *reinterpret_cast<half8_t *>(k_cache + dst + 64) = k1;
        *reinterpret_cast<half8_t *>(v_cache + dst) = v0, *reinterpret_cast<half8_t *>(v_cache + dst + 64) = v1;
    }
    half8_t *const kd = kf + ((size_t)(head * 2 * VB + 2 * block + (r >> 4)) * 4 + (c >> 2)) * 64 + (c & 3) * 16 + (r & 15);
    kd[0] = k0, kd[2 * 64] = k1;
    *reinterpret_cast<half8_t *>(&s_v[r][8 * c]) = v0, *reinterpret_cast<half8_t *>(&s_v[r][8 * c + 64]) = v1;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int e = t + 256 * p, lane = e & 63, q = lane >> 4, dim = 16 * (e >> 6) + (lane & 15);
        half8_t o;
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = s_v[16 * (j >> 2) + 4 * q + (j & 3)][dim];
        vf[(size_t)(head * VB + block) * 512 + e] = o;
    }
}

// ---- causal attention over the prompt ------------------------------------------------------------------------
// A workgroup owns 16 R queries of one head; its four wavefronts take blocks of 32 keys in turn, each with its own running
// maximum and sum, and meet once in LDS.  Scores are formed as keys x queries, so that a lane holds 8 keys of ONE query:
// maximum and sum need two exchanges a block, and the probabilities already lie as the value product reads
// them.  Queries are rotated on their way in.  Long prompts first: tiles run from the last queries to the first.
// R = 2 halves the reads of keys and values, R = 1 gives twice the workgroups.
//   BITS > 0: the result is written as the output projection (codes of BITS bits) reads its rows: gathered around that layer's
// cherry channels, in operand order (prompt_prep_kernel, cq_prompt.hip), 16 rows of 8 positions in 256 bytes.  The head's 128 channels are
// consecutive positions but for its cherries, which go to their own places; where a head does not begin at a multiple of eight
// positions, the eight that it shares with a neighbour are written value by value.  (7B, 128 tokens, us: attention 4.8 and a launch of 4.9
// that gathered its rows behind it; now 7.1.)
template <int R, int BITS>
__global__ __launch_bounds__(256) void prefill_attention_kernel(const __half *__restrict__ q, const __half *__restrict__ cos_t,
                                                                const __half *__restrict__ sin_t, const half8_t *__restrict__ kf,
                                                                const half8_t *__restrict__ vf, __half *__restrict__ out, int T,
                                                                int n_heads, int rep, float scale_log2, PrefillOperands to) {
    __shared__ __attribute__((aligned(16))) float s_o[4][16][128 + 4];
    __shared__ float s_m[4][16 * R], s_l[4][16 * R];
    static_assert(R == 1 || BITS == 0, "");
    __shared__ __attribute__((aligned(16))) _Float16 s_row[BITS ? 16 : 1][128 + 8];
    __shared__ uint8_t s_normal[BITS ? 128 : 1], s_cherry[BITS ? 128 : 1];  // the head's channels: normal ones in order, cherries in order
    __shared__ int s_first[2];                                             // cherries in front of the head, and up to its end
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), kq = lane >> 4, i = lane & 15;
    // (neighbouring heads on one die, whose L2 holds the keys and values that they share and joins their pieces of the result)
    const int head = n_heads % 8 ? (int)blockIdx.x : ((int)blockIdx.x & 7) * (n_heads / 8) + ((int)blockIdx.x >> 3);
    const int q0 = 16 * R * ((int)gridDim.y - 1 - (int)blockIdx.y), VB = ceil_div(T, 32);
    const half8_t *const kh = kf + (size_t)(head / rep) * VB * 512 + lane, *const vh = vf + (size_t)(head / rep) * VB * 512 + lane;
    const int blocks = min(VB, (q0 + 16 * R + 31) / 32);

    half8_t qf[R][4];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int pos = min(q0 + 16 * r + i, T - 1);  // rows past the end are not stored
        const __half *src = q + ((size_t)pos * n_heads + head) * 128 + 8 * kq;
#pragma unroll
        for (int s = 0; s < 4; s++) qf[r][s] = *reinterpret_cast<const half8_t *>(src + 32 * s);
#pragma unroll
        for (int s = 0; s < 2; s++)
            rotate(qf[r][s], qf[r][s + 2], *reinterpret_cast<const half8_t *>(cos_t + (size_t)pos * 64 + 32 * s + 8 * kq),
                   *reinterpret_cast<const half8_t *>(sin_t + (size_t)pos * 64 + 32 * s + 8 * kq));
    }
    int channel = 0x7fffffff;  // asked for here, used behind the blocks
    if (BITS && wave < 2 && lane < to.C) channel = to.channels[lane];
    float4_t o[R][8];
    float m[R], l[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        m[r] = -__builtin_inff(), l[r] = 0.f;
#pragma unroll
        for (int d = 0; d < 8; d++) o[r][d] = (float4_t){0.f, 0.f, 0.f, 0.f};
    }
    for (int b = wave; b < blocks; b += 4) {
        half8_t kk[8], vv[8];
#pragma unroll
        for (int e = 0; e < 8; e++) kk[e] = kh[(size_t)b * 512 + e * 64];
#pragma unroll
        for (int e = 0; e < 8; e++) vv[e] = vh[(size_t)b * 512 + e * 64];
#pragma unroll
        for (int r = 0; r < R; r++) {
            float4_t s[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                s[h] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; e++) s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk[4 * h + e], qf[r][e], s[h], 0, 0, 0);
            }
            const int ahead = q0 + 16 * r + i - 32 * b - 4 * kq;  // key 16 h + e of the lane's is visible up to this one
            float top = m[r];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (16 * h + e > ahead) s[h][e] = -__builtin_inff();
                    top = fmaxf(top, s[h][e]);
                }
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(top, __shfl_xor(top, 32));  // finite: every block has a key that all its queries see
            const float keep = __builtin_amdgcn_exp2f((m[r] - top) * scale_log2);
            m[r] = top, l[r] *= keep;
            half8_t p;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float x = __builtin_amdgcn_exp2f((s[h][e] - top) * scale_log2);
                    l[r] += x;
                    p[4 * h + e] = (_Float16)x;
                }
#pragma unroll
            for (int d = 0; d < 8; d++) o[r][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv[d], p, o[r][d] * keep, 0, 0, 0);
        }
    }
    if (BITS && wave < 2) {
        // A lane is a channel: which cherry it is, if it is one, and how many lie in front of it
        const int c0 = 128 * head, mine0 = c0 + 64 * wave;
        int front = 0, before = 0, cherry = -1;
        for (int k = 0; k < to.C; k += 64) {
            const int v = k == 0 ? channel : k + lane < to.C ? to.channels[k + lane] : 0x7fffffff;
            front += __popcll(__ballot(v < c0)), before += __popcll(__ballot(v < mine0));
            for (unsigned long long in = __ballot(v >= mine0 && v < mine0 + 64); in; in &= in - 1) {
                const int j = __builtin_ctzll(in);
                if (__builtin_amdgcn_readlane(v, j) == mine0 + lane) cherry = k + j;
            }
        }
        const unsigned long long cherries = __ballot(cherry >= 0);
        const int behind = 64 * wave + lane - (before - front) - __popcll(cherries & ((1ull << lane) - 1ull));  // normal ones of the head in front
        // (channels that are not in order or not distinct are nobody's: what becomes of them stays within the arrays, by the masks here and
        // where the bytes are read, of which some are then never written, and by the bound on `cherries`)
        if (cherry >= 0) s_cherry[(cherry - front) & 127] = (uint8_t)(64 * wave + lane);
        else s_normal[behind & 127] = (uint8_t)(64 * wave + lane);
        if (wave == 1 && lane == 0) s_first[0] = front, s_first[1] = before + __popcll(cherries);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        l[r] += __shfl_xor(l[r], 16);
        l[r] += __shfl_xor(l[r], 32);
        if (kq == 0) s_m[wave][16 * r + i] = m[r], s_l[wave][16 * r + i] = l[r];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r > 0) __syncthreads();
#pragma unroll
        for (int d = 0; d < 8; d++) *reinterpret_cast<float4_t *>(&s_o[wave][i][16 * d + 4 * kq]) = o[r][d];
        __syncthreads();
        const int row = t >> 4, c = t & 15, pos = q0 + 16 * r + row;
        float w[4], top = -__builtin_inff(), sum = 0.f;
#pragma unroll
        for (int k = 0; k < 4; k++) top = fmaxf(top, s_m[k][16 * r + row]);
#pragma unroll
        for (int k = 0; k < 4; k++) {  // a wavefront without a block: weight 0
            w[k] = __builtin_amdgcn_exp2f((s_m[k][16 * r + row] - top) * scale_log2);
            sum += w[k] * s_l[k][16 * r + row];
        }
        half8_t res;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < 4; k++) v += w[k] * s_o[k][row][8 * c + e];
            res[e] = (_Float16)(v / sum);
        }
        if constexpr (BITS == 0) {
            if (pos < T) *reinterpret_cast<half8_t *>(out + ((size_t)pos * n_heads + head) * 128 + 8 * c) = res;
        } else {
            *reinterpret_cast<half8_t *>(&s_row[row][8 * c]) = res;
            __syncthreads();
            const int front = s_first[0], cherries = min(s_first[1] - front, 128), p0 = max(128 * head - front, 0), p1 = p0 + 128 - cherries;
            const int last = head == n_heads - 1 ? to.units * 16 : ceil_div(p1, 8);  // the last head's: zeros up to the unit's end
            _Float16 *const a = reinterpret_cast<_Float16 *>(to.a + (size_t)(q0 / 16) * 64 + (t & 15));
            auto place = [&](int eight) { return a + ((size_t)(eight >> 2) * to.m16 * 64 + (eight & 3) * 16) * 8; };
            for (int eight = p0 / 8 + (t >> 4); eight < last; eight += 16) {
                half8_t v;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int p = 8 * eight + prompt_ord<BITS>(e);
                    v[e] = p >= p0 && p < p1 ? s_row[t & 15][s_normal[p - p0] & 127] : (_Float16)0.f;
                }
                if (8 * eight >= p0 && (8 * eight + 8 <= p1 || head == n_heads - 1)) {
                    *reinterpret_cast<half8_t *>(place(eight)) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int p = 8 * eight + prompt_ord<BITS>(e);
                        if (p >= p0 && p < p1) place(eight)[e] = v[e];
                    }
                }
            }
            for (int j = t >> 4; j < cherries; j += 16) place(to.units * 16 + (front + j) / 8)[(front + j) & 7] = s_row[t & 15][s_cherry[j] & 127];
            if (head == n_heads - 1) {
                const half8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
                for (int eight = to.C / 8 + (t >> 4); eight < to.csteps * 4; eight += 16)
                    *reinterpret_cast<half8_t *>(place(to.units * 16 + eight)) = zero;
            }
        }
    }
}

hipError_t launch_prefill_norm(__half *h, const __half *delta, const __half *weight, __half *y, int rows, int H, float eps,
                               hipStream_t stream) {
    hipLaunchKernelGGL(prefill_norm_kernel, dim3(rows), dim3(256), 0, stream, h, delta, weight, y, H, eps);
    return hipGetLastError();
}

// Operands of the output projection from the attention itself, or from a launch behind it.  Its end costs every workgroup about 2 us, the
// launch 5 and less the more rows there are: up to two workgroups a compute unit the former is faster (a layer of 4096 / 11008 with 32 heads, us: 64
// tokens 124.3 -> 122.2, 128: 126.0 -> 124.0, 256: 186 -> 184, 384: 248.0 -> 248.4, 600: 357 -> 361; of 8192 with 64: 128 tokens 231.7 -> 230.6, 400: 422 -> 424).
bool prefill_attention_operands(int T, int n_heads) { return (long long)ceil_div(T, 16) * n_heads <= 512; }

size_t prefill_attention_bytes(int T, int n_kv_heads) { return (size_t)ceil_div(T, 32) * n_kv_heads * 512 * 16 * 2; }

hipError_t launch_prefill_attention(const __half *q, const __half *k, const __half *v, const __half *cos_t, const __half *sin_t,
                                    __half *k_cache, __half *v_cache, __half *out, void *scratch, int T, int n_heads,
                                    int n_kv_heads, int max_len, int bits, const PrefillOperands &to, hipStream_t stream) {
    const int VB = ceil_div(T, 32), rep = n_heads / n_kv_heads;
    half8_t *const kf = reinterpret_cast<half8_t *>(scratch), *const vf = kf + (size_t)VB * n_kv_heads * 512;
    hipLaunchKernelGGL(prefill_kv_kernel, dim3(VB, n_kv_heads), dim3(256), 0, stream, k, v, cos_t, sin_t, k_cache, v_cache, kf, vf, T,
                       max_len);
    const float scale_log2 = 0.08838834764831845f * 1.4426950408889634f;  // 1 / sqrt(128), base 2
    // From two workgroups a compute unit on 32 queries each are faster, below that twice the workgroups are (us, 16 / 32
    // queries: 32 heads, 128 positions 4.5 / 6.5, 384: 9.3 / 11.1, 512: 15.7 / 12.9, 2048: 98 / 80; 64 heads over 8, 256: 11.1 / 10.3)
    const bool two = bits == 0 && (long long)ceil_div(T, 32) * n_heads >= 512;
    auto *const kernel = two         ? prefill_attention_kernel<2, 0>
                         : bits == 0 ? prefill_attention_kernel<1, 0>
                         : bits == 4 ? prefill_attention_kernel<1, 4> : prefill_attention_kernel<1, 3>;
    hipLaunchKernelGGL(kernel, dim3(n_heads, ceil_div(T, two ? 32 : 16)), dim3(256), 0, stream, q, cos_t, sin_t, kf, vf, out, T, n_heads, rep,
                       scale_log2, to);
    return hipGetLastError();
}

}  // namespace cq
