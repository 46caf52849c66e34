// Device-side pack(): dense fp16 weight (N, K) + sorted cherry channels -> the packed buffers
// (scales, qweight, cherry_weight), bit for bit what the host path computes.
//
// Arithmetic follows the reference's offline path: llama/qlinear.py:67-118 (column split, code
// offset, byte layout), llama/cherry_linear.py:69-75 (groups over the COMPACTED normal columns),
// llama/quantizer.py:148-158 (scale and rounding rule).  For fp16 weights every torch operation
// there is "compute in fp32, round to fp16":
//   s    = RN16( f32( RN16( f32(max|w|) + 1e-6f ) ) / 2^(b-1) )
//   q    = rint( clamp( f32( RN16( f32(w) / f32(s) ) ), -qmax, qmax ) - 0.5 ),  qmax = 2^(b-1) - 0.01
//   code = q + 2^(b-1)
// (fp32 division followed by rounding to fp16 equals the correctly rounded fp16 quotient: 24 >= 2*11+2.)
#include "cq_device.h"
#include "cq_kernels.h"

namespace cq {

// source channel of compacted normal position k: k + #{m : idx[m] - m <= k}
__device__ inline int normal_source(const int16_t *__restrict__ idx, int C, int k) {
    int lo = 0, hi = C;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)idx[mid] - mid <= k) lo = mid + 1; else hi = mid;
    }
    return k + lo;
}

// The general form (any group size, any N): scales by one wavefront per (group, output row), then the codes.
__global__ __launch_bounds__(256) void pack_scales_kernel(const __half *__restrict__ w,
                                                          const int16_t *__restrict__ idx,
                                                          __half *__restrict__ scales, int K, int N, int C, int G,
                                                          int bits) {
    const int lane = threadIdx.x & 63;
    const long long item = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int Kn = K - C, ng = ceil_div(Kn, G);
    if (item >= (long long)ng * N) return;
    const int g = (int)(item / N), n = (int)(item % N);
    const int k0 = g * G, k1 = min(k0 + G, Kn);
    float mx = 0.f;
    for (int k = k0 + lane; k < k1; k += 64)
        mx = fmaxf(mx, fabsf(__half2float(w[(size_t)n * K + normal_source(idx, C, k)])));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) {
        const float a = __half2float(__float2half_rn(mx + 1e-6f));
        scales[(size_t)g * N + n] = __float2half_rn(a / (float)(1 << (bits - 1)));
    }
}

// Tile of 64 output rows x 128 compacted positions per workgroup: the weights are read along K
// (contiguous in the dense layout), staged in LDS, and the packed bytes written along N
// (contiguous in the packed layout).
template <int BITS>
__global__ __launch_bounds__(256) void pack_codes_kernel(const __half *__restrict__ w,
                                                         const int16_t *__restrict__ idx,
                                                         const __half *__restrict__ scales,
                                                         uint8_t *__restrict__ qweight, int K, int N, int C, int G) {
    __shared__ unsigned short s_w[64][130];
    const int Kn = K - C;
    const int k0 = blockIdx.x * 128, n0 = blockIdx.y * 64;
    const int t = threadIdx.x;
    for (int e = t; e < 64 * 128; e += 256) {
        const int nl = e >> 7, kl = e & 127;
        const int n = n0 + nl, k = k0 + kl;
        unsigned short v = 0;
        if (n < N && k < Kn) v = __half_as_ushort(w[(size_t)n * K + normal_source(idx, C, k)]);
        s_w[nl][kl] = v;
    }
    __syncthreads();
    const float qmax = (float)(1 << (BITS - 1)) - 1e-2f;
    for (int e = t; e < 16 * 64; e += 256) {
        const int nl = e & 63, j = e >> 6;  // unit of 8 positions
        const int n = n0 + nl, k = k0 + 8 * j;
        if (n >= N || k >= Kn) continue;
        uint32_t word = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            // a group boundary can fall inside a unit when G is not a multiple of 8
            const float s = __half2float(scales[(size_t)((k + i) / G) * N + n]);
            const float x = __half2float(__ushort_as_half(s_w[nl][8 * j + i]));
            float r = __half2float(__float2half_rn(x / s));
            r = fminf(fmaxf(r, -qmax), qmax) - 0.5f;
            const int code = (int)rintf(r) + (1 << (BITS - 1));
            word |= (uint32_t)(code & ((1 << BITS) - 1)) << (BITS * i);
        }
        const size_t row = (size_t)(k / 8) * BITS;
#pragma unroll
        for (int b = 0; b < BITS; b++) qweight[(row + b) * N + n] = (uint8_t)(word >> (8 * b));
    }
}

// cherry_weight[c, n] = w[n, idx[c]]
__global__ __launch_bounds__(256) void pack_cherry_kernel(const __half *__restrict__ w,
                                                          const int16_t *__restrict__ idx,
                                                          __half *__restrict__ cherry_weight, int K, int N, int C) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long long)C * N) return;
    const int c = (int)(e / N), n = (int)(e % N);
    cherry_weight[e] = w[(size_t)n * K + idx[c]];
}

// The common form (groups of whole units up to 128, N a multiple of 4): scales, codes and cherry rows from ONE
// read of the dense weight.  A workgroup owns 128 output rows x one group.  The group's dense columns are
// a contiguous range; 16 threads take a row of it in 16-byte chunks and scatter the halves to their
// compacted positions in LDS.  Where a chunk's halves go does not depend on the row, so a thread
// finds it once for the 8 rows it loads (two searches of the index list per chunk and row were what the
// general form spent its time on).  A row of 65 dwords spreads the scatter (16 chunks x 4 rows) and
// the later reads over the banks; bytes of four neighbouring rows leave as one dword, 128 bytes a line.
// No one unit bounds it: of 130 k cycles the vector ALU is busy 68 k (16 operations an element) and a compute unit's LDS 48 k, 29 k of
// these in bank conflicts; the weight's lines are fetched 1.4 times, since neighbouring groups share them.  Twice as many
// wavefronts a CU change nothing.  MI355X, 13824 x 5120 to 3 bits: 49 us (3.5 TB/s read + written),
// with an address formed for each half and row, comparisons around loads and stores, cherry columns stored half by
// half in the scatter and quotients of six operations 59 (188); the general form's three launches took 549.
constexpr int kPackRows = 128, kPackStride = 65;  // dwords of LDS a row; halves 128 and 129 take what belongs nowhere
constexpr int kPackMaxCherries = 1024;
constexpr int kPackThreads = 256, kPackLoads = kPackRows * 16 / kPackThreads;  // 16-byte chunks a thread loads

struct PackChunk {
    uint32_t off[8];   // LDS half of each of the 8 columns
    uint32_t valid[4]; // per pair of columns: 0x7fff where the column belongs to the group
};

__device__ __forceinline__ PackChunk pack_chunk(const int16_t *s_idx, int C, int col0, int k0, int k1) {
    PackChunk m;
    int lo = 0, hi = C;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)s_idx[mid] < col0) lo = mid + 1; else hi = mid;
    }
    uint32_t cherry = 0;
    for (int c = lo; c < C && (int)s_idx[c] < col0 + 8; c++) cherry |= 1u << ((int)s_idx[c] - col0);
    int pos = col0 - lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const bool normal = !((cherry >> e) & 1u), in = normal && pos >= k0 && pos < k1;
        m.off[e] = in ? pos - k0 : 128;
        if (e & 1) m.valid[e >> 1] |= in ? 0x7fff0000u : 0u;
        else m.valid[e >> 1] = in ? 0x7fffu : 0u;
        pos += normal;
    }
    return m;
}

// Two quotients x / s: the product with the reciprocal and one correction step.  The mixed-precision forms read the
// halves where they lie and round once, to fp16: three operations a value instead of six.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2_t pack_quotients(uint32_t x, float s, float rs) {
    float q0, q1, e0, e1;
    uint32_t r;
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(q0) : "v"(x), "v"(rs));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(q1) : "v"(x), "v"(rs));
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(e0) : "v"(q0), "v"(s), "v"(x));
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(e1) : "v"(q1), "v"(s), "v"(x));
    asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(r) : "v"(e0), "v"(rs), "v"(q0));
    asm("v_fma_mixhi_f16 %0, %1, %2, %3" : "+v"(r) : "v"(e1), "v"(rs), "v"(q1));
    return __builtin_bit_cast(half2_t, r);
}
// Both halves clamped to +-(2^(BITS-1) - 0.01) rounded to fp16, NaN to the lower end.
template <int BITS>
__device__ __forceinline__ half2_t pack_clamp(half2_t v) {
    constexpr uint32_t top = BITS == 4 ? 0x47fd47fdu : 0x43fb43fbu;
    asm("v_pk_max_f16 %0, %0, %1\n\tv_pk_min_f16 %0, %0, %2" : "+v"(v) : "s"(top | 0x80008000u), "s"(top));
    return v;
}

template <int BITS>
__global__ __launch_bounds__(kPackThreads) void pack_group_kernel(const __half *__restrict__ w, const int16_t *__restrict__ idx,
                                                         uint8_t *__restrict__ qweight, __half *__restrict__ scales,
                                                         __half *__restrict__ cherry_weight, int K, int N, int C, int G) {
    __shared__ uint32_t s_w[kPackRows * kPackStride];
    __shared__ uint32_t s_max[kPackRows];
    __shared__ float s_s[kPackRows], s_r[kPackRows];
    __shared__ int16_t s_idx[kPackMaxCherries];
    const int t = threadIdx.x, g = blockIdx.x, n0 = blockIdx.y * kPackRows;
    const int Kn = K - C, k0 = g * G, k1 = min(k0 + G, Kn);
    for (int i = t; i < C; i += kPackThreads) s_idx[i] = idx[i];
    if (t < kPackRows) s_max[t] = 0;
    __syncthreads();
    // the group's columns, with the cherries behind its last normal column (in front of column 0's too)
    auto source = [&](int k) {
        int lo = 0, hi = C;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if ((int)s_idx[mid] - mid <= k) lo = mid + 1; else hi = mid;
        }
        return k + lo;
    };
    const int col0 = g == 0 ? 0 : source(k0), col1 = k1 == Kn ? K : source(k1);  // [col0, col1)
    const int c0 = col0 >> 3, nch = ((col1 - 1) >> 3) - c0 + 1;

    // `at`: where the chunk's columns go in the row's LDS -> the chunk's largest magnitude in the group
    auto place = [&](const PackChunk &m, unsigned short *const (&at)[8], const uint4 &q, int step) {
        const uint32_t d[4] = {q.x, q.y, q.z, q.w};
        // Two halves at a time, moved up by 0x83ff: magnitudes up to infinity (0x7c00) end at 0xffff, a NaN's wrap to below
        // 0x83ff and take no part in the maximum.
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        u16x2 top = {0x83ff, 0x83ff};
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const u16x2 a = __builtin_bit_cast(u16x2, d[p] & m.valid[p]) + (u16x2){0x83ff, 0x83ff};
            top = __builtin_elementwise_max(top, a);
            at[2 * p][step * 2 * kPackStride] = (unsigned short)d[p];
            at[2 * p + 1][step * 2 * kPackStride] = (unsigned short)(d[p] >> 16);
        }
        return (uint32_t)max(top[0], top[1]) - 0x83ffu;
    };
    auto columns = [&](const PackChunk &m, int row, unsigned short *(&at)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e++) at[e] = reinterpret_cast<unsigned short *>(s_w + row * kPackStride) + m.off[e];
    };
    // The chunk or two that cherries and alignment push the range beyond 16, one a thread, and the first cherry columns, one value a
    // thread, are asked for with the rest: behind it their round trip was one more (13824 x 5120 to 3 bits 51.2 -> 49.2 us).
    const int more_row = t % kPackRows, more = 16 + t / kPackRows, cherry0 = col0 - k0, cherries = col1 - k1 - cherry0, cherry = t / kPackRows;
    const __half *const more_at = w + (size_t)min(n0 + more_row, N - 1) * K;
    uint4 mq = make_uint4(0, 0, 0, 0);
    __half first_cherry = __half(0.f);
    {
        // A thread without a chunk or a row of its own repeats the last one: the same bytes to the same place (rows past N are
        // not read again), and neither loads nor stores wait for a comparison.
        const int ci = min(t & 15, nch - 1), r0 = t >> 4;
        uint4 q[kPackLoads];
#pragma unroll
        for (int i = 0; i < kPackLoads; i++)
            q[i] = *reinterpret_cast<const uint4 *>(w + (size_t)min(n0 + r0 + kPackThreads / 16 * i, N - 1) * K + 8 * (c0 + ci));
        if (more < nch) mq = *reinterpret_cast<const uint4 *>(more_at + 8 * (c0 + more));
        if (cherry < cherries) first_cherry = more_at[s_idx[cherry0 + cherry]];
        const PackChunk m = pack_chunk(s_idx, C, 8 * (c0 + ci), k0, k1);
        unsigned short *at[8];
        columns(m, r0, at);
#pragma unroll
        for (int i = 0; i < kPackLoads; i++) {
            // across the row's 16 lanes first: 16 atomics on one word of LDS take turns
            const uint32_t mx = (uint32_t)row_max((int)place(m, at, q[i], kPackThreads / 16 * i));
            if ((t & 15) == 0) atomicMax(&s_max[r0 + kPackThreads / 16 * i], mx);
        }
    }
    for (int e = t; e < (nch - 16) * kPackRows; e += kPackThreads) {
        const int row = e % kPackRows, c = c0 + 16 + e / kPackRows;
        if (e != t) mq = *reinterpret_cast<const uint4 *>(more_at + 8 * c);
        const PackChunk m = pack_chunk(s_idx, C, 8 * c, k0, k1);
        unsigned short *at[8];
        columns(m, row, at);
        atomicMax(&s_max[row], place(m, at, mq, 0));
    }
    // the cherry columns: 128 neighbouring halves of an output row leave together
    for (int e = t; e < cherries * kPackRows; e += kPackThreads) {
        const int c = cherry0 + e / kPackRows;
        if (n0 + more_row < N) cherry_weight[(size_t)c * N + n0 + more_row] = e == t ? first_cherry : more_at[s_idx[c]];
    }
    __syncthreads();
    if (t < kPackRows) {
        const float mx = __half2float(__ushort_as_half((unsigned short)s_max[t]));
        const float a = __half2float(__float2half_rn(mx + 1e-6f));
        const __half sh = __float2half_rn(a / (float)(1 << (BITS - 1)));
        if (n0 + t < N) scales[(size_t)g * N + n0 + t] = sh;
        s_s[t] = __half2float(sh);
        s_r[t] = __builtin_amdgcn_rcpf(__half2float(sh));
    }
    __syncthreads();
    const float magic = 12582912.f + (float)(1 << (BITS - 1));  // 1.5 * 2^23: adding it rounds to the nearest even integer
    const int units = (k1 - k0) / 8;
    for (int it = t; it < 32 * units; it += kPackThreads) {
        const int rq = it & 31, j = it >> 5;
        if (n0 + 4 * rq >= N) continue;
        uint32_t word[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 4 * rq + r;
            const float s = s_s[row], rs = s_r[row];
            const float sf = __builtin_isinf(s) ? 0.f : s;  // finite / inf: the correction below must not form inf * 0
            const uint32_t *src = s_w + row * kPackStride + 4 * j;
            uint32_t half[2];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                // RN16(x / s) from the reciprocal and one correction step (less than one fp32 ulp off; a
                // quotient of two 11-bit significands stays more than 2^-23 away from every fp16 tie), then
                // clamped to +-(2^(BITS-1) - 0.01), in fp16 the neighbour of that with the same code
                const half2_t v = pack_clamp<BITS>(pack_quotients(src[p], sf, rs));
                float f0, f1;  // v - 0.5, exact
                asm("v_fma_mix_f32 %0, %1, 1.0, -0.5 op_sel_hi:[1,0,0]" : "=v"(f0) : "v"(v));
                asm("v_fma_mix_f32 %0, %1, 1.0, -0.5 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(f1) : "v"(v));
                const uint32_t lo = __float_as_uint(f0 + magic), hi = __float_as_uint(f1 + magic);
                // the sum's low 22 bits are 0..2^BITS - 1: four codes leave its exponent above 22 - 3 * 4 unmasked
                uint32_t &w2 = half[p >> 1];
                w2 = (p & 1) ? (lo << (2 * BITS)) | w2 : lo;
                w2 = (hi << (BITS * (2 * (p & 1) + 1))) | w2;
            }
            word[r] = (half[1] << (4 * BITS)) | (half[0] & ((1u << (4 * BITS)) - 1u));
        }
        uint8_t *o = qweight + (size_t)(k0 / 8 + j) * BITS * N + n0 + 4 * rq;
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            uint32_t d = 0;
#pragma unroll
            for (int r = 0; r < 4; r++) d |= ((word[r] >> (8 * b)) & 0xffu) << (8 * r);
            *reinterpret_cast<uint32_t *>(o + (size_t)b * N) = d;
        }
    }
}

// Distinct channels in any order -> ascending int16.  *bad: 1 where one is outside [0, K) or named twice (the
// output then still holds channels within [0, K)).  One workgroup: a bit per channel and a count of the bits before.
constexpr int kSortWords = 1024;  // K <= 32768, what int16 can name
template <typename I>
__global__ __launch_bounds__(256) void sort_channels_kernel(const I *__restrict__ idx, int16_t *__restrict__ out,
                                                            int *__restrict__ bad, int C, int K) {
    __shared__ uint32_t s_mask[kSortWords];
    __shared__ uint32_t s_sum[4];
    __shared__ int s_bad;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    for (int i = t; i < kSortWords; i += 256) s_mask[i] = 0;
    if (t == 0) s_bad = 0;
    __syncthreads();
    for (int i = t; i < C; i += 256) {
        const long long j = (long long)idx[i];
        if (j < 0 || j >= K) s_bad = 1;
        else if (atomicOr(&s_mask[j >> 5], 1u << (j & 31)) & (1u << (j & 31))) s_bad = 1;
    }
    __syncthreads();
    uint32_t mine = 0;
    for (int i = 0; i < kSortWords / 256; i++) mine += __popc(s_mask[t * (kSortWords / 256) + i]);
    uint32_t incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
    }
    if (lane == 63) s_sum[wave] = incl;
    __syncthreads();
    uint32_t at = incl - mine, all = 0;
    for (int v = 0; v < 4; v++) {
        if (v < wave) at += s_sum[v];
        all += s_sum[v];
    }
    for (int i = 0; i < kSortWords / 256; i++) {
        const int wd = t * (kSortWords / 256) + i;
        for (uint32_t m = s_mask[wd]; m; m &= m - 1) out[at++] = (int16_t)(32 * wd + __builtin_ctz(m));
    }
    for (int i = (int)all + t; i < C; i += 256) out[i] = (int16_t)(K - 1);
    if (t == 0) *bad = s_bad;
}

hipError_t launch_sort_channels(const void *idx, int index_bytes, int16_t *out, int *bad, int C, int K, hipStream_t stream) {
    if (index_bytes == 2)
        hipLaunchKernelGGL(sort_channels_kernel<int16_t>, dim3(1), dim3(256), 0, stream, reinterpret_cast<const int16_t *>(idx), out, bad, C, K);
    else if (index_bytes == 4)
        hipLaunchKernelGGL(sort_channels_kernel<int32_t>, dim3(1), dim3(256), 0, stream, reinterpret_cast<const int32_t *>(idx), out, bad, C, K);
    else
        hipLaunchKernelGGL(sort_channels_kernel<int64_t>, dim3(1), dim3(256), 0, stream, reinterpret_cast<const int64_t *>(idx), out, bad, C, K);
    return hipGetLastError();
}

hipError_t launch_pack(int bits, const __half *w, const int16_t *idx, uint8_t *qweight, __half *scales,
                       __half *cherry_weight, int K, int N, int C, int G, hipStream_t stream) {
    const int Kn = K - C;
    // one read of the weight wherever a group fits a workgroup's LDS and chunks and dwords are aligned
    if (Kn > 0 && G % 8 == 0 && G <= 128 && N % 4 == 0 && C <= kPackMaxCherries && aligned(w, 16) && aligned(qweight, 4)) {
        const dim3 grid(ceil_div(Kn, G), ceil_div(N, kPackRows));
        if (bits == 4)
            hipLaunchKernelGGL(pack_group_kernel<4>, grid, dim3(kPackThreads), 0, stream, w, idx, qweight, scales, cherry_weight, K, N, C, G);
        else
            hipLaunchKernelGGL(pack_group_kernel<3>, grid, dim3(kPackThreads), 0, stream, w, idx, qweight, scales, cherry_weight, K, N, C, G);
        return hipGetLastError();
    }
    if (Kn > 0) {
        const long long items = (long long)ceil_div(Kn, G) * N;
        hipLaunchKernelGGL(pack_scales_kernel, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, stream, w, idx, scales,
                           K, N, C, G, bits);
        const dim3 grid(ceil_div(Kn, 128), ceil_div(N, 64));
        if (bits == 4)
            hipLaunchKernelGGL(pack_codes_kernel<4>, grid, dim3(256), 0, stream, w, idx, scales, qweight, K, N, C, G);
        else
            hipLaunchKernelGGL(pack_codes_kernel<3>, grid, dim3(256), 0, stream, w, idx, scales, qweight, K, N, C, G);
    }
    if (C > 0)
        hipLaunchKernelGGL(pack_cherry_kernel, dim3((unsigned)(((long long)C * N + 255) / 256)), dim3(256), 0, stream,
                           w, idx, cherry_weight, K, N, C);
    return hipGetLastError();
}

}  // namespace cq
