// QAT-side fake quantisation on the device: weight (N, K) -> weight with every non-cherry input
// channel replaced by its group-wise quantise-dequantise value, in ONE launch (the matrix is read
// from memory once and written once), in the weight's own dtype (fp16, bf16 or fp32).
//
// Arithmetic follows the reference's training forward, llama/cherry_linear.py:77-99
// (_adjust_weight: groups of G consecutive COMPACTED normal columns, cherry columns untouched,
// optional straight-through form  (q - w) + w) with llama/quantizer.py:148-152 (scale) and
// :165-170 (transform).  Every torch operation there rounds to the weight dtype, so with
// rnd() = "round to the weight dtype" (identity for fp32):
//   s = rnd( rnd(max|w| + 1e-6f) / 2^(b-1) )
//   r = clamp( rnd(w / s), -Q, Q ),  Q = rnd(2^(b-1) - 0.01)
//   q = rnd( (rint(rnd(r - 0.5)) + 0.5) * s )
// and, for the straight-through form, rnd( rnd(q - w) + w ) on every column.
//
// Every workgroup walks whole rows.  The cherry channels become a bit mask over the K columns in
// LDS (so the indices need neither be sorted nor distinct, as in the reference's scatter) with
// a prefix count per 32-column word: a column's compacted position is its index minus the
// cherries before it.
//
// row_kernel (rows of whole 16-byte chunks, groups of at least 8, up to 65536 columns): bound by HBM,
// one read and one write of the weight.  A thread owns the SAME chunks of 8 columns in every row its
// workgroup walks, so which elements are cherries and where the next group starts (a chunk meets at
// most two groups) is found once and kept in registers, not once per row and pass; the row
// itself stays in registers between the fold of |w| into its groups' maxima (LDS) and the
// quantisation, and the next row's chunks are requested before the workgroup waits for the maxima.
// Cherry elements are computed like the others and replaced by their original bits: no branch
// depends on the data.  MI355X, 4096 -> 11008: fp16 48-52 us (3.6 TB/s read + written; finding the chunk
// maps anew in both passes over a row took 69-73), fp32 78 us (4.6 TB/s; 81-91), bf16 47 us; 2000 x 1032: 8 us.
//
// element_kernel: everything else (ragged or misaligned rows, groups below 8), element by element.
#include "cq_device.h"
#include "cq_kernels.h"

#pragma clang fp contract(off)

namespace cq {

constexpr int kFqMaxWords = 2048;    // 32-column mask words: K <= 65536
constexpr int kFqMaxGroups = 4096;   // quantisation groups per row
constexpr int kFqThreads = 256;

bool fake_quant_supported(int K, int C, int G) {
    (void)C;
    if (K <= 0 || K > kFqMaxWords * 32 || G <= 0) return false;
    // the group count is at most ceil(K / G) whatever the indices hold
    return ceil_div(K, G) <= kFqMaxGroups;
}

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef unsigned short us2_t __attribute__((ext_vector_type(2)));

// 0 or 0xffffffff from bit i of m
__device__ __forceinline__ uint32_t bit_mask(uint32_t m, int i) { return (uint32_t)__builtin_amdgcn_sbfe((int)m, i, 1); }
// per 16-bit half of a pair (elements 2p, 2p+1): 0xffff where the element's bit of m is set
__device__ __forceinline__ uint32_t pair_mask(uint32_t m, int p) {
    return (bit_mask(m, 2 * p) & 0x0000ffffu) | (bit_mask(m, 2 * p + 1) & 0xffff0000u);
}
__device__ __forceinline__ uint32_t select_bits(uint32_t mask, uint32_t if_set, uint32_t if_clear) {
    return (if_set & mask) | (if_clear & ~mask);
}

// What a chunk of 8 columns needs to know about its groups: elements whose bit in `in_a` is set
// use the scale of group `a`, the others that of group `b`; bits of `cherry` mark elements that are
// left untouched.
struct ChunkMap {
    uint32_t in_a;      // 8 bits
    uint32_t cherry;    // 8 bits
};

// storage of a bfloat16 weight
struct bf16_t {
    uint16_t v;
};

// Per dtype: a chunk of 8 consecutive weights in registers, and the arithmetic on it.
template <typename T>
struct FqType;

// what the two 16-bit types share: 8 weights in 4 dwords
struct Fq16 {
    struct Raw { uint32_t d[4]; };
    static __device__ __forceinline__ Raw load_bits(const uint16_t *p, bool vec, int valid) {
        Raw r;
        if (vec) {
            const uint4 q = *reinterpret_cast<const uint4 *>(p);
            r.d[0] = q.x, r.d[1] = q.y, r.d[2] = q.z, r.d[3] = q.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t lo = 2 * i < valid ? p[2 * i] : 0u;
                const uint32_t hi = 2 * i + 1 < valid ? p[2 * i + 1] : 0u;
                r.d[i] = lo | (hi << 16);
            }
        }
        return r;
    }
    static __device__ __forceinline__ void store_bits(uint16_t *p, const Raw &r, bool vec, int valid) {
        if (vec) {
            *reinterpret_cast<uint4 *>(p) = make_uint4(r.d[0], r.d[1], r.d[2], r.d[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i < valid) p[i] = (uint16_t)(r.d[i >> 1] >> (16 * (i & 1)));
        }
    }
    // max |w| per group of the chunk as 16-bit patterns (which order like the magnitudes)
    static __device__ __forceinline__ void absmax_bits(const Raw &v, const ChunkMap &cm, uint32_t &ma, uint32_t &mb) {
        us2_t xa = {0, 0}, xb = {0, 0};
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint32_t a = v.d[p] & 0x7fff7fffu & ~pair_mask(cm.cherry, p);
            const uint32_t ina = pair_mask(cm.in_a, p);
            xa = __builtin_elementwise_max(xa, __builtin_bit_cast(us2_t, a & ina));
            xb = __builtin_elementwise_max(xb, __builtin_bit_cast(us2_t, a & ~ina));
        }
        ma = max(xa[0], xa[1]);
        mb = max(xb[0], xb[1]);
    }
};

template <>
struct FqType<__half> : Fq16 {
    static __device__ __forceinline__ float rnd(float x) { return __half2float(__float2half_rn(x)); }
    static __device__ __forceinline__ Raw load(const __half *p, bool vec, int valid) {
        return load_bits(reinterpret_cast<const uint16_t *>(p), vec, valid);
    }
    static __device__ __forceinline__ void store(__half *p, const Raw &r, bool vec, int valid) {
        store_bits(reinterpret_cast<uint16_t *>(p), r, vec, valid);
    }
    static __device__ __forceinline__ float get(const Raw &r, int i) {
        return __half2float(__ushort_as_half((unsigned short)(r.d[i >> 1] >> (16 * (i & 1)))));
    }
    static __device__ __forceinline__ void set(Raw &r, int i, float v) {
        const uint32_t h = __half_as_ushort(__float2half_rn(v));
        r.d[i >> 1] = (i & 1) ? ((r.d[i >> 1] & 0x0000ffffu) | (h << 16)) : ((r.d[i >> 1] & 0xffff0000u) | h);
    }
    // RN16(w / s) without the IEEE division sequence: one Newton step on w * (1/s) leaves less
    // than one fp32 ulp of error, and a quotient of two 11-bit significands that is not itself
    // an fp16 rounding boundary stays more than 2^-23 (relative) away from every boundary, so
    // the rounding to fp16 sees the same side as the exact quotient.
    static __device__ __forceinline__ float quot32(float w, float s, float rs) {
        const float q0 = w * rs;
        const float e = __builtin_fmaf(-q0, s, w);
        return __builtin_fmaf(e, rs, q0);
    }
    static __device__ __forceinline__ float one(float w, float s, float qmax) {
        float r = rnd(quot32(w, s, __builtin_amdgcn_rcpf(s)));
        r = fminf(fmaxf(r, -qmax), qmax);
        r = rnd(r - 0.5f);
        r = rintf(r) + 0.5f;  // both exact in fp16 for |r| <= 8.5
        return rnd(r * s);
    }
    static __device__ __forceinline__ void absmax(const Raw &v, const ChunkMap &cm, uint32_t &ma, uint32_t &mb) {
        absmax_bits(v, cm, ma, mb);
        ma = __float_as_uint(__half2float(__ushort_as_half((unsigned short)ma)));
        mb = __float_as_uint(__half2float(__ushort_as_half((unsigned short)mb)));
    }
    // fp16 addition and multiplication round like "fp32 operation, then round to fp16" (the
    // fp32 result of two fp16 operands is exact or far from any fp16 tie), so everything after
    // the quotient runs on packed fp16 instructions
    static __device__ __forceinline__ Raw all(const Raw &w, const ChunkMap &cs, float sa, float sb, float qmax, int ste) {
        const float rsa = __builtin_amdgcn_rcpf(sa), rsb = __builtin_amdgcn_rcpf(sb);
        const uint32_t sa16 = __half_as_ushort(__float2half_rn(sa)), sb16 = __half_as_ushort(__float2half_rn(sb));
        const uint32_t aa = sa16 | (sa16 << 16), bb = sb16 | (sb16 << 16);
        const _Float16 qh = (_Float16)qmax;
        const h2_t hi = {qh, qh}, lo = {-qh, -qh}, half2 = {(_Float16)0.5f, (_Float16)0.5f};
        Raw o;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const h2_t wv = __builtin_bit_cast(h2_t, w.d[p]);
            const h2_t s2 = __builtin_bit_cast(h2_t, select_bits(pair_mask(cs.in_a, p), aa, bb));
            const float rs0 = __uint_as_float(select_bits(bit_mask(cs.in_a, 2 * p), __float_as_uint(rsa), __float_as_uint(rsb)));
            const float rs1 = __uint_as_float(select_bits(bit_mask(cs.in_a, 2 * p + 1), __float_as_uint(rsa), __float_as_uint(rsb)));
            h2_t r = {(_Float16)quot32((float)wv[0], (float)s2[0], rs0), (_Float16)quot32((float)wv[1], (float)s2[1], rs1)};
            r = __builtin_elementwise_min(__builtin_elementwise_max(r, lo), hi);
            r = r - half2;
            r = __builtin_elementwise_rint(r) + half2;
            const h2_t q = r * s2;
            uint32_t bits = select_bits(pair_mask(cs.cherry, p), w.d[p], __builtin_bit_cast(uint32_t, q));
            if (ste) {
                const h2_t qq = __builtin_bit_cast(h2_t, bits);
                bits = __builtin_bit_cast(uint32_t, (h2_t)((qq - wv) + wv));
            }
            o.d[p] = bits;
        }
        return o;
    }
};

template <>
struct FqType<bf16_t> : Fq16 {
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {  // two round-to-nearest-even conversions
        typedef float f2_t __attribute__((ext_vector_type(2)));
        typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){lo, hi}, b2_t));
    }
    static __device__ __forceinline__ float low(uint32_t d) { return __uint_as_float(d << 16); }
    static __device__ __forceinline__ float high(uint32_t d) { return __uint_as_float(d & 0xffff0000u); }
    static __device__ __forceinline__ float rnd(float x) { return low(pack2(x, x)); }
    static __device__ __forceinline__ Raw load(const bf16_t *p, bool vec, int valid) {
        return load_bits(reinterpret_cast<const uint16_t *>(p), vec, valid);
    }
    static __device__ __forceinline__ void store(bf16_t *p, const Raw &r, bool vec, int valid) {
        store_bits(reinterpret_cast<uint16_t *>(p), r, vec, valid);
    }
    static __device__ __forceinline__ float get(const Raw &r, int i) {
        return (i & 1) ? high(r.d[i >> 1]) : low(r.d[i >> 1]);
    }
    static __device__ __forceinline__ void set(Raw &r, int i, float v) {
        const uint32_t h = pack2(v, v) & 0xffffu;
        r.d[i >> 1] = (i & 1) ? ((r.d[i >> 1] & 0x0000ffffu) | (h << 16)) : ((r.d[i >> 1] & 0xffff0000u) | h);
    }
    // a clamp that hands a NaN through, as torch's does
    static __device__ __forceinline__ float clamp(float r, float qmax) { return r < -qmax ? -qmax : (r > qmax ? qmax : r); }
    // RN_bf16(w / s) from w * (1/s): the quotient of two 8-bit significands is never an odd multiple of
    // half a bf16 step (times s that would need more than 8 bits for w) and stays 2^-17 (relative)
    // away from one, the product is off by less than 2^-22.
    static __device__ __forceinline__ float one(float w, float s, float qmax) {
        float r = clamp(rnd(w * __builtin_amdgcn_rcpf(s)), qmax);
        r = rintf(rnd(r - 0.5f)) + 0.5f;  // exact in bf16 for |r| <= 8.5
        return rnd(r * s);
    }
    static __device__ __forceinline__ void absmax(const Raw &v, const ChunkMap &cm, uint32_t &ma, uint32_t &mb) {
        absmax_bits(v, cm, ma, mb);
        ma <<= 16;
        mb <<= 16;
    }
    static __device__ __forceinline__ Raw all(const Raw &w, const ChunkMap &cm, float sa, float sb, float qmax, int ste) {
        const float rsa = __builtin_amdgcn_rcpf(sa), rsb = __builtin_amdgcn_rcpf(sb);
        Raw o;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const bool a0 = (cm.in_a >> (2 * p)) & 1u, a1 = (cm.in_a >> (2 * p + 1)) & 1u;
            const float s0 = a0 ? sa : sb, s1 = a1 ? sa : sb;
            const float w0 = low(w.d[p]), w1 = high(w.d[p]);
            uint32_t r = pack2(w0 * (a0 ? rsa : rsb), w1 * (a1 ? rsa : rsb));
            r = pack2(clamp(low(r), qmax) - 0.5f, clamp(high(r), qmax) - 0.5f);
            const uint32_t q = pack2((rintf(low(r)) + 0.5f) * s0, (rintf(high(r)) + 0.5f) * s1);
            uint32_t bits = select_bits(pair_mask(cm.cherry, p), w.d[p], q);
            if (ste) {
                bits = pack2(low(bits) - w0, high(bits) - w1);
                bits = pack2(low(bits) + w0, high(bits) + w1);
            }
            o.d[p] = bits;
        }
        return o;
    }
};

template <>
struct FqType<float> {
    struct Raw { float v[8]; };
    static __device__ __forceinline__ float rnd(float x) { return x; }
    static __device__ __forceinline__ Raw load(const float *p, bool vec, int valid) {
        Raw r;
        if (vec) {
            const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
            r.v[0] = a.x, r.v[1] = a.y, r.v[2] = a.z, r.v[3] = a.w, r.v[4] = b.x, r.v[5] = b.y, r.v[6] = b.z, r.v[7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) r.v[i] = i < valid ? p[i] : 0.f;
        }
        return r;
    }
    static __device__ __forceinline__ void store(float *p, const Raw &r, bool vec, int valid) {
        if (vec) {
            *reinterpret_cast<float4 *>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
            *reinterpret_cast<float4 *>(p + 4) = make_float4(r.v[4], r.v[5], r.v[6], r.v[7]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (i < valid) p[i] = r.v[i];
        }
    }
    static __device__ __forceinline__ float get(const Raw &r, int i) { return r.v[i]; }
    static __device__ __forceinline__ void set(Raw &r, int i, float v) { r.v[i] = v; }
    // fp32 weights: the correctly rounded division, as torch's
    static __device__ __forceinline__ float one(float w, float s, float qmax) {
        float r = w / s;
        r = fminf(fmaxf(r, -qmax), qmax);
        r = rintf(r - 0.5f) + 0.5f;
        return r * s;
    }
    static __device__ __forceinline__ void absmax(const Raw &v, const ChunkMap &cs, uint32_t &ma, uint32_t &mb) {
        ma = 0, mb = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t a = __float_as_uint(v.v[i]) & 0x7fffffffu & ~bit_mask(cs.cherry, i);
            const uint32_t ina = bit_mask(cs.in_a, i);
            ma = max(ma, a & ina);
            mb = max(mb, a & ~ina);
        }
    }
    static __device__ __forceinline__ Raw all(const Raw &w, const ChunkMap &cs, float sa, float sb, float qmax, int ste) {
        Raw o;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float s = __uint_as_float(select_bits(bit_mask(cs.in_a, i), __float_as_uint(sa), __float_as_uint(sb)));
            float q = __uint_as_float(select_bits(bit_mask(cs.cherry, i), __float_as_uint(w.v[i]),
                                                  __float_as_uint(one(w.v[i], s, qmax))));
            if (ste) q = (q - w.v[i]) + w.v[i];
            o.v[i] = q;
        }
        return o;
    }
};

// The cherry mask of a layer and the count of cherries before each of its words; returns all of them.
// s_scan: one word per wavefront of the workgroup.
__device__ __forceinline__ int cherry_mask(const int32_t *__restrict__ idx, int C, int K, int words, uint32_t *s_mask,
                                           uint32_t *s_pre, uint32_t *s_scan) {
    const int t = threadIdx.x, nt = blockDim.x, lane = t & 63, wave = t >> 6;
    for (int i = t; i < words; i += nt) s_mask[i] = 0;
    __syncthreads();
    for (int m = t; m < C; m += nt) {
        const int j = idx[m];
        if (j >= 0 && j < K) atomicOr(&s_mask[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    // exclusive prefix of the words' popcounts: `per` words a thread, then over lanes and wavefronts
    const int per = ceil_div(words, nt);
    uint32_t mine = 0;
    for (int i = 0; i < per; i++)
        if (t * per + i < words) mine += __popc(s_mask[t * per + i]);
    uint32_t incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
    }
    if (lane == 63) s_scan[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int v = 0; v < nt / 64; v++) {
        if (v < wave) before += s_scan[v];
        all += s_scan[v];
    }
    uint32_t run = before + incl - mine;
    for (int i = 0; i < per; i++) {
        const int wd = t * per + i;
        if (wd < words) {
            s_pre[wd] = run;
            run += __popc(s_mask[wd]);
        }
    }
    __syncthreads();
    return (int)all;
}

// `w` and `out` may be the same buffer in both kernels: a row (a chunk) is read before it is written
// and not again afterwards.

// Dynamic LDS: mask and prefix words (K / 32 each), 16 words for the scan, then three buffers of group
// maxima: row i folds into buffer i % 3 and clears, after the barrier behind which everyone
// has read row i - 1's, the one that row i + 2 will use, so one barrier a row is enough.
// AHEAD: the next row is requested before the barrier (8 chunks a thread leave no registers for it).
template <typename T, int CH, bool AHEAD>
__global__ __launch_bounds__(1024) void fake_quant_row_kernel(const T *w, const int32_t *__restrict__ idx, T *out, int K,
                                                              int N, int C, int G, int bits, int ste) {
    using F = FqType<T>;
    using Raw = typename F::Raw;
    extern __shared__ uint32_t lds[];
    const int t = threadIdx.x, nt = blockDim.x, words = ceil_div(K, 32), chunks = K / 8;
    uint32_t *s_mask = lds, *s_pre = lds + words, *s_scan = s_pre + words, *s_grp = s_scan + 16;
    const int Kn = K - cherry_mask(idx, C, K, words, s_mask, s_pre, s_scan);
    const int groups = ceil_div(Kn, G), last_group = max(groups - 1, 0), stride = last_group + 1;
    for (int g = t; g < 3 * stride; g += nt) s_grp[g] = 0;

    ChunkMap cm[CH];
    int ga[CH], gb[CH];
#pragma unroll
    for (int i = 0; i < CH; i++) {
        const int c = t + i * nt, j0 = 8 * min(c, chunks - 1);
        const uint32_t word = s_mask[j0 >> 5];
        const int pos = j0 - (int)s_pre[j0 >> 5] - __popc(word & ((1u << (j0 & 31)) - 1u));
        cm[i].cherry = (word >> (j0 & 31)) & 0xffu;
        ga[i] = min(pos / G, last_group);  // a chunk of trailing cherries has no group
        gb[i] = min(ga[i] + 1, last_group);
        int room = max((ga[i] + 1) * G - pos, 0);
        cm[i].in_a = 0;
        for (int e = 0; e < 8; e++) {
            if ((cm[i].cherry >> e) & 1u) continue;
            if (room-- > 0) cm[i].in_a |= 1u << e;
        }
    }
    const float half_levels = (float)(1 << (bits - 1)), inv = 1.f / half_levels;
    const float qmax = F::rnd((float)((double)(1 << (bits - 1)) - 1e-2));
    auto scale = [&](uint32_t m) { return F::rnd(F::rnd(__uint_as_float(m) + 1e-6f) * inv); };  // inv: a power of two
    __syncthreads();

    Raw v[CH];
    auto load = [&](Raw (&r)[CH], int n) {
        const T *wr = w + (size_t)n * K;
#pragma unroll
        for (int i = 0; i < CH; i++)
            if (t + i * nt < chunks) r[i] = F::load(wr + 8 * (t + i * nt), true, 8);
    };
    if (AHEAD) load(v, blockIdx.x);
    uint32_t *cur = s_grp, *spare = s_grp + 2 * stride;
    for (int n = blockIdx.x; n < N; n += gridDim.x) {
        if (!AHEAD) load(v, n);
        if (CH >= 4) {  // the maps stay 2 registers a chunk: their masks are formed anew in every row
#pragma unroll
            for (int i = 0; i < CH; i++) asm volatile("" : "+v"(cm[i].cherry), "+v"(cm[i].in_a));
        }
#pragma unroll
        for (int i = 0; i < CH; i++) {
            if (t + i * nt < chunks) {
                uint32_t ma, mb;
                F::absmax(v[i], cm[i], ma, mb);
                atomicMax(&cur[ga[i]], ma);
                if (cm[i].in_a != 0xffu) atomicMax(&cur[gb[i]], mb);
            }
        }
        Raw ahead[CH];
        if (AHEAD && n + (int)gridDim.x < N) load(ahead, n + gridDim.x);
        __syncthreads();
        T *orow = out + (size_t)n * K;
#pragma unroll
        for (int i = 0; i < CH; i++) {
            if (t + i * nt < chunks) {
                const float sa = scale(cur[ga[i]]), sb = scale(cur[gb[i]]);
                F::store(orow + 8 * (t + i * nt), F::all(v[i], cm[i], sa, sb, qmax, ste), true, 8);
            }
        }
        for (int g = t; g < stride; g += nt) spare[g] = 0;
        uint32_t *last = cur;
        cur = cur == s_grp + 2 * stride ? s_grp : cur + stride;
        spare = last;
        if (AHEAD) {
#pragma unroll
            for (int i = 0; i < CH; i++) v[i] = ahead[i];
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kFqThreads) void fake_quant_element_kernel(const T *w, const int32_t *__restrict__ idx, T *out,
                                                                       int K, int N, int C, int G, int bits, int ste,
                                                                       int vec_ok) {
    using F = FqType<T>;
    using Raw = typename F::Raw;
    __shared__ uint32_t s_mask[kFqMaxWords];  // bit j & 31 of word j >> 5: column j is a cherry
    __shared__ uint32_t s_pre[kFqMaxWords];   // cherries in the words before
    __shared__ uint32_t s_grp[kFqMaxGroups];  // per group: max |w| as float bits, then the scale
    __shared__ uint32_t s_scan[kFqThreads / 64];
    const int t = threadIdx.x;
    const int Kn = K - cherry_mask(idx, C, K, ceil_div(K, 32), s_mask, s_pre, s_scan);
    const int groups = ceil_div(Kn, G);

    const float half_levels = (float)(1 << (bits - 1));
    const float qmax = F::rnd((float)((double)(1 << (bits - 1)) - 1e-2));
    const int chunks = ceil_div(K, 8);
    const int last_group = max(groups - 1, 0);

    // compacted position of column j0 (a multiple of 8) and the cherry bits of its chunk
    auto locate = [&](int j0, uint32_t &cherry) {
        const uint32_t word = s_mask[j0 >> 5];
        cherry = (word >> (j0 & 31)) & 0xffu;
        return j0 - (int)s_pre[j0 >> 5] - __popc(word & ((1u << (j0 & 31)) - 1u));
    };

    for (int n = blockIdx.x; n < N; n += gridDim.x) {
        const T *wr = w + (size_t)n * K;
        T *orow = out + (size_t)n * K;
        for (int g = t; g < groups; g += kFqThreads) s_grp[g] = 0;
        __syncthreads();

        // ---- pass 1: group maxima
        for (int c = t; c < chunks; c += kFqThreads) {
            const int j0 = 8 * c;
            const int valid = min(8, K - j0);
            const Raw v = F::load(wr + j0, vec_ok, valid);
            uint32_t cherry;
            int pos = locate(j0, cherry);
            if (cherry == (valid == 8 ? 0xffu : ((1u << valid) - 1u))) continue;  // cherries only
            int g = pos / G;
            int bound = (g + 1) * G;
            uint32_t mx = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (i >= valid || ((cherry >> i) & 1u)) continue;
                if (pos >= bound) {
                    atomicMax(&s_grp[g], mx);
                    mx = 0;
                    do {
                        g++;
                        bound += G;
                    } while (pos >= bound);
                }
                mx = max(mx, __float_as_uint(fabsf(F::get(v, i))));
                pos++;
            }
            atomicMax(&s_grp[g], mx);
        }
        __syncthreads();
        for (int g = t; g < groups; g += kFqThreads) {
            const float a = F::rnd(__uint_as_float(s_grp[g]) + 1e-6f);
            s_grp[g] = __float_as_uint(F::rnd(a / half_levels));
        }
        __syncthreads();

        // ---- pass 2: quantise-dequantise, write
        for (int c = t; c < chunks; c += kFqThreads) {
            const int j0 = 8 * c;
            const int valid = min(8, K - j0);
            const Raw v = F::load(wr + j0, vec_ok, valid);
            uint32_t cherry;
            int pos = locate(j0, cherry);
            int g = min(pos / G, last_group);
            int bound = (g + 1) * G;
            float s = groups > 0 ? __uint_as_float(s_grp[g]) : 1.f;
            Raw o = v;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float wv = F::get(v, i);
                float ov = wv;
                if (i < valid && !((cherry >> i) & 1u)) {
                    if (pos >= bound) {
                        do {
                            g++;
                            bound += G;
                        } while (pos >= bound);
                        s = __uint_as_float(s_grp[g]);
                    }
                    ov = F::one(wv, s, qmax);
                    pos++;
                }
                // the straight-through expression is evaluated on cherry channels too
                if (ste) ov = F::rnd(F::rnd(ov - wv) + wv);
                F::set(o, i, ov);
            }
            F::store(orow + j0, o, vec_ok, valid);
        }
        // the next row clears s_grp: not before every thread has read its scales
        __syncthreads();
    }
}

template <typename T>
static hipError_t launch_fake_quant_t(int bits, const T *w, const int32_t *idx, T *out, int K, int N, int C, int G,
                                      int ste, hipStream_t stream) {
    // 16-byte accesses need whole chunks and 16-byte aligned rows; anything else goes element-wise
    const int vec_ok = K % 8 == 0 && ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (!(vec_ok && G >= 8)) {
        hipLaunchKernelGGL(fake_quant_element_kernel<T>, dim3(min(N, 256 * 4)), dim3(kFqThreads), 0, stream, w, idx, out, K,
                           N, C, G, bits, ste, vec_ok);
        return hipGetLastError();
    }
    // as few chunks a thread as keep a row within one workgroup: two where there are enough of them that
    // a workgroup has its four wavefronts, so that two loads a lane are in flight
    const int chunks = K / 8;
    const int ch = chunks <= 256 ? 1 : chunks <= 2048 ? 2 : chunks <= 4096 ? 4 : 8;
    const int threads = ceil_div(ceil_div(chunks, ch), 64) * 64;
    const size_t lds = (size_t)(2 * ceil_div(K, 32) + 16 + 3 * ceil_div(K, G)) * 4;
    const dim3 grid((unsigned)min(N, 256 * max(1, 2048 / threads)));  // every compute unit filled once, workgroups walk rows
#define CQ_FQ(CH_, AHEAD_)                                                                                           \
    hipLaunchKernelGGL((fake_quant_row_kernel<T, CH_, AHEAD_>), grid, dim3(threads), lds, stream, w, idx, out, K, N, C, G, \
                       bits, ste)
    if (ch == 1) CQ_FQ(1, true);
    else if (ch == 2) CQ_FQ(2, true);
    else if (ch == 4) CQ_FQ(4, true);
    else CQ_FQ(8, false);
#undef CQ_FQ
    return hipGetLastError();
}

hipError_t launch_fake_quant(int bits, FqDtype dtype, const void *w, const int32_t *idx, void *out, int K, int N, int C,
                             int G, int ste, hipStream_t stream) {
    if (dtype == FqDtype::f32)
        return launch_fake_quant_t<float>(bits, reinterpret_cast<const float *>(w), idx,
                                          reinterpret_cast<float *>(out), K, N, C, G, ste, stream);
    if (dtype == FqDtype::bf16)
        return launch_fake_quant_t<bf16_t>(bits, reinterpret_cast<const bf16_t *>(w), idx,
                                           reinterpret_cast<bf16_t *>(out), K, N, C, G, ste, stream);
    return launch_fake_quant_t<__half>(bits, reinterpret_cast<const __half *>(w), idx,
                                       reinterpret_cast<__half *>(out), K, N, C, G, ste, stream);
}

}  // namespace cq
