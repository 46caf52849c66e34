// 3-bit fused dequant + matmul on fp32 tensors (fp32 activations, scales, cherry rows and
// outputs, int32 channel indices): the variant behind vecquant3matmul_cherryq(..., fp16=False),
// the call the reference's benchmark_speed.py:20-45 times (batch 16, 4096 -> 13824).
//
// fp32 products on the fp16 matrix cores, exactly: a code minus 3.5 is a 4-bit number, and an fp32 activation is the
// sum of three fp16 numbers (11 + 11 + 2 of its 24 bits, split by truncation after its row of the unit has
// been scaled to the top of the fp16 range by a power of two), so that three v_mfma_f32_16x16x32_f16 form the products
// the fp32 instruction forms, without rounding, into the same fp32 accumulators, at 16 times its
// rate per instruction.  (On v_mfma_f32_16x16x4_f32 the call was bound by that instruction: 43 us plus 5 us of
// activation preparation at 4096 -> 13824 with 16 rows; now 16 + 4, the packed bytes at 1.6 TB/s.)
//
//   * A workgroup of 8 wavefronts owns 64 columns and, where there are enough columns to fill the chip, all of
//     K, so no partial results leave it; a wavefront takes units of 128 compacted positions in turn.  Four lane
//     groups split each 32 positions, a lane owns 4 adjacent columns and loads dwords: 64 bytes of each byte row.
//     Neighbouring tiles share 128-byte lines; they run on the same XCD.
//   * B operands from registers: two v_perm_b32 collect a column's three bytes of 8 positions, masks cut out code
//     pairs, OR-ing 0x6400 makes them the fp16 numbers 1024 + u * 2^p, one packed fma turns that into u - 3.5
//     (code 0's field is first moved from bit 0 to bit 1: 1024 + 3.5 has no fp16 value).
//   * A operands come from a small kernel in front (gathered around the cherry channels, split, in the per-lane operand
//     order, zero padded to 16 rows): contiguous 1 KB loads.  Splitting the rows in every workgroup instead cost as
//     much vector work as the decode and scattered 16-byte requests: 22 us against 4 + 16 at that shape.
//   * At every group end the tile is multiplied by the group's scale and the row's power of two and added to the
//     totals, which is where the reference applies the scale too (csrc/quant_cuda_kernel.cu:312).
//   * Cherry rows are fp32 times fp32: v_mfma_f32_16x16x4_f32.
//
// Where columns are few, K is split over workgroups and the totals meet in one 64-bit fixed-point atomic per output
// element (cq_device.h).  Up to 16 rows per pass; more rows are further passes over the weights.
//
// Arithmetic contract: csrc/quant_cuda_kernel.cu:191-314 (group 64) and 441-556 (group 128):
// fp32 products and sums; the summation order differs (the reference adds 64 or 128 products in
// sequence per thread and combines blocks with fp32 atomics in arrival order).
#include "cq_device.h"
#include "cq_kernels.h"

namespace cq {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kF32Rows = 16;   // MFMA M dimension; smaller batches are zero padded
constexpr int kF32Waves = 8;  // wavefronts per workgroup
constexpr int kF32Cols = 64;   // columns per workgroup
constexpr int kF32Staged = 4096;  // cherry channels held in LDS while the offsets are found
constexpr uint32_t kRsrcFlagsF = 0x00020000u;
constexpr uint32_t kOobF = 0x80000000u;

// position order inside the 8 positions a lane contributes to one MFMA (cq_batch.hip), and the bit at which each
// code's field sits when 0x6400 is OR-ed in
__host__ __device__ constexpr int f32_ord(int kk) { return (int)((0x72654130u >> (4 * kk)) & 7u); }

struct F32Scratch {  // byte offsets
    size_t down, cherry, total;
};
// parts: per unit and step of 32 positions, three parts of 64 lanes x 16 bytes; down: what undoes the scaling, per
// unit and row; cherry: the rows at the cherry channels, [channel][row], padded to whole steps of 4
static F32Scratch f32_scratch(int K, int C) {
    F32Scratch s;
    const size_t units = ceil_div(K - C, kUnitK);
    s.down = units * 4 * 3 * 64 * 16;
    s.cherry = s.down + units * kF32Rows * sizeof(float);
    s.total = (s.cherry + (size_t)ceil_div(C, 4) * 4 * kF32Rows * sizeof(float) + 255) / 256 * 256;
    return s;
}
size_t f32_scratch_bytes(int K, int C) { return f32_scratch(K, C).total; }

// ---- activation preparation ------------------------------------------------------------------------
// One workgroup per unit (thread = step s, lane (q, i): positions 128 u + 32 s + 8 q + ord[0..7] of row i), further ones
// for the cherry channels.
__global__ __launch_bounds__(256) void f32_prep_kernel(const float *__restrict__ x, const int32_t *__restrict__ cherry_indices,
                                                       u32x4 *__restrict__ parts, float *__restrict__ down,
                                                       float *__restrict__ cherry, int B, int K, int C, int units) {
    const int t = threadIdx.x;
    if ((int)blockIdx.x >= units) {
        const int e = ((int)blockIdx.x - units) * 256 + t, c = e / kF32Rows, i = e % kF32Rows;
        if (c < ceil_div(C, 4) * 4) cherry[e] = c < C && i < B ? x[(size_t)i * K + cherry_indices[c]] : 0.f;
        return;
    }
    __shared__ unsigned s_max[kF32Rows];
    __shared__ int s_t[kF32Staged];
    const int u = blockIdx.x, s = t >> 6, lane = t & 63, q = lane >> 4, i = lane & 15, Kn = K - C;
    if (t < kF32Rows) s_max[t] = 0;
    // idx[m] - m: position k sits behind every cherry m with idx[m] - m <= k
    const int staged = min(C, kF32Staged);
    for (int m = t; m < staged; m += 256) s_t[m] = cherry_indices[m] - m;
    __syncthreads();
    auto offset = [&](int m) { return m < staged ? s_t[m] : cherry_indices[m] - m; };
    const int k0 = u * kUnitK + 32 * s + 8 * q;
    int lo = 0, hi = C;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (offset(mid) <= k0) lo = mid + 1; else hi = mid;
    }
    const bool ok = k0 < Kn && i < B;
    float v[8];
    unsigned mx = 0;
    int next = lo < C ? offset(lo) : 0x7fffffff;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        while (next <= k0 + j) next = ++lo < C ? offset(lo) : 0x7fffffff;
        v[j] = ok ? x[(size_t)i * K + k0 + j + lo] : 0.f;
        mx = max(mx, __float_as_uint(v[j]) & 0x7fffffffu);
    }
    atomicMax(&s_max[i], mx);
    __syncthreads();
    // 2^shift brings the row's largest |x| of the unit into [2^14, 2^15)
    const int shift = min(141 - (int)(s_max[i] >> 23), 126);
    const float up = ldexpf(1.f, shift);
    uint32_t part[3][4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        float t0 = v[f32_ord(2 * p)] * up, t1 = v[f32_ord(2 * p + 1)] * up;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const half2_t h = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(t0, t1));
            part[k][p] = __builtin_bit_cast(uint32_t, h);
            t0 -= (float)h[0];
            t1 -= (float)h[1];
            if (!(fabsf(t0) < __builtin_inff())) t0 = 0.f;  // an infinity or a NaN is one part
            if (!(fabsf(t1) < __builtin_inff())) t1 = 0.f;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        parts[((size_t)(u * 4 + s) * 3 + k) * 64 + lane] = (u32x4){part[k][0], part[k][1], part[k][2], part[k][3]};
    if (t < kF32Rows) down[u * kF32Rows + t] = ldexpf(1.f, -min(141 - (int)(s_max[t] >> 23), 126));
}

// ---- main kernel -----------------------------------------------------------------------------------
struct F32Ctx {
    __amdgpu_buffer_rsrc_t rw, rs, rc;
    const u32x4 *parts;
    const float *down, *cherry;
    int N, Kn, C, G, kq, nl, n0;
    bool col_ok;
};

struct F32Unit {
    uint32_t w[12];   // 4 steps x 3 byte rows, 4 columns each
    u32x4 a[12];      // 4 steps x 3 parts
    u32x4 sc;         // whole groups: the group's scales of the 4 columns
    float4 down;      // of the 4 rows this lane accumulates
};

template <bool WHOLE>
__device__ __forceinline__ void f32_issue(F32Unit &r, const F32Ctx &cx, int u, int lane) {
    const uint32_t woff = cx.col_ok ? (uint32_t)((u * 48 + cx.kq * 3) * cx.N + cx.n0) : kOobF;
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int b = 0; b < 3; b++)
            r.w[3 * s + b] = __builtin_amdgcn_raw_buffer_load_b32(cx.rw, woff + (uint32_t)((12 * s + b) * cx.N), 0, 2);
    const u32x4 *pa = cx.parts + (size_t)u * 12 * 64 + lane;
#pragma unroll
    for (int i = 0; i < 12; i++) r.a[i] = pa[i * 64];
    if (WHOLE)
        r.sc = __builtin_amdgcn_raw_buffer_load_b128(
            cx.rs, cx.col_ok ? (uint32_t)(u * kUnitK / cx.G * cx.N + cx.n0) * 4u : kOobF, 0, 0);
    r.down = *reinterpret_cast<const float4 *>(cx.down + u * kF32Rows + 4 * cx.kq);
}

// WHOLE: groups are whole units
template <bool WHOLE>
__device__ __forceinline__ void f32_compute(const F32Unit &r, const F32Ctx &cx, int u, float4_t (&tot)[4]) {
    // one literal an instruction at most, and none in the three-operand forms: the constants of the decode live in
    // registers, so that mask and OR are one v_and_or_b32
    uint32_t one, m0, m1, m2, m3, m4;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(one));
    asm("s_mov_b32 %0, 0x001c000e" : "=s"(m0));
    asm("s_mov_b32 %0, 0x00700038" : "=s"(m1));
    asm("s_mov_b32 %0, 0x001c0380" : "=s"(m2));
    asm("s_mov_b32 %0, 0x000001c0" : "=s"(m3));
    asm("s_mov_b32 %0, 0x00e00000" : "=s"(m4));
    const float down[4] = {r.down.x, r.down.y, r.down.z, r.down.w};
    float4_t d[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        u32x4 sc = r.sc;
        const bool ends = WHOLE ? s == 3 : (s == 3 || (u * kUnitK + 32 * (s + 1)) % cx.G == 0);
        const bool begins = WHOLE ? s == 0 : (s == 0 || (u * kUnitK + 32 * s) % cx.G == 0);
        if (!WHOLE && ends)
            sc = __builtin_amdgcn_raw_buffer_load_b128(
                cx.rs, cx.col_ok ? (uint32_t)((u * kUnitK + 32 * s) / cx.G * cx.N + cx.n0) * 4u : kOobF, 0, 0);
        // B: 8 codes minus 3.5 of each of the lane's columns.  Fields: codes (0, 3) at bits 1, 2 (moved up by one);
        // (1, 4) at 3, 4; (5, 6) at 7, 2; (2, 7) at 6, 5
        u32x4 bv[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t sel = 0x0c000000u | (uint32_t)(c << 16) | (uint32_t)(c << 8) | (uint32_t)(4 + c);
            const uint32_t p1 = __builtin_amdgcn_perm(r.w[3 * s], r.w[3 * s + 1], sel);
            const uint32_t p2 = __builtin_amdgcn_perm(r.w[3 * s + 1], r.w[3 * s + 2], sel);
            const uint32_t f[4] = {((p1 << 1) & m0) | one, (p1 & m1) | one, (p2 & m2) | one, (p2 & m4) | ((p1 & m3) | one)};
#define CQ_CODES(i, a, b)                                                                                                  \
    bv[c][i] = __builtin_bit_cast(                                                                                         \
        uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2_t, f[i]),                                             \
                                            (half2_t){(_Float16)(1.f / (1 << a)), (_Float16)(1.f / (1 << b))},             \
                                            (half2_t){(_Float16)(-(1024.f / (1 << a) + 3.5f)), (_Float16)(-(1024.f / (1 << b) + 3.5f))}))
            CQ_CODES(0, 1, 2);
            CQ_CODES(1, 3, 4);
            CQ_CODES(2, 7, 2);
            CQ_CODES(3, 6, 5);
#undef CQ_CODES
        }
        if (begins)
#pragma unroll
            for (int c = 0; c < 4; c++) d[c] = (float4_t){0.f, 0.f, 0.f, 0.f};
        // the small parts first; consecutive MFMAs go to different accumulators
#pragma unroll
        for (int k = 2; k >= 0; k--)
#pragma unroll
            for (int c = 0; c < 4; c++)
                d[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, r.a[3 * s + k]),
                                                              __builtin_bit_cast(half8_t, bv[c]), d[c], 0, 0, 0);
        if (ends)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int q = 0; q < 4; q++) tot[c][q] += __uint_as_float(sc[c]) * (d[c][q] * down[q]);
    }
}

struct F32Plan {
    int tiles, per_xcd;             // tiles of 64 columns; tiles an XCD takes in sequence
    int units;                      // of 128 positions
    int splits, units_per_wg;
};

template <bool WHOLE>
__global__ __launch_bounds__(64 * kF32Waves, 2) void f32_kernel(const uint8_t *__restrict__ qweight,
                                                               const float *__restrict__ cherry_weight,
                                                               const float *__restrict__ scales, const u32x4 *__restrict__ parts,
                                                               const float *__restrict__ down, const float *__restrict__ cherry,
                                                               float *__restrict__ mul,
                                                               unsigned long long *__restrict__ acc_words,
                                                               float *__restrict__ side, int B, int K, int N, int C, int G,
                                                               int accumulate, F32Plan plan) {
    __shared__ float s_red[kF32Waves][kF32Rows][kF32Cols];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int split = blockIdx.x / (8 * plan.per_xcd), slot = blockIdx.x % (8 * plan.per_xcd);
    const int tile = (slot & 7) * plan.per_xcd + (slot >> 3);  // consecutive workgroups go to different XCDs
    if (tile >= plan.tiles) return;

    F32Ctx cx;
    cx.N = N, cx.Kn = K - C, cx.C = C, cx.G = G;
    cx.kq = lane >> 4, cx.nl = lane & 15;
    cx.n0 = tile * kF32Cols + 4 * cx.nl;
    cx.col_ok = cx.n0 < N;
    cx.parts = parts, cx.down = down, cx.cherry = cherry;
    cx.rw = __builtin_amdgcn_make_buffer_rsrc((void *)qweight, 0, cx.Kn / 8 * 3 * N, kRsrcFlagsF);
    cx.rs = __builtin_amdgcn_make_buffer_rsrc((void *)scales, 0, ceil_div(cx.Kn, G) * N * 4, kRsrcFlagsF);
    cx.rc = __builtin_amdgcn_make_buffer_rsrc((void *)cherry_weight, 0, C * N * 4, kRsrcFlagsF);

    // Requested in the order of use: the first two units, four cherry rows (they are dealt to all wavefronts of all
    // splits, one a lane group), what the output already holds.
    const int u0 = split * plan.units_per_wg + wave, u_end = min((split + 1) * plan.units_per_wg, plan.units);
    F32Unit a, b;
    if (u0 < u_end) f32_issue<WHOLE>(a, cx, u0, lane);
    if (u0 + kF32Waves < u_end) f32_issue<WHOLE>(b, cx, u0 + kF32Waves, lane);
    const int steps = ceil_div(C, 4), step0 = split * kF32Waves + wave;
    auto cherry_row = [&](int step, float &x, u32x4 &w) {
        const int c = 4 * step + cx.kq;
        x = cherry[c * kF32Rows + cx.nl];
        w = __builtin_amdgcn_raw_buffer_load_b128(cx.rc, c < C && cx.col_ok ? (uint32_t)(c * N + cx.n0) * 4u : kOobF, 0, 0);
    };
    float cx0 = 0.f;
    u32x4 cw0 = {0u, 0u, 0u, 0u};
    if (step0 < steps) cherry_row(step0, cx0, cw0);
    constexpr int RPT = kF32Rows / kF32Waves;  // rows a thread finishes
    const int first = wave * RPT, n = tile * kF32Cols + lane;
    float before[RPT];
#pragma unroll
    for (int q = 0; q < RPT; q++)
        before[q] = accumulate && plan.splits == 1 && n < N && first + q < B ? mul[(size_t)(first + q) * N + n] : 0.f;

    // tot[c][r]: column n0 + c, batch row 4 * kq + r
    float4_t tot[4];
#pragma unroll
    for (int c = 0; c < 4; c++) tot[c] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma nounroll
    for (int u = u0; u < u_end; u += 2 * kF32Waves) {
        f32_compute<WHOLE>(a, cx, u, tot);
        if (u + 2 * kF32Waves < u_end) f32_issue<WHOLE>(a, cx, u + 2 * kF32Waves, lane);
        if (u + kF32Waves >= u_end) break;
        f32_compute<WHOLE>(b, cx, u + kF32Waves, tot);
        if (u + 3 * kF32Waves < u_end) f32_issue<WHOLE>(b, cx, u + 3 * kF32Waves, lane);
    }
    for (int step = step0; step < steps; step += kF32Waves * plan.splits) {
        if (step != step0) cherry_row(step, cx0, cw0);
#pragma unroll
        for (int c = 0; c < 4; c++)
            tot[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(cx0, __uint_as_float(cw0[c]), tot[c], 0, 0, 0);
    }

    // across the wavefronts
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4 *>(&s_red[wave][4 * cx.kq + r][4 * cx.nl]) =
            make_float4(tot[0][r], tot[1][r], tot[2][r], tot[3][r]);
    __syncthreads();
    float vals[RPT][1];
#pragma unroll
    for (int q = 0; q < RPT; q++) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kF32Waves; w++) v += s_red[w][first + q][lane];
        vals[q][0] = v + before[q];
    }
    splitk_finish<float, RPT, 1>(vals, B - first, N, n, n < N, plan.splits, acc_words + (size_t)first * N,
                                 mul + (size_t)first * N, accumulate && plan.splits > 1, side + (size_t)first * N);
}

bool f32_supported(int B, int K, int N, int C, int G) {
    if (B < 1) return false;
    if (G % 32) return false;  // an MFMA's 32 positions must not straddle a group
    if (K - C <= 0) return false;
    const long long wbytes = (long long)(K - C) / 8 * 3 * N;
    const long long cbytes = (long long)C * N * 4;
    const long long sbytes = (long long)ceil_div(K - C, G) * N * 4;
    if (wbytes >= 0x7fff0000ll || cbytes >= 0x7fff0000ll || sbytes >= 0x7fff0000ll) return false;
    return true;
}

hipError_t launch_f32(const float *vec, const uint8_t *qweight, const float *cherry_weight,
                      const int32_t *cherry_indices, const float *scales, float *mul, int B, int K, int N, int C,
                      int G, int accumulate, void *workspace, void *scratch, hipStream_t stream) {
    const F32Scratch sc = f32_scratch(K, C);
    u32x4 *parts = reinterpret_cast<u32x4 *>(scratch);
    float *down = reinterpret_cast<float *>(reinterpret_cast<char *>(scratch) + sc.down);
    float *cherry = reinterpret_cast<float *>(reinterpret_cast<char *>(scratch) + sc.cherry);
    F32Plan plan;
    plan.tiles = ceil_div(N, kF32Cols);
    plan.per_xcd = ceil_div(plan.tiles, 8);
    plan.units = ceil_div(K - C, kUnitK);
    // K is split only as far as it takes one workgroup per compute unit, each with a unit for every wavefront
    const int want = min(max(1, 256 / plan.tiles), min(kMaxSplits, ceil_div(plan.units, kF32Waves)));
    plan.units_per_wg = ceil_div(plan.units, want);
    plan.splits = ceil_div(plan.units, plan.units_per_wg);
    auto *const kernel = G % kUnitK == 0 ? f32_kernel<true> : f32_kernel<false>;
    const int prep = plan.units + ceil_div(ceil_div(C, 4) * 4 * kF32Rows, 256);
    for (int b0 = 0; b0 < B; b0 += kF32Rows) {
        const int nb = min(kF32Rows, B - b0);
        hipLaunchKernelGGL(f32_prep_kernel, dim3(prep), dim3(256), 0, stream, vec + (size_t)b0 * K, cherry_indices, parts, down,
                           cherry, nb, K, C, plan.units);
        hipLaunchKernelGGL(kernel, dim3(8 * plan.per_xcd * plan.splits), dim3(64 * kF32Waves), 0, stream, qweight,
                           cherry_weight, scales, parts, down, cherry, mul + (size_t)b0 * N,
                           reinterpret_cast<unsigned long long *>(workspace), splitk_side(workspace, B, N), nb, K, N, C, G,
                           accumulate, plan);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace cq
