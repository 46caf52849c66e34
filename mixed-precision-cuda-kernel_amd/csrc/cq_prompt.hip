// Prompt-sized batches (17 rows and more) over the checkpoint layout: fused dequantise + matrix product.
//
//   Y[M, N] (+)= Xn[M, Kn] * Wn[Kn, N] + Xc[M, C] * Wc[C, N]
//
// Wn are the packed codes, Wc the fp16 cherry rows; Xn / Xc are the activations gathered at the normal / cherry
// input channels.  Bound by the matrix cores for many rows, by the decode (vector ALU) and the weights' bytes for few.
//
// A workgroup of 8 or 4 wavefronts owns an output tile of 16 MT rows x 64, 128 or 256 columns and the wavefronts share K:
// each takes units of 128 positions in turn, so that the main loop has no LDS traffic and no barrier, and partial
// results meet once, in LDS, at the end.  (Wavefronts that share the columns instead need the dequantised weights passed
// through LDS in every step and, where the tiles do not fill the chip, several workgroups' fp32 tiles passed
// through memory: at 4096 -> 11008 with 128 rows those were 28 MB each way, more than the weights.)
//   What a tile shape is bound by: a compute unit reads 44 to 50 bytes a clock from its caches whatever their level, and
// every wavefront fetches its own fragments of the activations, so 64 columns of 128 rows wait for those; 128 columns (NC = 8,
// the fragments feed twice the MFMAs) take 256 accumulator and 200 other registers, one wavefront a SIMD.  Two such
// wavefronts side by side (NS = 2) halve the tile's partial results in LDS and its row tiles' weight reads from the L2.
//   Measured, 4 bits, preparation included, against the kernel of wavefronts side by side that this replaces (us):
//     rows              17      64     128     256     512    1024    2048
//     4096 -> 11008   18.0    21.2    29.2    39.7    64.3     118     196
//             before  22.8    26.8    37.1    51.9    80.0     131     248
//     4096 -> 4096    12.9    16.0    18.5    23.1    33.3    47.7    77.3
//             before  16.7    19.8    25.8    30.2    40.7    60.4    97.8
//     11008 -> 4096   19.5    23.5    32.9    48.3    72.5    99.8     184
//             before  25.4    29.2    37.1    53.3    78.0     132     241
//   At 2048 rows of 4096 -> 11008 that is 0.94 PFLOP/s of 1.4 to 1.5 that a large library product reaches: 87 us are the
// MFMAs at their issue rate, the preparation takes 14, decoding and loads between the MFMAs about 70, the three rounds' prologues
// and reductions about 30.
//   * B operands (weights) go straight from registers to v_mfma_f32_16x16x32_f16: a lane owns 4 adjacent columns
//     (dword loads, 64 bytes of a byte row), lane group kq the 8 positions 8 kq .. 8 kq + 7 of each 32.  v_perm_b32
//     interleaves a column's bytes, masks cut out code pairs, OR-ing 0x6400 makes them the fp16 numbers
//     1024 + u * 2^p, one packed fma gives u - c_b (exact: the fields are first moved up one bit, 1024 + c_b itself has
//     no fp16 value) and one packed multiply applies the group scale with the reference's single rounding, so
//     the operands are the dense weight's values (llama/qlinear.py:120-162).
//   * A operands (activations) come from a small kernel in front, gathered around the cherry channels and in operand
//     order: one contiguous 1 KB load per 16 rows and 32 positions.
//   * Registers are reloaded in place: a step's packed bytes for the wavefront's next unit as soon as they are
//     decoded, a fragment for the next step as soon as its four MFMAs are issued.
// Neighbouring column tiles share 128-byte lines of the packed bytes and a column tile's row tiles share all of them:
// tiles run in XCD-contiguous ranges.
//
// Where there are too few tiles, K is split over workgroups too: fp32 tiles in scratch and one ticket per tile; the last
// workgroup adds them in split order, so the result does not depend on arrival order.
//
// Arithmetic contract: csrc/quant_cuda_kernel.cu:797-834 (the reference loops its batch-1 body over the rows); here
// fp16 weights as the dense path's (qlinear.py:183-195), fp32 accumulation, one final rounding.
#include "cq_device.h"
#include "cq_kernels.h"

namespace cq {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// wavefronts of a workgroup: a tile of 128 x 128 leaves registers for one a SIMD, others for two and more
__host__ __device__ constexpr int prompt_waves(int mt, int nc) { return mt * nc == 64 ? 4 : 8; }
// ... of which this many share K where ns of them lie side by side
__host__ __device__ constexpr int prompt_kways(int mt, int nc, int ns) { return prompt_waves(mt, nc) / ns; }
constexpr uint32_t kRsrcFlagsP = 0x00020000u;
constexpr uint32_t kOobP = 0x80000000u;

// Position order inside a lane's 8 positions as the decode produces it (dword d holds kk = 2 d, 2 d + 1), and the bit
// of each code's field in its half after the shift.
//   4-bit: ord = {0, 2, 1, 3, 4, 6, 5, 7}   p = {1, 1, 5, 5, 1, 1, 5, 5}
//   3-bit: ord = {0, 3, 1, 4, 5, 6, 2, 7}   p = {1, 2, 3, 4, 7, 2, 6, 5}
template <int BITS>
__host__ __device__ constexpr int prompt_ord(int kk) {
    return BITS == 4 ? (int)((0x75643120u >> (4 * kk)) & 7u) : (int)((0x72654130u >> (4 * kk)) & 7u);
}
template <int BITS>
__host__ __device__ constexpr int prompt_pos(int kk) {
    return BITS == 4 ? ((kk & 2) ? 5 : 1) : (int)((0x56274321u >> (4 * kk)) & 7u);
}
static_assert(prompt_ord<4>(1) == 2 && prompt_ord<4>(2) == 1 && prompt_ord<4>(5) == 6 && prompt_ord<4>(7) == 7, "");

// What a call takes with one of the tile shapes, in microseconds: a fit to about 4000 measured calls (4 bits, K 1024 to
// 28672, N 512 to 28672, M 17 to 2048, every shape and up to 16 K splits).  `first` is a launch with one round of
// workgroups and no unit, `round` what each further round of 256 adds, `unit` a unit of 128 positions of every wavefront
// (`pair`: of a second workgroup on the same compute unit), `split` and `mbyte` a split call and each megabyte of its
// partial tiles.  On those calls the shape and split chosen by it are 1.4 % slower than the best on average, 22 % at worst.
struct PromptShape {
    int mt, nc, ns;
    float first, round, unit, pair, split, mbyte;
};
constexpr PromptShape kPromptShapes[] = {
    {2, 4, 1, 5.65f, 0.91f, 2.66f, 2.15f, 2.60f, 0.74f},   // 32 x 64: two workgroups a compute unit
    {4, 4, 1, 6.00f, 2.04f, 3.32f, 0.f, 3.58f, 0.48f},     // 64 x 64
    {8, 4, 1, 7.11f, 3.64f, 4.71f, 0.f, 5.15f, 0.38f},     // 128 x 64
    {8, 8, 1, 10.63f, 5.90f, 3.04f, 0.f, 8.06f, 0.58f},    // 128 x 128, one wavefront a SIMD
    {8, 8, 2, 10.80f, 3.50f, 2.89f, 0.f, 14.20f, 0.51f},   // 128 x 256, pairs of wavefronts side by side
};

PromptPlan prompt_plan(int M, int K, const int *N, int count, int C) {
    PromptPlan best;
    float best_cost = 3.4e38f;
    const int units = K > C ? ceil_div(K - C, kUnitK) : 1;  // sizes are asked for before the launch is refused
    for (const PromptShape &s : kPromptShapes) {
        if (s.mt > 2 && M <= 8 * s.mt) break;  // half of every tile would be padding
        PromptPlan p;
        p.mt = s.mt, p.nc = s.nc, p.ns = s.ns;
        p.mtiles = ceil_div(M, 16 * s.mt);
        p.ntiles = 0;
        for (int i = 0; i < count; i++) p.ntiles += ceil_div(N[i], 16 * s.nc * s.ns);
        const long long tiles = (long long)p.mtiles * p.ntiles;
        const int kways = prompt_kways(s.mt, s.nc, s.ns);
        for (int splits = 1; splits <= kPromptMaxSplits; splits++) {
            // more splits than one round (two for the small tile) of workgroups or than leave a wavefront a unit never pay
            if (splits > 1 && (tiles * splits > 512 || splits > ceil_div(units, kways))) break;
            p.units_per_split = ceil_div(units, splits);
            p.splits = ceil_div(units, p.units_per_split);
            if (p.splits < splits) continue;  // the same plan as with fewer
            const long long load = (tiles * splits + 255) / 256;
            const float u = (float)ceil_div(p.units_per_split, kways);
            float cost = s.first;
            if (s.pair > 0.f)
                cost += s.round * (float)((load + 1) / 2 - 1) + u * (s.unit * (float)((load + 1) / 2) + s.pair * (float)(load / 2));
            else
                cost += s.round * (float)(load - 1) + u * s.unit * (float)load;
            if (splits > 1) cost += s.split + s.mbyte * (float)(tiles * splits) * (float)(s.mt * s.nc * s.ns * 1024) * 1e-6f;
            if (cost < best_cost) best_cost = cost, best = p;
        }
    }
    PromptPlan &p = best;
    const size_t tiles = (size_t)p.mtiles * p.ntiles;
    p.units = units;
    p.csteps = ceil_div(C, 32);
    p.steps = p.units * 4 + p.csteps;
    p.a_bytes = ((size_t)p.steps * p.mtiles * p.mt * 1024 + 255) / 256 * 256;
    p.partial_bytes = p.splits > 1 ? p.splits * tiles * p.mt * p.nc * p.ns * 256 * sizeof(float) : 0;
    p.scratch_bytes = count * p.a_bytes + p.partial_bytes;
    p.workspace_bytes = (tiles * sizeof(unsigned) + 255) / 256 * 256;
    return p;
}

PromptPlan prompt_plan(int M, int K, int N, int C) { return prompt_plan(M, K, &N, 1, C); }

// ---- activation preparation ------------------------------------------------------------------------
// a[(step * m16 + tile) * 64 + lane], lane = (q, i): x[16 tile + i][positions 32 step + 8 q + ord[0..7]].  A workgroup
// takes one unit (4 steps) of 16 rows: the unit's dense columns are a contiguous range, loaded in whole lines
// into LDS and gathered from there.  Rows >= M and positions past the end read as 0.  Every layer of a group has its own
// cherry channels and so its own copy (blockIdx.z).
// Bound by its chain of round trips, so the rows and the channels are asked for together and a position's offset is
// found once for the 16 rows (99 rows of a 4096 -> 11008 product, both launches: 28.6 -> 27.6 us).
// (The two staged chunks are two variables: as an array the compiler keeps them in LDS, addressed through the dispatch
// packet in host memory, and the launch takes 18 us.)
constexpr int kPrepCols = 256;     // dense columns of a unit that are staged; a wider range is gathered from memory
constexpr int kPrepIdx = 1024;     // cherry channels staged
struct PromptIndices {
    const int16_t *of[kPromptMaxGroup];
};
template <int BITS>
__global__ __launch_bounds__(256) void prompt_prep_kernel(const __half *__restrict__ x, PromptIndices indices, uint4 *__restrict__ a,
                                                          size_t a_bytes, int M, int K, int C, int units, int m16, int wide) {
    __shared__ __attribute__((aligned(16))) uint16_t s_x[16][kPrepCols + 8];
    __shared__ int16_t s_idx[kPrepIdx];
    __shared__ __attribute__((aligned(16))) uint16_t s_off[kUnitK];
    const int t = threadIdx.x, lane = t & 63, q = lane >> 4, i = lane & 15, tile = blockIdx.y, Kn = K - C;
    const int row = 16 * tile + i, layer = blockIdx.z;
    const int16_t *__restrict__ cherry_indices = layer == 0 ? indices.of[0] : layer == 1 ? indices.of[1] : indices.of[2];
    a += layer * (a_bytes / sizeof(uint4));
    unsigned short h[8];
#pragma unroll
    for (int kk = 0; kk < 8; kk++) h[kk] = 0;
    int step;
    if ((int)blockIdx.x >= units) {  // cherry channels
        const int cs = ((int)blockIdx.x - units) * 4 + (t >> 6);
        if (cs >= ceil_div(C, 32)) return;
        step = units * 4 + cs;
        const int c0 = 32 * cs + 8 * q;
        if (c0 < C && row < M) {  // C is a multiple of 8: all eight or none.  One load names them, eight go out together
            typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
            const u32x4_a4 ch = *reinterpret_cast<const u32x4_a4 *>(cherry_indices + c0);
#pragma unroll
            for (int kk = 0; kk < 8; kk++)
                h[kk] = __half_as_ushort(x[(size_t)row * K + ((ch[kk >> 1] >> (16 * (kk & 1))) & 0xffffu)]);
        }
    } else {
        const int u = blockIdx.x, k0 = u * kUnitK, k1 = min(k0 + kUnitK, Kn);
        step = 4 * u + (t >> 6);
        // Wherever the cherries lie, the unit's columns are within the C behind its first position: few cherries, and the rows
        // are asked for before the channels are known, one round trip to memory instead of two.
        const bool near = wide && C <= kPrepCols - kUnitK;
        const int sr = 16 * tile + (t >> 5), sch = t & 31;  // this thread's staged chunks: rows sr and sr + 8
        u32x4 v0 = {0, 0, 0, 0}, v1 = {0, 0, 0, 0};
        const bool chunk = near && sch < ceil_div(k1 - k0 + C, 8);
        if (chunk && sr < M) v0 = *reinterpret_cast<const u32x4 *>(x + (size_t)sr * K + k0 + 8 * sch);
        if (chunk && sr + 8 < M) v1 = *reinterpret_cast<const u32x4 *>(x + (size_t)(sr + 8) * K + k0 + 8 * sch);
        if (C <= kPrepIdx) {
#pragma unroll 1
            for (int m = t; m < C; m += 256) s_idx[m] = cherry_indices[m];
        }
        if (chunk) {
            *reinterpret_cast<u32x4 *>(&s_x[t >> 5][8 * sch]) = v0;
            *reinterpret_cast<u32x4 *>(&s_x[(t >> 5) + 8][8 * sch]) = v1;
        }
        __syncthreads();
        // the offsets of the unit's positions, once for all rows
        if (t < kUnitK) {
            const int k = min(k0 + t, Kn - 1);
            s_off[t] = (uint16_t)(C <= kPrepIdx ? gather_offset(s_idx, C, k) : gather_offset(cherry_indices, C, k));
        }
        __syncthreads();
        int c0 = k0;
        bool staged = near;
        if (!near) {
            c0 = (k0 + s_off[0]) & ~7;
            const int c1 = k1 + s_off[k1 - 1 - k0];
            staged = wide && c1 - c0 <= kPrepCols;
            if (staged) {
#pragma unroll
                for (int p = 0; p < 2; p++)
                    if (sch < ceil_div(c1 - c0, 8) && sr + 8 * p < M)
                        *reinterpret_cast<uint4 *>(&s_x[(t >> 5) + 8 * p][8 * sch]) =
                            *reinterpret_cast<const uint4 *>(x + (size_t)(sr + 8 * p) * K + c0 + 8 * sch);
                __syncthreads();
            }
        }
        const int p0 = 32 * (t >> 6) + 8 * q;  // a lane's 8 positions, in operand order
        if (row < M && k0 + p0 < Kn) {
            if (staged) {
#pragma unroll
                for (int kk = 0; kk < 8; kk++) {
                    const int p = p0 + prompt_ord<BITS>(kk);
                    h[kk] = s_x[i][k0 + p + s_off[p] - c0];
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < 8; kk++) {
                    const int p = p0 + prompt_ord<BITS>(kk);
                    h[kk] = __half_as_ushort(x[(size_t)row * K + k0 + p + s_off[p]]);
                }
            }
        }
    }
    a[((size_t)step * m16 + tile) * 64 + lane] =
        make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
}

// ---- main kernel -----------------------------------------------------------------------------------
template <int BITS>
struct PromptDecode {
    // one literal an instruction at most, and none in the three-operand forms: the constants live in registers, so that
    // mask and OR are one v_and_or_b32
    uint32_t one, m[5];
    __device__ __forceinline__ PromptDecode() {
        asm("v_mov_b32 %0, 0x64006400" : "=v"(one));
        if (BITS == 4) {
            asm("s_mov_b32 %0, 0x001e001e" : "=s"(m[0]));
            asm("s_mov_b32 %0, 0x01e001e0" : "=s"(m[1]));
        } else {
            asm("s_mov_b32 %0, 0x001c000e" : "=s"(m[0]));
            asm("s_mov_b32 %0, 0x00700038" : "=s"(m[1]));
            asm("s_mov_b32 %0, 0x001c0380" : "=s"(m[2]));
            asm("s_mov_b32 %0, 0x000001c0" : "=s"(m[3]));
            asm("s_mov_b32 %0, 0x00e00000" : "=s"(m[4]));
        }
    }
};

// One column's 8 operands on their way from packed codes, as 8 small groups of independent instructions: the caller puts an
// MFMA between any two.
template <int BITS>
struct PromptColumn {
    uint32_t p[2], t[2], s2, f[4], y[4];
    __device__ __forceinline__ void pair(const PromptDecode<BITS> &k, int d) {  // codes of dword d as 1024 + u * 2^p
        if (BITS == 4) f[d] = (t[d >> 1] & k.m[d & 1]) | k.one;
        else if (d == 0) f[d] = (t[0] & k.m[0]) | k.one;
        else if (d == 1) f[d] = (p[0] & k.m[1]) | k.one;
        else if (d == 2) f[d] = (p[1] & k.m[2]) | k.one;
        else f[d] = (p[1] & k.m[4]) | ((p[0] & k.m[3]) | k.one);
    }
    __device__ __forceinline__ void centre(int d) {  // u - c_b
        constexpr float grid = BITS == 4 ? 7.5f : 3.5f;
        const float ma = 1.f / (1 << prompt_pos<BITS>(2 * d)), mb = 1.f / (1 << prompt_pos<BITS>(2 * d + 1));
        y[d] = __builtin_bit_cast(
            uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2_t, f[d]), (half2_t){(_Float16)ma, (_Float16)mb},
                                                (half2_t){(_Float16)(-(1024.f * ma + grid)), (_Float16)(-(1024.f * mb + grid))}));
    }
    __device__ __forceinline__ uint32_t scaled(int d) const {
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, y[d]) * __builtin_bit_cast(half2_t, s2));
    }
    // w: the byte rows' dwords that hold the column in byte c; scale: the dword with its scale in half c & 1
    __device__ __forceinline__ void group(const PromptDecode<BITS> &k, int g, const uint32_t (&w)[BITS], int c, uint32_t scale,
                                          u32x4 &o) {
        switch (g) {
            case 0:
                if (BITS == 4) {
                    const uint32_t sel = 0x0c000c00u | (uint32_t)(c << 16) | (uint32_t)(4 + c);
                    p[0] = __builtin_amdgcn_perm(w[0], w[1], sel);
                    p[1] = __builtin_amdgcn_perm(w[2], w[BITS - 1], sel);
                } else {
                    const uint32_t sel = 0x0c000000u | (uint32_t)(c << 16) | (uint32_t)(c << 8) | (uint32_t)(4 + c);
                    p[0] = __builtin_amdgcn_perm(w[0], w[1], sel);
                    p[1] = __builtin_amdgcn_perm(w[1], w[2], sel);
                }
                break;
            case 1:
                t[0] = p[0] << 1;
                if (BITS == 4) t[1] = p[1] << 1;
                break;
            case 2:
                s2 = __builtin_amdgcn_perm(scale, scale, (c & 1) ? 0x03020302u : 0x01000100u);
                pair(k, 0);
                break;
            case 3: pair(k, 1), centre(0); break;
            case 4: pair(k, 2), centre(1), o[0] = scaled(0); break;
            case 5: pair(k, 3), centre(2), o[1] = scaled(1); break;
            case 6: centre(3), o[2] = scaled(2); break;
            default: o[3] = scaled(3); break;
        }
    }
};

__device__ __forceinline__ void prompt_mfma(float4_t &acc, const u32x4 &a, const u32x4 &b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), acc, 0, 0, 0);
}

// The layers of a launch: their column tiles follow one another.  Layers that read the same rows fill the chip together
// and with larger tiles (128 rows, 4 bits, preparation included: three of 4096 -> 4096 54 -> 33 us, two of 4096 -> 11008
// 58 -> 41, two of 8192 -> 28672 140 -> 121; with 500 rows 99 -> 71, 130 -> 116, 452 -> 447).
struct PromptMembers {
    const uint8_t *qweight[kPromptMaxGroup];
    const __half *cherry_weight[kPromptMaxGroup], *scales[kPromptMaxGroup];
    __half *out[kPromptMaxGroup];
    int N[kPromptMaxGroup], first[kPromptMaxGroup];  // columns, first column tile (past the end: no such layer)
};

// WHOLE: groups are whole units
template <int BITS, int MT, int NC, int NS, bool WHOLE>
__global__ __launch_bounds__(64 * prompt_waves(MT, NC), MT * NC == 64 ? 1 : MT * NC == 8 ? 4 : 2) void prompt_kernel(
    PromptMembers members, const u32x4 *__restrict__ a_all, float *__restrict__ partial, unsigned *__restrict__ tickets, int M, int K,
    int C, int G, int accumulate, PromptPlan plan) {
    constexpr int WAVES = prompt_waves(MT, NC), KW = WAVES / NS, COLS = 16 * NC, ND = NC / 4;  // ND: dwords of a byte row a lane
    typedef uint32_t wd_t __attribute__((ext_vector_type(ND)));
    typedef uint32_t sc_t __attribute__((ext_vector_type(NC / 2)));
    constexpr int ROWS = WAVES * COLS == 1024 ? 16 : 32;  // rows that meet at a time: 64 KB of LDS
    __shared__ __attribute__((aligned(16))) float s_red[WAVES][ROWS][COLS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kq = lane >> 4, nl = lane & 15;
    const int tiles = plan.mtiles * plan.ntiles, per_xcd = ceil_div(tiles, 8);
    const int tile = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3), split = blockIdx.y;
    if (tile >= tiles) return;
    const int mtile = tile % plan.mtiles;
    int ntile = tile / plan.mtiles;
    // selected, not indexed: the arguments arrive with one scalar load
    const int layer = (ntile >= members.first[1] ? 1 : 0) + (ntile >= members.first[2] ? 1 : 0);
    auto of = [&](auto &what) { return layer == 0 ? what[0] : layer == 1 ? what[1] : what[2]; };
    const uint8_t *__restrict__ const qweight = of(members.qweight);
    const __half *__restrict__ const cherry_weight = of(members.cherry_weight);
    const __half *__restrict__ const scales = of(members.scales);
    __half *__restrict__ const out = of(members.out);
    const u32x4 *__restrict__ const a_frag = a_all + layer * (plan.a_bytes / sizeof(u32x4));
    const int N = of(members.N);
    ntile -= of(members.first);
    const int kpart = wave % KW, npart = wave / KW;
    const int n0 = (ntile * NS + npart) * COLS + NC * nl, m16 = plan.mtiles * MT, Kn = K - C;
    const bool col_ok = n0 < N;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)qweight, 0, Kn / 8 * BITS * N, kRsrcFlagsP);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)scales, 0, ceil_div(Kn, G) * N * 2, kRsrcFlagsP);
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void *)cherry_weight, 0, C * N * 2, kRsrcFlagsP);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)a_frag, 0, plan.steps * m16 * 1024, kRsrcFlagsP);

    wd_t w[4][BITS];
    sc_t sc[WHOLE ? 2 : 4];
    u32x4 a[MT], b[2][NC];
    // Units past the wavefront's last one are asked for as unit `plan.units`, which lies past the end of the packed bytes:
    // the bounds of the buffer answer with zeros.
    const uint32_t w_lane = col_ok ? (uint32_t)(kq * BITS * N + n0) : kOobP, sc_lane = col_ok ? (uint32_t)n0 * 2u : kOobP;
    auto load_w = [&](int s, int u) {
        const uint32_t off = w_lane + (uint32_t)((u * 4 + s) * 4 * BITS * N);
#pragma unroll
        for (int r = 0; r < BITS; r++) {
            if constexpr (ND == 1) w[s][r] = __builtin_amdgcn_raw_buffer_load_b32(rw, off + (uint32_t)(r * N), 0, 2);
            else w[s][r] = __builtin_amdgcn_raw_buffer_load_b64(rw, off + (uint32_t)(r * N), 0, 2);
        }
    };
    auto load_sc = [&](int s, int u) -> sc_t {
        const uint32_t off = sc_lane + (uint32_t)((u * kUnitK + 32 * s) / G * N) * 2u;
        if constexpr (NC == 4) return __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
        else return __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
    };
    auto load_a = [&](int m, int step) {
        return __builtin_amdgcn_raw_buffer_load_b128(ra, lane * 16, (step * m16 + mtile * MT + m) * 1024, 0);
    };
    const PromptDecode<BITS> decoder;
    PromptColumn<BITS> column;
    auto decode = [&](int s, const sc_t &scale, int c, int g, u32x4 &o) {
        uint32_t d[BITS];
#pragma unroll
        for (int r = 0; r < BITS; r++) d[r] = w[s][r][c >> 2];
        column.group(decoder, g, d, c & 3, scale[c >> 1], o);
    };

    float4_t acc[MT][NC];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[m][c] = (float4_t){0.f, 0.f, 0.f, 0.f};

    const int u0 = split * plan.units_per_split + kpart, u_end = min((split + 1) * plan.units_per_split, plan.units);
    auto unit_after = [&](int u) { return u + KW < u_end ? u + KW : plan.units; };
    if (u0 < u_end) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            load_w(s, u0);
            if (!WHOLE || s == 0) sc[s] = load_sc(s, u0);
        }
        if (WHOLE) sc[1] = load_sc(0, unit_after(u0));
    }
    // Cherry steps (32 dense fp16 rows, 8 per lane group) while the packed bytes are on their way: behind the loop their own
    // round trip to memory would be one more.
    if (split == plan.splits - 1) {
        for (int cs = KW - 1 - kpart; cs < plan.csteps; cs += KW) {
            sc_t cw[8];
            const uint32_t off = col_ok ? (uint32_t)((32 * cs + 8 * kq) * N + n0) * 2u : kOobP;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                if constexpr (NC == 4) cw[r] = __builtin_amdgcn_raw_buffer_load_b64(rc, off + (uint32_t)(r * N * 2), 0, 0);
                else cw[r] = __builtin_amdgcn_raw_buffer_load_b128(rc, off + (uint32_t)(r * N * 2), 0, 0);
            }
#pragma unroll
            for (int m = 0; m < MT; m++) a[m] = load_a(m, plan.units * 4 + cs);
#pragma unroll
            for (int c = 0; c < NC; c++) {
                u32x4 bc;
#pragma unroll
                for (int d = 0; d < 4; d++)
                    bc[d] = __builtin_amdgcn_perm(cw[2 * d + 1][c >> 1], cw[2 * d][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
                for (int m = 0; m < MT; m++) prompt_mfma(acc[m][c], a[m], bc);
            }
        }
    }
    if (u0 < u_end) {
#pragma unroll
        for (int m = 0; m < MT; m++) a[m] = load_a(m, u0 * 4);
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int g = 0; g < 8; g++) decode(0, sc[0], c, g, b[0][c]);
        load_w(0, unit_after(u0));
        if (!WHOLE) sc[0] = load_sc(0, unit_after(u0));
    }
    // In every step the columns of the next step are decoded between this step's MFMAs, a few instructions behind each: an
    // MFMA occupies the matrix core four times as long as its issue takes, so two vector instructions behind each
    // are free, a block of them behind a block of MFMAs is not (the scheduling barriers keep the order).
    // A step's packed bytes are reloaded for the unit after as soon as they are decoded, the fragments for the next step.
#pragma nounroll
    for (int u = u0; u < u_end;) {
        const int un = unit_after(u), unn = unit_after(un);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int t = (s + 1) & 3;
            const int next = s < 3 ? u * 4 + s + 1 : un < plan.units ? un * 4 : u * 4;  // the last step's own again
#pragma unroll
            for (int m = 0; m < MT; m++) {
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    prompt_mfma(acc[m][c], a[m], b[s & 1][c]);
                    // MT * NC MFMAs take turns with NC columns' 8 groups
                    const int slot = m * NC + c;
#pragma unroll
                    for (int k = slot * 8 / MT; k < (slot + 1) * 8 / MT; k++)
                        decode(t, WHOLE ? sc[s < 3 ? 0 : 1] : sc[t], k / 8, k % 8, b[(s + 1) & 1][k / 8]);
                    if (c == NC - 1) a[m] = load_a(m, next);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            load_w(t, s < 3 ? un : unn);
            if (!WHOLE) sc[t] = load_sc(t, s < 3 ? un : unn);
        }
        if (WHOLE) {
            sc[0] = sc[1];
            sc[1] = load_sc(0, unn);
        }
        u = un < plan.units ? un : u_end;
    }

    // ---- across the wavefronts, ROWS rows at a time; a thread finishes QUADS x 4 columns of each
    constexpr int ROUNDS = MT * 16 / ROWS, THREADS = 64 * WAVES, QUADS = ROWS * COLS * NS / 4 / THREADS;
    float4 sum[ROUNDS][QUADS];
    // 16 lanes that write every second quad of a row would meet in half the banks: the upper half of a row is stored with
    // neighbouring quads exchanged
    auto swizzled = [](int quad) { return ND == 2 ? quad ^ ((quad >> 4) & 1) : quad; };
#pragma unroll
    for (int p = 0; p < ROUNDS; p++) {
        if (p > 0) __syncthreads();
#pragma unroll
        for (int h = 0; h < ROWS / 16; h++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int d = 0; d < ND; d++) {
                    const int m = p * (ROWS / 16) + h;
                    *reinterpret_cast<float4 *>(&s_red[wave][16 * h + 4 * kq + e][4 * swizzled(ND * nl + d)]) =
                        make_float4(acc[m][4 * d][e], acc[m][4 * d + 1][e], acc[m][4 * d + 2][e], acc[m][4 * d + 3][e]);
                }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < QUADS; q++) {
            const int e = tid + q * THREADS, row = e / (NS * COLS / 4), quad = e % (COLS / 4), part = e / (COLS / 4) % NS;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int k = 0; k < KW; k++) {
                const float4 o = *reinterpret_cast<const float4 *>(&s_red[part * KW + k][row][4 * swizzled(quad)]);
                v.x += o.x, v.y += o.y, v.z += o.z, v.w += o.w;
            }
            sum[p][q] = v;
        }
    }
    // ---- across workgroups: tiles in scratch in the order [round][quad][thread]
    if (plan.splits > 1) {
        constexpr size_t TILE = (size_t)MT * 16 * COLS * NS;
        float *base = partial + (size_t)tile * TILE + tid * 4;
        const size_t per_split = (size_t)tiles * TILE;
        auto word = [&](int s, int p, int q, int h) {
            return reinterpret_cast<unsigned long long *>(base + s * per_split + (size_t)(p * QUADS + q) * THREADS * 4) + h;
        };
#pragma unroll
        for (int p = 0; p < ROUNDS; p++)
#pragma unroll
            for (int q = 0; q < QUADS; q++) {
                const float2 lo = make_float2(sum[p][q].x, sum[p][q].y), hi = make_float2(sum[p][q].z, sum[p][q].w);
                __hip_atomic_store(word(split, p, q, 0), __builtin_bit_cast(unsigned long long, lo), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(word(split, p, q, 1), __builtin_bit_cast(unsigned long long, hi), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        int *s_last = reinterpret_cast<int *>(&s_red[0][0][0]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0) {
            const unsigned old = __hip_atomic_fetch_add(&tickets[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *s_last = old == (unsigned)(plan.splits - 1);
        }
        __syncthreads();
        if (!*s_last) return;
        if (tid == 0) __hip_atomic_store(&tickets[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int p = 0; p < ROUNDS; p++)
#pragma unroll
            for (int q = 0; q < QUADS; q++) sum[p][q] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 2
        for (int s = 0; s < plan.splits; s++) {
            float2 v[ROUNDS][QUADS][2];
#pragma unroll
            for (int p = 0; p < ROUNDS; p++)
#pragma unroll
                for (int q = 0; q < QUADS; q++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        v[p][q][h] = __builtin_bit_cast(
                            float2, __hip_atomic_load(word(s, p, q, h), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
            for (int p = 0; p < ROUNDS; p++)
#pragma unroll
                for (int q = 0; q < QUADS; q++) {
                    sum[p][q].x += v[p][q][0].x, sum[p][q].y += v[p][q][0].y;
                    sum[p][q].z += v[p][q][1].x, sum[p][q].w += v[p][q][1].y;
                }
        }
    }
#pragma unroll
    for (int p = 0; p < ROUNDS; p++)
#pragma unroll
        for (int q = 0; q < QUADS; q++) {
            const int e = (tid + q * THREADS) * 4, m = mtile * MT * 16 + p * ROWS + e / (COLS * NS),
                      n = ntile * COLS * NS + e % (COLS * NS);
            if (m < M && n < N) {
                uint2 *o = reinterpret_cast<uint2 *>(out + (size_t)m * N + n);
                float v[4] = {sum[p][q].x, sum[p][q].y, sum[p][q].z, sum[p][q].w};
                if (accumulate) {
                    const uint2 was = *o;
                    v[0] += __half2float(__ushort_as_half((unsigned short)was.x));
                    v[1] += __half2float(__ushort_as_half((unsigned short)(was.x >> 16)));
                    v[2] += __half2float(__ushort_as_half((unsigned short)was.y));
                    v[3] += __half2float(__ushort_as_half((unsigned short)(was.y >> 16)));
                }
                uint32_t h[4];
#pragma unroll
                for (int c = 0; c < 4; c++) h[c] = __half_as_ushort(__float2half_rn(v[c]));
                *o = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            }
        }
}

bool prompt_supported(int bits, int M, int K, int N, int C, int G) {
    if (M < 2 || G % 32 || K - C <= 0) return false;  // an MFMA's 32 positions must not straddle a group
    const long long wbytes = (long long)(K - C) / 8 * 4 * N;
    const long long cbytes = (long long)C * N * 2;
    const long long sbytes = (long long)ceil_div(K - C, G) * N * 2;
    const long long abytes = (long long)prompt_plan(M, K, N, C).a_bytes;
    return wbytes < 0x7fff0000ll && cbytes < 0x7fff0000ll && sbytes < 0x7fff0000ll && abytes < 0x7fff0000ll;
}

template <int BITS, int MT, int NC, int NS>
static hipError_t launch_prompt_mt(const __half *vec, const PromptMember *layers, int count, int M, int K, int C, int G, int accumulate,
                                   const PromptPlan &plan, void *workspace, void *scratch, hipStream_t stream) {
    u32x4 *a = reinterpret_cast<u32x4 *>(scratch);
    float *partial = reinterpret_cast<float *>(reinterpret_cast<char *>(scratch) + count * plan.a_bytes);
    unsigned *tickets = reinterpret_cast<unsigned *>(workspace);
    PromptIndices indices;
    PromptMembers members;
    int first = 0;
    for (int i = 0; i < kPromptMaxGroup; i++) {
        const PromptMember &l = layers[i < count ? i : 0];
        indices.of[i] = l.cherry_indices;
        members.qweight[i] = l.qweight, members.cherry_weight[i] = l.cherry_weight, members.scales[i] = l.scales, members.out[i] = l.out;
        members.N[i] = l.N, members.first[i] = first;
        if (i < count) first += ceil_div(l.N, 16 * NC * NS);
    }
    hipLaunchKernelGGL(prompt_prep_kernel<BITS>, dim3(plan.units + ceil_div(plan.csteps, 4), plan.mtiles * MT, count), dim3(256), 0, stream,
                       vec, indices, reinterpret_cast<uint4 *>(a), plan.a_bytes, M, K, C, plan.units, plan.mtiles * MT,
                       aligned(vec, 16) ? 1 : 0);
    const dim3 grid(8 * ceil_div(plan.mtiles * plan.ntiles, 8), plan.splits);
    auto *const kernel = G % kUnitK == 0 ? prompt_kernel<BITS, MT, NC, NS, true> : prompt_kernel<BITS, MT, NC, NS, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(64 * prompt_waves(MT, NC)), 0, stream, members, a, partial, tickets, M, K, C, G, accumulate, plan);
    return hipGetLastError();
}

template <int BITS>
static hipError_t launch_prompt_bits(const __half *vec, const PromptMember *layers, int count, int M, int K, int C, int G, int accumulate,
                                     void *workspace, void *scratch, hipStream_t stream) {
    int N[kPromptMaxGroup];
    for (int i = 0; i < count; i++) N[i] = layers[i].N;
    const PromptPlan plan = prompt_plan(M, K, N, count, C);
#define CQ_PROMPT(MT_, NC_, NS_)                            \
    if (plan.mt == MT_ && plan.nc == NC_ && plan.ns == NS_) \
    return launch_prompt_mt<BITS, MT_, NC_, NS_>(vec, layers, count, M, K, C, G, accumulate, plan, workspace, scratch, stream)
    CQ_PROMPT(2, 4, 1);
    CQ_PROMPT(4, 4, 1);
    CQ_PROMPT(8, 4, 1);
    CQ_PROMPT(8, 8, 1);
    CQ_PROMPT(8, 8, 2);
#undef CQ_PROMPT
    return hipErrorInvalidConfiguration;
}

hipError_t launch_prompt(int bits, const __half *vec, const PromptMember *layers, int count, int M, int K, int C, int G, int accumulate,
                         void *workspace, void *scratch, hipStream_t stream) {
    if (count < 1 || count > kPromptMaxGroup) return hipErrorInvalidValue;
    return bits == 4 ? launch_prompt_bits<4>(vec, layers, count, M, K, C, G, accumulate, workspace, scratch, stream)
                     : launch_prompt_bits<3>(vec, layers, count, M, K, C, G, accumulate, workspace, scratch, stream);
}

}  // namespace cq
