// Dense 16-bit matrix products of quantisation-aware training,  D[M, N] = sum_k A(m, k) B(n, k)  with fp32 sums and one rounding:
// the training layer's output  x W'^T  and its gradients  g W'  and  g^T x  (llama/cherry_linear.py:101-126 and autograd).
//
// Either operand may lie as [free][K] or as [K][free], so no transposed copy is made.  One whole round of tiles is bound by the power
// that the matrix cores draw: 4096 x 4096 x 8192 runs at 1.35 PFLOP/s with the clock at 1.91 GHz (of 2.4) and the matrix cores busy
// 68 % of the time.  2048 rows of 4096 -> 11008 are not: 53 to 59 % at 2.05 to 2.14 GHz.  Their tiles leave an uneven last round (96, 86
// and 96 steps where a compute unit's share is 86); the rest are a tile's two ends (7 us), sums through scratch (8 us) and the barrier a step.
//   * A workgroup of eight wavefronts owns a tile of 256 x 256, a wavefront 128 x 64 of it: 128 accumulators, two wavefronts a
//     SIMD, so that one's waits lie behind the other's products (four wavefronts of 128 x 128: 5 to 10 % slower at every size).
//   * K in steps of 64 through two LDS buffers of 64 KB, filled by loads that go straight to LDS (through registers: 3 us a tile
//     more at its ends).  A buffer is asked for again while its other half of products is still running, a load every three
//     products (all at once, in front or behind: 3 to 5 % slower).
//   * LDS holds the operands as they come, 128 bytes of a row of [free][K], 512 of a row of [K][free], in 16- or 32-byte pieces
//     exchanged by row so that neither the loads' writes nor the fragments' reads meet in a bank; [K][free] fragments are
//     transposed by the read (ds_read_b64_tr_b16).
//   * A tile's first step is (row tile + column tile) steps into K: rows of [free][K] a power of two apart lie on the same few
//     channels of the L2 (2048 rows of 4096 -> 11008: 167 -> 157 us; two steps a tile: the L2 no longer holds what tiles share).
// Tiles that are left behind the last whole round of 256 are split along K where that ends earlier: all but the last workgroup
// to arrive leave fp32 sums in scratch (the two gradients and the output of 2048 rows of 4096 -> 11008: 513 -> 455 us against
// every workgroup writing its sums with 8-byte atomic stores).  Two parts are added as they are, more in split order: the
// result does not depend on who is last.
//
// us, the library's product / this, bf16:                          x W'^T        g W'        g^T x
//     2048 rows, 4096 -> 11008                                    159 / 155   172 / 148    208 / 153
//     728 rows, 10712 -> 9728                                     229 / 195   175 / 150    250 / 191
//     135 rows, 6080 -> 6840                                       40 / 52     48 / 53      70 / 32
// (few tiles: the library, gemm_preferred)
#include <algorithm>
#include <type_traits>

#include "cq_device.h"
#include "cq_kernels.h"

namespace cq {

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bhalf4_t __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 256, kStep = 64;          // rows and columns of a tile, positions of K a step
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kRowFrags = 8, kColFrags = 4;     // fragments of 16 of a wavefront's 128 x 64
constexpr int kOperand = kTile * kStep * 2;     // bytes of an operand's tile
constexpr int kBuffer = 2 * kOperand;
constexpr int kChunks = kOperand / 16 / kThreads;  // 16-byte pieces of it that a thread asks for
constexpr int kLoads = 2 * kChunks;
constexpr uint32_t kTileSums = kTile * kTile * sizeof(float);
constexpr uint32_t kRsrcFlagsG = 0x00020000u, kOobG = 0x80000000u;
constexpr int kDeviceScope = 16;  // of a buffer access: past the die's L2
constexpr int kPolls = 1 << 18;   // a microsecond or so each

// (The compiler's own form may name another destination and then copies accumulators.  Distances: products into the same accumulator
// need none, fragments come from LDS behind a wait, and the results are read behind the s_nop at the loop's end, which names the last
// ones, so that they cannot be read in front of it.  tests/test_mfma_distances.py reads the built code.)
template <bool BF16>
__device__ __forceinline__ void gemm_mma(float4_t &acc, const u32x4 &a, const u32x4 &b) {
    if constexpr (BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}

// This wavefront's LDS reads are done and what it asked for is in LDS; then everybody's.
__device__ __forceinline__ void step_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// One operand of a tile, [free][K] or (BY_K) [K][free], and this thread's part in moving it.
template <bool BY_K, int FRAGS>
struct GemmOperand {
    const char *base;  // the tile, at the step that is asked for next
    int left;          // bytes from there to the array's end: past it loads give zeros
    uint32_t voff, jump, advance;
    int first;         // [free][K]: this thread's first position of a step
    uint32_t place;    // LDS address of this wavefront's first 1 KB
    uint32_t read[BY_K ? FRAGS : 2];
    static constexpr int kReads = BY_K ? 2 * FRAGS : FRAGS;  // LDS reads of the fragments of half a step

    // A row's pieces are exchanged by the row's number: 16-byte pieces of the 128 bytes of a row of [free][K], 32-byte pieces of [K][free]
    static __device__ __forceinline__ int exchange(int row) { return BY_K ? (row & 3) | ((row >> 3) & 1) << 2 : (row >> 1) & 7; }

    __device__ __forceinline__ void init(const void *array, int rows, int cols, int free0, int k0, int tid, int wave, int wave_free, uint32_t lds) {
        const uint32_t pitch = (uint32_t)cols * 2u, total = (uint32_t)rows * pitch;
        const uint32_t at = BY_K ? (uint32_t)k0 * pitch + (uint32_t)free0 * 2u : (uint32_t)free0 * pitch + (uint32_t)k0 * 2u;
        base = reinterpret_cast<const char *>(array) + at;
        left = (int)(total - min(at, total));
        place = lds + wave * 1024;
        const int lane = tid & 63, q = lane >> 4, i = lane & 15;
        if constexpr (BY_K) {
            const int r = tid >> 5, c = (tid & 31) ^ (2 * exchange(r));
            voff = (uint32_t)r * pitch + c * 16, jump = kThreads / 32 * pitch, advance = kStep * pitch;
            first = 0;
            // lanes 4 e .. 4 e + 3 of 16 name the 16 values of position e; the read gives lane i the four positions of value i
            const int row = 8 * q + (i >> 2);
#pragma unroll
            for (int m = 0; m < FRAGS; m++) read[m] = lds + row * 512 + ((wave_free / 16 + m) ^ exchange(row)) * 32 + (i & 3) * 8;
        } else {
            const int r = tid >> 3, c = (tid & 7) ^ exchange(r);
            voff = (uint32_t)r * pitch + c * 16, jump = kThreads / 8 * pitch, advance = kStep * 2;
            first = 8 * c;
#pragma unroll
            for (int p = 0; p < 2; p++) read[p] = lds + (wave_free + i) * 128 + ((4 * p + q) ^ exchange(i)) * 16;
        }
    }
    // 1 KB a wavefront straight into LDS; k_left: positions of K from the step's first one on
    __device__ __forceinline__ void load(uint32_t buffer, int j, int k_left) const {
        const uint64_t b = reinterpret_cast<uint64_t>(base);
        const u32x4 r = {(uint32_t)__builtin_amdgcn_readfirstlane((int)b), (uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32) & 0xffff),
                         (uint32_t)__builtin_amdgcn_readfirstlane(max(left, 0)), kRsrcFlagsG};
        const uint32_t off = BY_K || first < k_left ? voff + j * jump : kOobG;
        const uint32_t to = (uint32_t)__builtin_amdgcn_readfirstlane(buffer + place + j * (kThreads * 16));
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(r), "s"(to) : "memory");
    }
    __device__ __forceinline__ void next(int steps) {  // backwards where K starts again
        base += (long long)steps * (int)advance;
        left = __builtin_amdgcn_readfirstlane(left - steps * (int)advance);
    }
    __device__ __forceinline__ void fragment(char *lds, uint32_t buffer, int half, int n, u32x4 (&f)[FRAGS]) const {
        if constexpr (BY_K) {
            const int m = n >> 1, h = n & 1;
            typedef __attribute__((address_space(3))) s16x4 lds4;
            const u32x2 u = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(lds + buffer + read[m] + (32 * half + 4 * h) * 512)));
            f[m][2 * h] = u[0], f[m][2 * h + 1] = u[1];
        } else {
            f[n] = *reinterpret_cast<const u32x4 *>(lds + buffer + read[half] + n * 16 * 128);
        }
    }
};

template <bool BF16, bool A_BY_K, bool B_BY_K>
__global__ __launch_bounds__(kThreads, 2) void gemm_kernel(const void *__restrict__ a_all, const void *__restrict__ b_all, uint16_t *__restrict__ out,
                                                           char *__restrict__ scratch, unsigned *__restrict__ tickets, int M, int N, int K,
                                                           GemmPlan plan) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kBuffer];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    // ---- which tile, and which steps of K.  A die (every eighth workgroup) takes neighbouring tiles, 8 rows of tiles at a time: its 32
    // workgroups read 4 + 8 operands' tiles a step, not 64
    int tile, split = 0, rest = -1;
    if ((int)blockIdx.x < plan.full) {
        tile = (blockIdx.x & 7) * (plan.full >> 3) + (blockIdx.x >> 3);
    } else {
        const int pieces = plan.rest * plan.splits, at = blockIdx.x - plan.full, piece = (at & 7) * ((pieces + 7) >> 3) + (at >> 3);
        if (piece >= pieces) return;
        split = (unsigned)piece / (unsigned)plan.rest, rest = piece - split * plan.rest;
        tile = plan.full + rest;
    }
    int mt = 0, nt = tile, mrows = plan.mtiles;
    if (mrows > 8) {
        mt = (unsigned)tile / (unsigned)(8 * plan.ntiles) * 8;
        nt -= mt * plan.ntiles, mrows = min(8, mrows - mt);
    }
    const int in_block = nt;
    nt = (unsigned)in_block / (unsigned)mrows, mt += in_block - nt * mrows;
    const int s0 = rest < 0 ? 0 : split * plan.per_split, steps = rest < 0 ? plan.steps : min(plan.per_split, plan.steps - s0);
    const int turn = (unsigned)(mt + nt) % (unsigned)steps;

    GemmOperand<A_BY_K, kRowFrags> A;
    GemmOperand<B_BY_K, kColFrags> B;
    A.init(a_all, A_BY_K ? K : M, A_BY_K ? M : K, mt * kTile, (s0 + turn) * kStep, tid, wave, wm * 128, 0);
    B.init(b_all, B_BY_K ? K : N, B_BY_K ? N : K, nt * kTile, (s0 + turn) * kStep, tid, wave, wn * 64, kOperand);
    int k_left = K - (s0 + turn) * kStep, to_end = steps - turn, ahead = steps;
    auto load = [&](uint32_t buffer, int j) {
        if (j < kChunks) A.load(buffer, j, k_left);
        else B.load(buffer, j - kChunks, k_left);
    };
    auto advance = [&]() {
        const int by = --to_end == 0 ? 1 - steps : 1;
        k_left -= by * kStep;
        A.next(by), B.next(by);
        if (--ahead <= 0) A.left = B.left = -0x40000000;  // nothing left to ask for
    };
#pragma unroll
    for (int p = 0; p < 2; p++) {
#pragma unroll
        for (int j = 0; j < kLoads; j++) load(p * kBuffer, j);
        advance();
    }
    float4_t acc[kRowFrags][kColFrags];
#pragma unroll
    for (int m = 0; m < kRowFrags; m++)
#pragma unroll
        for (int n = 0; n < kColFrags; n++) {
            acc[m][n] = (float4_t){0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+v"(acc[m][n]));  // written here, not right in front of the first product
        }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kLoads) : "memory");
    __builtin_amdgcn_sched_barrier(0);

    // Half a step: 32 products a wavefront, and behind them the next half's fragments, A's in place as soon as their last product is
    // issued, B's into the other set.  Half a step's products in front of a buffer change its last fragments have been read, so everybody
    // meets eight products on, and the buffer is asked for again.
    u32x4 fa[kRowFrags], fb[2][kColFrags];
    constexpr int A_READS = A.kReads / kRowFrags, B_READS = B.kReads, SLOTS = kRowFrags * kColFrags, MEET = 8;
    auto read_a = [&](uint32_t buffer, int half, int m) {
#pragma unroll
        for (int r = 0; r < A_READS; r++) A.fragment(lds, buffer, half, m * A_READS + r, fa);
    };
#pragma unroll
    for (int n = 0; n < B_READS; n++) {
        B.fragment(lds, 0, 0, n, fb[0]);
        __builtin_amdgcn_sched_barrier(0);  // in this order: the compiler's waits in the loop count on it, too
    }
#pragma unroll
    for (int m = 0; m < kRowFrags; m++) {
        read_a(0, 0, m);
        __builtin_amdgcn_sched_barrier(0);
    }
    uint32_t here = 0;
    auto phase = [&](auto which) {
        constexpr int half = which, next = half ^ 1;
        const uint32_t there = half ? here ^ kBuffer : here;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < SLOTS; i++) {
            if (half && i == MEET) step_barrier();
            gemm_mma<BF16>(acc[i / kColFrags][i % kColFrags], fb[half][i % kColFrags], fa[i / kColFrags]);
            // (the two of A that are free before everybody has met follow right behind)
#pragma unroll
            for (int m = 0; m < kRowFrags; m++)
                if (i == (half ? m == 0 ? MEET + 2 : m == kRowFrags - 1 ? SLOTS - 1 : (m + 1) * kColFrags : (m + 1) * kColFrags - 1)) read_a(there, next, m);
            constexpr int from = half ? MEET + 1 : 0, span = SLOTS - (half ? 16 : 4);
#pragma unroll
            for (int r = 0; r < B_READS; r++)
                if (i >= from && r >= (i - from) * B_READS / span && r < (i + 1 - from) * B_READS / span) B.fragment(lds, there, next, r, fb[next]);
            if constexpr (half) {
#pragma unroll
                for (int l = 0; l < kLoads; l++)
                    if (i >= MEET && l >= (i - MEET) * kLoads / 22 && l < (i + 1 - MEET) * kLoads / 22) load(here, l);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (half) advance();
        here = there;
    };
#pragma nounroll
    for (int t = 0; t < steps; t++) {
        phase(std::integral_constant<int, 0>{});
        phase(std::integral_constant<int, 1>{});
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15" : "+v"(acc[7][0]), "+v"(acc[7][1]), "+v"(acc[7][2]), "+v"(acc[7][3]) : : "memory");
    __builtin_amdgcn_sched_barrier(0);

    // ---- results, through LDS, so that the 128 bytes of a row are stored together
    auto finish = [&](auto sums_of) {
        __syncthreads();
        char *const mine = lds + wave * (128 * 128);
#pragma unroll
        for (int m0 = 0; m0 < kRowFrags; m0 += 4) {  // two round trips to scratch, and registers enough for them
            float4_t sums[4][kColFrags];
#pragma unroll
            for (int m = 0; m < 4; m++) sums_of(m0 + m, sums[m]);
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int n = 0; n < kColFrags; n++) {
                    u32x2 v;
                    if constexpr (BF16) v = __builtin_bit_cast(u32x2, __builtin_convertvector(sums[m][n], bhalf4_t));
                    else v = __builtin_bit_cast(u32x2, __builtin_convertvector(sums[m][n], half4_t));
                    const int row = 16 * (m0 + m) + (lane & 15), piece = 2 * n + (lane >> 5);
                    *reinterpret_cast<u32x2 *>(mine + row * 128 + (piece ^ (row & 7)) * 16 + ((lane >> 4) & 1) * 8) = v;
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read with another type, by other lanes of the wavefront
        const int col = nt * kTile + wn * 64 + 8 * (lane & 7);
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int r = 8 * j + (lane >> 3), row = mt * kTile + wm * 128 + r;
            const u32x4 v = *reinterpret_cast<const u32x4 *>(mine + r * 128 + ((lane & 7) ^ (r & 7)) * 16);
            if (row < M && col < N) *reinterpret_cast<u32x4 *>(out + (size_t)row * N + col) = v;
        }
    };
    // ---- across workgroups where K is split.  All but the last to arrive leave their sums and end (more than two: the last one too); the
    // last one waits only for workgroups that have arrived, which wait for nobody.  It waits for some 10 us at most; counts that another
    // call has changed (a workspace that is shared against the rule) end the wait all the same, and the tile is NaN
    if (rest >= 0 && plan.splits > 1) {
        unsigned *const arrived = tickets + 2 * rest, *const written = arrived + 1;
        char *const all = scratch + (size_t)rest * plan.splits * kTileSums;
        const uint32_t at = wave * (kRowFrags * kColFrags * 1024) + lane * 16;
        int *const s_order = reinterpret_cast<int *>(lds);
        __syncthreads();
        if (tid == 0) *s_order = (int)__hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const bool last = *s_order == plan.splits - 1;
        if (!last || plan.splits > 2) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(all + (size_t)split * kTileSums, 0, kTileSums, kRsrcFlagsG);
#pragma unroll
            for (int e = 0; e < kRowFrags * kColFrags; e++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[e / kColFrags][e % kColFrags]), r, at + e * 1024, 0, kDeviceScope);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (!last) {
                if (tid == 0) __hip_atomic_fetch_add(written, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return;
            }
        }
        if (tid == 0) {
            int polls = kPolls;
            while (__hip_atomic_load(written, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (unsigned)(plan.splits - 1) && --polls) __builtin_amdgcn_s_sleep(2);
            s_order[1] = polls;
            __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(written, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(s_order[1]) == 0) {  // counts that are not this call's: say so, and end
            const u32x4 nan = {0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu};  // in fp16 and in bfloat16
            const int col = nt * kTile + 8 * (tid & 31);
            for (int row = mt * kTile + (tid >> 5); row < min(M, (mt + 1) * kTile) && col < N; row += kThreads / 32)
                *reinterpret_cast<u32x4 *>(out + (size_t)row * N + col) = nan;
            return;
        }
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(all, 0, plan.splits * kTileSums, kRsrcFlagsG);
        auto part = [&](int s, int m, int n) {
            return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, at + (m * kColFrags + n) * 1024, s * kTileSums, kDeviceScope));
        };
        if (plan.splits == 2)
            return finish([&](int m, float4_t (&v)[kColFrags]) {
#pragma unroll
                for (int n = 0; n < kColFrags; n++) v[n] = part(1 - split, m, n);
#pragma unroll
                for (int n = 0; n < kColFrags; n++) v[n] += acc[m][n];
            });
        return finish([&](int m, float4_t (&v)[kColFrags]) {
#pragma unroll
            for (int n = 0; n < kColFrags; n++) v[n] = part(0, m, n);
#pragma nounroll
            for (int s = 1; s < plan.splits; s++) {
                float4_t o[kColFrags];
#pragma unroll
                for (int n = 0; n < kColFrags; n++) o[n] = part(s, m, n);
#pragma unroll
                for (int n = 0; n < kColFrags; n++) v[n] += o[n];
            }
        });
    }
    finish([&](int m, float4_t (&v)[kColFrags]) {
#pragma unroll
        for (int n = 0; n < kColFrags; n++) v[n] = acc[m][n];
    });
}

// Microseconds, fitted to 180 products of the training layer's range (rows 128 to 2048, 1024 to 11008 channels, 512 to 11008 columns,
// each of the three forms; 5.5 % off on average): a step of a whole round and of the one behind it, alone and when all compute units are
// at it, a round's ends, and sums that go through scratch.
GemmPlan gemm_plan(int M, int N, int K) {
    GemmPlan p = {};
    p.mtiles = ceil_div(M, kTile), p.ntiles = ceil_div(N, kTile), p.steps = ceil_div(K, kStep);
    const int tiles = p.mtiles * p.ntiles;
    p.full = tiles / 256 * 256, p.rest = tiles - p.full, p.splits = 1, p.per_split = p.steps;
    p.cost = 0.8f + (float)(tiles / 256) * (7.f + 1.55f * (float)p.steps);
    float best = 3.4e38f;
    for (int s = 1; s <= 8 && p.rest && (s == 1 || s * p.rest <= 256); s++) {
        const int per = ceil_div(p.steps, s), splits = ceil_div(p.steps, per);
        const float share = (float)(splits * p.rest) / 256.f;
        const float cost = 7.f + (float)per * (0.92f + 0.67f * share) + (splits > 1 ? 2.2f + 2.3f * (float)splits + 8.8f * share : 0.f);
        if (cost < best) best = cost, p.per_split = per, p.splits = splits;
    }
    if (p.rest) p.cost += best;
    p.scratch_bytes = p.splits > 1 ? (size_t)p.splits * p.rest * kTileSums : 0;
    p.workspace_bytes = p.splits > 1 ? (size_t)p.rest * 2 * sizeof(unsigned) : 0;
    return p;
}

// Where the library's product takes longer: its time on the same 180 products (11 % off on average), by operations, bytes, depth, and for
// two [K][free] operands the results' size, where it is slowest.  Chosen so, all of them take 8.1 ms, the library alone 9.8, the faster of
// both each time 7.9; none is more than 6 % slower than the library.  The fourth form, `a` as [K][M] and `b` as [N][K], is no product of the
// layer and none of these: nothing is said of it.
bool gemm_preferred(bool a_by_k, bool b_by_k, int M, int N, int K) {
    if ((a_by_k && !b_by_k) || !gemm_supported(a_by_k, b_by_k, M, N, K)) return false;
    const float m = (float)M, n = (float)N, k = (float)K, mbytes = 2e-6f * (m * k + n * k + m * n);
    float library = 7.1f + 1.69e-9f * m * n * k + 0.23f * mbytes + 1.9e-3f * k;
    if (a_by_k && b_by_k) library += 0.16f * mbytes + 0.55e-6f * m * n;
    return gemm_plan(M, N, K).cost < 0.95f * library;
}

// One buffer descriptor an operand, and numbers of tiles that fit the plan's
bool gemm_sizes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return false;
    const long long most = 0x7fff0000ll, mtiles = (M - 1ll) / kTile + 1, ntiles = (N - 1ll) / kTile + 1;
    return 2ll * M * K < most && 2ll * N * K < most && 2ll * M * N < (1ll << 40) && mtiles * ntiles < (1 << 24);
}

// Besides, whole 16-byte pieces along every row.  A step's last row of [K][free] starts 63 rows on: that has to fit 32 bits, or rows past K come
// round to the array's start instead of reading zeros (only rows of 64 MB and more, of which there are few).
bool gemm_supported(bool a_by_k, bool b_by_k, int M, int N, int K) {
    constexpr int longest = ((1ll << 32) - 512) / (2 * 63);
    return gemm_sizes(M, N, K) && N % 8 == 0 && (!a_by_k || (M % 8 == 0 && M <= longest)) && (!b_by_k || N <= longest) &&
           ((a_by_k && b_by_k) || K % 8 == 0);
}

template <bool BF16>
static hipError_t launch_gemm_type(bool a_by_k, bool b_by_k, const void *a, const void *b, void *out, int M, int N, int K, const GemmPlan &p,
                                   void *workspace, void *scratch, hipStream_t stream) {
    auto *const kernel = a_by_k ? (b_by_k ? gemm_kernel<BF16, true, true> : gemm_kernel<BF16, true, false>)
                                : (b_by_k ? gemm_kernel<BF16, false, true> : gemm_kernel<BF16, false, false>);
    const dim3 grid(p.full + 8 * ceil_div(p.rest * p.splits, 8));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, a, b, reinterpret_cast<uint16_t *>(out), reinterpret_cast<char *>(scratch),
                       reinterpret_cast<unsigned *>(workspace), M, N, K, p);
    return hipGetLastError();
}

hipError_t launch_gemm(bool bf16, bool a_by_k, bool b_by_k, const void *a, const void *b, void *out, int M, int N, int K, const GemmPlan &plan,
                       void *workspace, void *scratch, hipStream_t stream) {
    return bf16 ? launch_gemm_type<true>(a_by_k, b_by_k, a, b, out, M, N, K, plan, workspace, scratch, stream)
                : launch_gemm_type<false>(a_by_k, b_by_k, a, b, out, M, N, K, plan, workspace, scratch, stream);
}

}  // namespace cq
