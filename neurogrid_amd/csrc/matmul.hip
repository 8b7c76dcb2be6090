// matmul.hip - cuda_gemm_int8 and cuda_gemm_fp16 for gfx950.
//
// Reference: gpu/cuda/matmul.cu:75-156 (cuda_gemm_fp16: cublasHgemm with the
// row-major -> column-major operand swap) and :169-244 (cuda_gemm_int8:
// cudaMalloc a K*N fp16 copy, dequantize_and_copy, cuda_gemm_fp16, cudaFree).
//
// Weight-streaming path (transpose_b, M <= 128). The engine's INT8 layers call
// cuda_gemm_int8 with B stored [N, K] and one scale per row of B
// (layer.cu:487-501,551,575). For up to a few hundred tokens the product is
// bound by reading B once, 1 byte per weight; the reference moves 5 (read
// int8, write fp16, read fp16). Here the kernel reads the codes, turns them
// into exact fp16 integers in registers and feeds the matrix cores:
//   C[m, n] = fp16( scale[n] * sum_k A[m, k] * q[n, k] )
// with the sum in fp32 (every product of an fp16 activation and an integer
// code in [-128, 127] is exact in fp32). The reference rounds q * scale to
// fp16 first and sums those; the two differ by at most 2^-11 of
// sum_k |A[m, k] * q[n, k] * scale[n]| plus the accumulation error.
//
// Four kernels, by M, K and N (see gemm_i8w):
//   M <= 2, and M <= 4 with K, N < 8192: gemv_i8w_kernel, dot-product
//       instructions, each load reads 1 KiB contiguous of one row of B;
//   4 < M <= 16 with K, N < 8192: gemm_i8w_kernel, matrix cores, A read from
//       L2, waves split K within the block;
//   otherwise, up to M = 32: gemm_i8w_split_kernel, matrix cores, A staged
//       in LDS, K split between wave groups of a block and between blocks
//       (slices whose sums a second kernel adds);
//   32 < M <= 128: gemm_i8w_ring_kernel, A and B straight into LDS several
//       steps ahead, K split likewise.
// Above 128 rows of A (prefill) the product is bound by the matrix cores:
// gemm_i8w_tile_kernel, a tiled GEMM that loads A and the codes of B straight
// into LDS and converts the codes on their way to the matrix cores (see the
// prefill section), with the residual add or SwiGLU in its epilogue; from 4096
// rows on (kLtMinM) the reference's composition through hipBLASLt, which is
// faster there. B stored [K, N] always goes through the composition (dequantize,
// then hipBLASLt).
// Each fused kernel also has a shared form (ng_gemm_int8_shared_a) that runs
// several products with the same A and the same launch shape in one launch,
// each product's blocks as in its own launch; the GEMV kernel's shared form
// can also normalise A itself (ng_rmsnorm_gemm_int8_shared_a and the add +
// RMSNorm form), each block in registers, for the decode steps norm -> q/k/v.
// MFMA layout: v_mfma_f32_16x16x32_f16 multiplies a 16 x 32 tile of A (rows
// m) by a 32 x 16 tile of B^T (columns n). Lane l supplies row (l % 16) of
// each operand and 8 values of k; the accumulator lane l holds rows
// 4 * (l / 16) + i, column l % 16. In a chunk of 64 k, lane group g = l / 16
// holds k = 16g .. 16g + 15 of its row of B (16 codes); the first 8 feed one
// MFMA and the last 8 another, and A's lanes take the same k, so each MFMA
// sums matching k. The two MFMA kernels read B in whole 128-byte lines (8 rows
// x 128 codes per load instruction) and reorder the codes into that layout
// through LDS: loading straight into it reads 64 bytes per row per
// instruction, which streams about 25% slower on MI355X.
// Every sum is taken in a fixed order (partial sums meet in LDS or in the
// slice buffer, never through atomics), so results do not depend on timing.
#include "ng_common.hpp"
#include "ng_exact.hpp"
#include "../../include/kernels.h"
#include "../../include/matmul.h"
#include "../../include/neurogrid_ext.h"

#include <hipblaslt/hipblaslt.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <map>
#include <mutex>
#include <set>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

// Partial sums of the allocation-free entry point (ng_gemm_int8_noalloc): a
// device array of fixed size that every GPU the library runs on holds until
// the process ends. In host code `scratch` names a host-side stand-in, not
// device memory: its device address is looked up once per device
// (hipGetSymbolAddress, see scratch_ptr) and only that address is used.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

namespace ng {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kChunk = 64;          // K granularity of the MFMA kernels (one 16x16x32 MFMA pair per lane group)
constexpr int kMaxFusedM = 128;     // rows of A the weight-streaming path takes

// Two int8 codes (bytes SEL0 and SEL1 of one dword) -> two exact fp16 values.
// The bytes are biased to u = q + 128, placed under an fp16 exponent of 2^10
// with v_perm (fp16 bits 0x6400 | u = 1024 + u), and 1152 is subtracted in
// fp16: every step is exact.
template <uint32_t SEL>
__device__ __forceinline__ uint32_t codes_to_f16x2(uint32_t w) {
    const f16x2 bias = {static_cast<f16>(-1152.0f), static_cast<f16>(-1152.0f)};
    const f16x2 v = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, w ^ 0x80808080u, SEL)) + bias;
    return __builtin_bit_cast(uint32_t, v);
}

// A dword as two fp16 values. Takes the dword by value: __builtin_bit_cast
// applied directly to an ext_vector element (v[i]) reads element 0.
__device__ __forceinline__ f16x2 as_f16x2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }

// 16 codes of one row of B -> the B operands of two MFMAs (codes 0-7, 8-15).
__device__ __forceinline__ void codes16_to_operands(const u32x4 v, f16x8& b0, f16x8& b1) {
    const u32x4 x = {codes_to_f16x2<0x04010400u>(v[0]), codes_to_f16x2<0x04030402u>(v[0]),
                     codes_to_f16x2<0x04010400u>(v[1]), codes_to_f16x2<0x04030402u>(v[1])};
    const u32x4 y = {codes_to_f16x2<0x04010400u>(v[2]), codes_to_f16x2<0x04030402u>(v[2]),
                     codes_to_f16x2<0x04010400u>(v[3]), codes_to_f16x2<0x04030402u>(v[3])};
    b0 = __builtin_bit_cast(f16x8, x);
    b1 = __builtin_bit_cast(f16x8, y);
}

// MT tiles of 16 rows of A x one tile of 16 rows of B per block. The WAVES
// waves split K in 128-k batches (batch b goes to wave b % WAVES); each loads
// U batches, then multiplies them, and the waves' partial sums are added
// through LDS in wave order. B is read in whole 128-byte lines (8 rows x 128
// codes per instruction) and reordered into the MFMA layout through a per-wave
// LDS buffer, as in the split kernel below.
//
// Products that share A (ng_gemm_int8_shared_a) run in one launch of the
// *_shared_kernel forms of this kernel and of the GEMV kernel below: blocks
// first[p] .. first[p + 1] - 1 run product p exactly as the blocks 0 .. of its
// own launch would, so each C is bit-identical to its own call. A product's
// pointers are picked with selects, not by indexing the argument arrays
// (which would copy them to scratch memory).
constexpr int kMaxShared = 4;
struct SharedSet {
    uint16_t* c[kMaxShared];
    const int8_t* b[kMaxShared];
    const float* scale[kMaxShared];
    int n[kMaxShared];
    int first[kMaxShared];  // first block of each product, increasing; INT_MAX past the last
};

// Per-product split-K parameters (gemm_i8w_split_shared_kernel): the
// product's partial-sum region, its slice count, tiles of B, batches per
// slice and row tiles.
struct SplitSet {
    float* part[kMaxShared];
    int S[kMaxShared];
    int tiles[kMaxShared];
    int cps[kMaxShared];
    int TT[kMaxShared];
};

// Element p of four (a select chain on a wave-uniform p).
template <typename V>
__device__ __forceinline__ V pick4(int p, V v0, V v1, V v2, V v3) {
    return p == 0 ? v0 : p == 1 ? v1 : p == 2 ? v2 : v3;
}

// Runs block(c, b, scale, n, block index within the product, p) for the
// product p that owns this block.
template <typename F>
__device__ __forceinline__ void shared_dispatch(const SharedSet& s, F&& block) {
    const int blk = blockIdx.x;
    const int p = (blk >= s.first[1]) + (blk >= s.first[2]) + (blk >= s.first[3]);
    block(pick4(p, s.c[0], s.c[1], s.c[2], s.c[3]), pick4(p, s.b[0], s.b[1], s.b[2], s.b[3]),
          pick4(p, s.scale[0], s.scale[1], s.scale[2], s.scale[3]), pick4(p, s.n[0], s.n[1], s.n[2], s.n[3]),
          blk - pick4(p, s.first[0], s.first[1], s.first[2], s.first[3]), p);
}

template <int MT, int NT, int WAVES, int U>
__device__ __forceinline__ void gemm_i8w_block(uint16_t* __restrict__ c, const uint16_t* __restrict__ a,
                                               const int8_t* __restrict__ b, const float* __restrict__ scale,
                                               int M, int N, int K, int blk) {
    static_assert(NT == 1, "one tile of B per block");
    __shared__ f32x4 partial[WAVES - 1][MT][kWave];
    __shared__ __align__(16) u32x4 lds_b[WAVES][2 * kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane & 15;
    const int grp = lane >> 4;
    const int n0 = blk * 16;
    const int nbatch = (K + 127) / 128;
    const bool half_last = (K % 128) != 0;

    const int8_t* brow[2];
    int bpiece[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int r = 8 * j + (lane >> 3);
        bpiece[j] = (lane & 7) ^ (r >> 1);
        brow[j] = b + static_cast<size_t>(min(n0 + r, N - 1)) * K;
    }
    const uint16_t* ap[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) ap[t] = a + static_cast<size_t>(min(16 * t + col, M - 1)) * K + 16 * grp;

    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int cnt = wave < nbatch ? (nbatch - wave + WAVES - 1) / WAVES : 0;
    if (cnt > 0) {
        const int last = wave + (cnt - 1) * WAVES;
        u32x4 bv[U][2];
        u32x4 av[U][MT][2][2];
        auto load = [&](int slot, int i) {
            // Batches past this wave's last are clamped to it (and skipped in multiply).
            const int bt = min(wave + i * WAVES, last);
            const bool half = half_last && bt == nbatch - 1;
            const size_t kb = static_cast<size_t>(bt) * 128;
#pragma unroll
            for (int j = 0; j < 2; ++j) bv[slot][j] = ld16_stream(brow[j] + kb + 16 * (half ? (bpiece[j] & 3) : bpiece[j]));
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    const size_t k = kb + ((half && st == 1) ? 0 : 64 * st);
                    av[slot][t][st][0] = ld16(ap[t] + k);
                    av[slot][t][st][1] = ld16(ap[t] + k + 8);
                }
        };
        auto multiply = [&](int u, int i) {
            const int bt = wave + i * WAVES;
            const bool past = i >= cnt;
            const bool half = half_last && bt == nbatch - 1;
            lds_b[wave][lane] = bv[u][0];
            lds_b[wave][kWave + lane] = bv[u][1];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                // A batch past this wave's last, and the second half of a half
                // batch, hold reloaded codes and activations: skipped (an inf
                // activation times a zero code would give NaN).
                if (past || (half && st == 1)) continue;
                const int p = 4 * st + grp;
                const u32x4 v = lds_b[wave][8 * col + (p ^ (col >> 1))];
                f16x8 b0, b1;
                codes16_to_operands(v, b0, b1);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av[u][t][st][0]), b0,
                                                                    acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av[u][t][st][1]), b1,
                                                                    acc[t], 0, 0, 0);
                }
            }
            __builtin_amdgcn_wave_barrier();
        };
        for (int i = 0; i < cnt; i += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) load(u, i + u);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) multiply(u, i + u);
        }
    }

    if (wave > 0) {
#pragma unroll
        for (int i = 0; i < MT; ++i) partial[wave - 1][i][lane] = acc[i];
    }
    __syncthreads();
    if (wave != 0) return;
    const int n = n0 + col;
    const float s = scale[min(n, N - 1)];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        f32x4 v = acc[i];
#pragma unroll
        for (int w = 0; w < WAVES - 1; ++w) v += partial[w][i][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = 16 * i + 4 * grp + e;
            if (m < M && n < N) c[static_cast<size_t>(m) * N + n] = from_f32<f16>(v[e] * s);
        }
    }
}

template <int MT, int NT, int WAVES, int U>
__global__ __launch_bounds__(WAVES * kWave) void gemm_i8w_kernel(uint16_t* __restrict__ c,
                                                                  const uint16_t* __restrict__ a,
                                                                  const int8_t* __restrict__ b,
                                                                  const float* __restrict__ scale, int M, int N,
                                                                  int K) {
    gemm_i8w_block<MT, NT, WAVES, U>(c, a, b, scale, M, N, K, blockIdx.x);
}

template <int MT, int NT, int WAVES, int U>
__global__ __launch_bounds__(WAVES * kWave) void gemm_i8w_shared_kernel(SharedSet s, const uint16_t* __restrict__ a,
                                                                         int M, int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int) {
        gemm_i8w_block<MT, NT, WAVES, U>(c, a, b, scale, M, n, K, blk);
    });
}

template <int MT, int NT, int WAVES, int U>
int launch_i8w(uint16_t* c, const uint16_t* a, const int8_t* b, const float* scale, int M, int N, int K) {
    const unsigned blocks = static_cast<unsigned>((N + 16 * NT - 1) / (16 * NT));
    gemm_i8w_kernel<MT, NT, WAVES, U>
        <<<dim3(blocks), dim3(WAVES * kWave), 0, stream()>>>(c, a, b, scale, M, N, K);
    NG_CHECK_LAUNCH("cuda_gemm_int8");
    return 0;
}

// ---- GEMV-shaped variant (M <= 4) -------------------------------------------
// With one to four rows of A the MFMA layout costs a 16-byte load of A per
// 16 codes in every lane and reads 64 bytes per row of B per instruction.
// Here lane l of a wave takes codes [16l, 16l + 16) of a 1024-code segment, so
// each load instruction reads 1 KiB contiguous of one row of B; the lane's A
// values for that segment are loaded once and reused for R rows. Products are
// summed with v_dot2_f32_f16 (pairs of fp16 products, fp32 sums); the block's
// waves take different segments, and the 256 partial sums of each output are
// added through LDS in a fixed order.
constexpr int kGvWaves = 4;
constexpr int kGvSeg = 1024;  // codes per wave step: 64 lanes x 16

// The products of one 1024-code segment in one lane: R rows of B (codes
// bv[r]) against the lane's 16 values of each of MR rows of A (av[m]). Lanes
// past K pass zeros in both operands: an inf activation times a zero code
// would give NaN.
template <int MR, int R>
__device__ __forceinline__ void gemv_segment(float (&acc)[R][MR], u32x4 (&av)[MR][2], const u32x4 (&bv)[R],
                                             bool kin) {
    if (!kin) {
#pragma unroll
        for (int m = 0; m < MR; ++m) av[m][0] = av[m][1] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const u32x4 q = kin ? bv[r] : u32x4{0u, 0u, 0u, 0u};
        f16x8 w0, w1;
        codes16_to_operands(q, w0, w1);
        const u32x4 wl = __builtin_bit_cast(u32x4, w0), wh = __builtin_bit_cast(u32x4, w1);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float s = acc[r][m];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s = __builtin_amdgcn_fdot2(as_f16x2(av[m][0][j]), as_f16x2(wl[j]), s, false);
                s = __builtin_amdgcn_fdot2(as_f16x2(av[m][1][j]), as_f16x2(wh[j]), s, false);
            }
            acc[r][m] = s;
        }
    }
}

// The block's sums: output o = r * MR + m adds red[(w * V + o) * 64 + l] over
// waves w and lanes l; kParts threads add 256 / kParts values each, then one
// thread adds the parts, both in a fixed order. Thread o < V returns output
// o's sum (others 0). The reduction buffer is free again after a barrier.
template <int MR, int R>
__device__ __forceinline__ float gemv_reduce(const float (&acc)[R][MR]) {
    constexpr int V = R * MR;                 // outputs per block
    constexpr int kParts = kGvWaves * kWave / V;  // threads that share one output in the first reduction stage
    static_assert(kGvWaves * kWave % V == 0 && kWave % kParts == 0, "reduction shape");
    __shared__ float red[kGvWaves * V * kWave];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) red[(wave * V + r * MR + m) * kWave + lane] = acc[r][m];
    __syncthreads();
    const int o = tid % V;
    const int part = tid / V;
    constexpr int kPerPart = kGvWaves * kWave / kParts;  // values summed by one thread
    float sum = 0.0f;
#pragma unroll 4
    for (int j = 0; j < kPerPart; ++j) {
        const int idx = part * kPerPart + j;  // (wave, lane) pair
        sum += red[((idx / kWave) * V + o) * kWave + idx % kWave];
    }
    __syncthreads();
    red[o * kParts + part] = sum;
    __syncthreads();
    float v = 0.0f;
    if (tid < V)
        for (int q = 0; q < kParts; ++q) v += red[tid * kParts + q];
    return v;
}

// C = fp16(sum * scale) for the block's rows n0 .. n0 + R - 1 of B.
template <int MR, int R>
__device__ __forceinline__ void gemv_finish(const float (&acc)[R][MR], uint16_t* __restrict__ c,
                                            const float* __restrict__ scale, int M, int N, int n0) {
    const float v = gemv_reduce<MR, R>(acc);
    const int tid = threadIdx.x;
    if (tid < R * MR) {
        const int r = tid / MR, m = tid % MR, n = n0 + r;
        if (m < M && n < N) c[static_cast<size_t>(m) * N + n] = from_f32<f16>(v * scale[n]);
    }
}

// One lane's sums of the GEMV kernels' block for rows n0 .. n0 + R - 1 of B.
template <int MR, int R>
__device__ __forceinline__ void gemv_i8w_sums(float (&acc)[R][MR], const uint16_t* __restrict__ a,
                                              const int8_t* __restrict__ b, int M, int N, int K, int n0) {
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int nseg = (K + kGvSeg - 1) / kGvSeg;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[r][m] = 0.0f;

    for (int sg = wave; sg < nseg; sg += kGvWaves) {
        const int k = sg * kGvSeg + 16 * lane;
        const bool kin = k < K;           // the last segment may end early (K % 16 == 0)
        const int kc = kin ? k : K - 16;  // lanes past K load the last codes and multiply zeros
        u32x4 av[MR][2];
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const uint16_t* ar = a + static_cast<size_t>(min(m, M - 1)) * K + kc;
            av[m][0] = ld16(ar);
            av[m][1] = ld16(ar + 8);
        }
        u32x4 bv[R];
#pragma unroll
        for (int r = 0; r < R; ++r) bv[r] = ld16_stream(b + static_cast<size_t>(min(n0 + r, N - 1)) * K + kc);
        __builtin_amdgcn_sched_barrier(0);
        gemv_segment<MR, R>(acc, av, bv, kin);
    }
}

// One block of the GEMV kernels: rows blk R .. blk R + R - 1 of B.
template <int MR, int R>
__device__ __forceinline__ void gemv_i8w_block(uint16_t* __restrict__ c, const uint16_t* __restrict__ a,
                                               const int8_t* __restrict__ b, const float* __restrict__ scale,
                                               int M, int N, int K, int blk) {
    float acc[R][MR];
    gemv_i8w_sums<MR, R>(acc, a, b, M, N, K, blk * R);
    gemv_finish<MR, R>(acc, c, scale, M, N, blk * R);
}

template <int MR, int R>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_kernel(uint16_t* __restrict__ c,
                                                                    const uint16_t* __restrict__ a,
                                                                    const int8_t* __restrict__ b,
                                                                    const float* __restrict__ scale, int M, int N,
                                                                    int K) {
    gemv_i8w_block<MR, R>(c, a, b, scale, M, N, K, blockIdx.x);
}

template <int MR, int R>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_shared_kernel(SharedSet s, const uint16_t* __restrict__ a,
                                                                           int M, int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int) {
        gemv_i8w_block<MR, R>(c, a, b, scale, M, n, K, blk);
    });
}

// gate/up and SwiGLU in one launch (ng_gemm_int8_silu_mul): block blk runs
// the GEMV kernel's block blk of the gate product and of the up product (the
// same R rows of each, both against one load of A), reduces each exactly as
// that block does, and writes gate = fp16(sum * scale), up likewise, and
// out = fp16(silu(gate) * up) with the element-wise kernel's expression. out
// may be gate or up itself: each element is written by one thread, out last.
struct SwigluArgs {
    uint16_t* out;
    uint16_t* gate;
    uint16_t* up;
    const int8_t* bg;
    const int8_t* bu;
    const float* sg;
    const float* su;
};

template <int MR, int R>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_swiglu_kernel(SwigluArgs sa, const uint16_t* __restrict__ a,
                                                                           int M, int N, int K) {
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int n0 = blockIdx.x * R;
    const int nseg = (K + kGvSeg - 1) / kGvSeg;
    float accg[R][MR], accu[R][MR];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) accg[r][m] = accu[r][m] = 0.0f;
    for (int sg = wave; sg < nseg; sg += kGvWaves) {
        const int k = sg * kGvSeg + 16 * lane;
        const bool kin = k < K;
        const int kc = kin ? k : K - 16;
        u32x4 av[MR][2];
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const uint16_t* ar = a + static_cast<size_t>(min(m, M - 1)) * K + kc;
            av[m][0] = ld16(ar);
            av[m][1] = ld16(ar + 8);
        }
        u32x4 bvg[R], bvu[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const size_t row = static_cast<size_t>(min(n0 + r, N - 1)) * K + kc;
            bvg[r] = ld16_stream(sa.bg + row);
            bvu[r] = ld16_stream(sa.bu + row);
        }
        __builtin_amdgcn_sched_barrier(0);
        gemv_segment<MR, R>(accg, av, bvg, kin);
        gemv_segment<MR, R>(accu, av, bvu, kin);
    }
    const float vg = gemv_reduce<MR, R>(accg);
    __syncthreads();  // the reduction buffer is reused
    const float vu = gemv_reduce<MR, R>(accu);
    if (tid < R * MR) {
        const int r = tid / MR, m = tid % MR, n = n0 + r;
        if (m < M && n < N) {
            const size_t o = static_cast<size_t>(m) * N + n;
            const uint16_t g = from_f32<f16>(vg * sa.sg[n]), u = from_f32<f16>(vu * sa.su[n]);
            sa.gate[o] = g;
            sa.up[o] = u;
            sa.out[o] = from_f32<f16>(swiglu_f32(to_f32<f16>(g), to_f32<f16>(u)));
        }
    }
}

// A product and the residual add after it (ng_gemm_int8_add): the GEMV
// kernel's blocks, then out = fp16(c + residual) on the rounded product, as
// cuda_add computes it. out may be c or the residual itself: each element is
// written by one thread, out last.
template <int MR, int R>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_add_kernel(uint16_t* out, uint16_t* c,
                                                                        const uint16_t* res,
                                                                        const uint16_t* __restrict__ a,
                                                                        const int8_t* __restrict__ b,
                                                                        const float* __restrict__ scale, int M,
                                                                        int N, int K) {
    const int n0 = blockIdx.x * R;
    float acc[R][MR];
    gemv_i8w_sums<MR, R>(acc, a, b, M, N, K, n0);
    const float v = gemv_reduce<MR, R>(acc);
    const int tid = threadIdx.x;
    if (tid < R * MR) {
        const int r = tid / MR, m = tid % MR, n = n0 + r;
        if (m < M && n < N) {
            const size_t o = static_cast<size_t>(m) * N + n;
            const uint16_t cv = from_f32<f16>(v * scale[n]);
            const float sum = to_f32<f16>(cv) + to_f32<f16>(res[o]);
            c[o] = cv;
            out[o] = from_f32<f16>(sum);
        }
    }
}

// RMSNorm (or residual add + RMSNorm) folded into the shared GEMV launch
// (ng_rmsnorm_gemm_int8_shared_a, ng_add_rmsnorm_gemm_int8_shared_a), for
// M <= 2 rows of K <= 8192. Every block normalises the rows itself, and each
// thread normalises exactly the 16-value pieces of A that its lane multiplies
// in the GEMV (segment sg = wave + 4 s, values 16 lane .. 16 lane + 15), so A
// stays in registers: the thread loads its pieces of x (and the residual) and
// of the norm weight, then its rows of B, and the row statistic (one block
// barrier for all rows) and the scaling run while the codes are in flight.
// Each block gets cuda_rmsnorm's (cuda_add_rmsnorm's) bits: the statistic is
// the sum of squares rounded once to fp32 (fp64 sums resolved with their
// error bound, else exact limb sums), which does not depend on the order of
// summation, and the scaling is the same expression. The products are the
// GEMV block's own segment and reduction code, so C is bit-identical too. The
// first block of the launch stores the normalised rows (and the residual sums).
struct NormArgs {
    const uint16_t* x;
    const uint16_t* res;  // residual input (ADD)
    const uint16_t* w;    // norm weight [K]
    uint16_t* normed;     // [M, K]
    uint16_t* res_out;    // [M, K] (ADD)
    float eps;
};

// Row m's exact statistic from the limb sums of the whole row, read from
// memory by every thread of the block (the fast path's rare fallback; the
// decision is uniform over the block).
template <bool ADD>
__device__ __noinline__ float norm_row_ss_exact(const NormArgs& na, int m, int K) {
    constexpr int kT = kGvWaves * kWave;
    __shared__ double s_limb[kGvWaves][3];
    __shared__ int s_flag[kGvWaves];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
    const uint16_t* xr = na.x + static_cast<size_t>(m) * K;
    const uint16_t* rr = ADD ? na.res + static_cast<size_t>(m) * K : nullptr;
    Limbs Lm{0.0, 0.0, 0.0, 0};
    for (int vi = tid; vi < K / 8; vi += kT) {
        float fx[8];
        unpack8<f16>(ld16(xr + vi * 8), fx);
        if (ADD) {
            float fr[8];
            unpack8<f16>(ld16(rr + vi * 8), fr);
#pragma unroll
            for (int i = 0; i < 8; ++i) fx[i] = fx[i] + fr[i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) limbs_add(Lm, fx[i]);
    }
    double t = wave_sum_f64_dpp(Lm.t), u = wave_sum_f64_dpp(Lm.u), w = wave_sum_f64_dpp(Lm.w);
    int bad = static_cast<int>(wave_max_u32_dpp(static_cast<uint32_t>(Lm.bad)));
    __syncthreads();  // a previous row's readers are done with s_limb
    if (lane == 0) {
        s_limb[wid][0] = t;
        s_limb[wid][1] = u;
        s_limb[wid][2] = w;
        s_flag[wid] = bad;
    }
    __syncthreads();
    t = u = w = 0.0;
    bad = 0;
    for (int j = 0; j < kGvWaves; ++j) {
        t += s_limb[j][0];
        u += s_limb[j][1];
        w += s_limb[j][2];
        bad |= s_flag[j];
    }
    return bad ? -1.0f : limbs_to_f32(t, u, w);
}

// One block of the fused kernels: the rows of A normalised in registers, then
// the products of the GEMV kernel's block blk (rows blk R .. blk R + R - 1 of
// B), exactly as that block computes them. SEGS: the most 1024-value segments
// of K one wave takes (K <= 4096 SEGS).
// RoPE on two of the products (ng_rmsnorm_qkv_rope_int8): split-half pairs
// (i, i + D/2) of each head of D values, as cuda_rope_with_theta style 0,
// for the tokens' positions.
constexpr int kRopeEpiMaxHalf = 128;  // D <= 256
struct RopeEpi {
    const int* pos;  // [M]
    int D;
    int half;  // D / 2
    int bph;   // blocks per head: half / 4
    float inv_freq[kRopeEpiMaxHalf];
};

template <int MR, int R, int SEGS, bool ADD, bool ROPE = false>
__device__ __forceinline__ void gemv_i8w_norm_block(uint16_t* __restrict__ c, const int8_t* __restrict__ b,
                                                    const float* __restrict__ scale, const NormArgs& na, int M,
                                                    int N, int K, int blk, bool store, bool rope = false,
                                                    const RopeEpi* re = nullptr) {
    static_assert(!ROPE || R == 8, "a RoPE block holds four rotation pairs");
    __shared__ double s_part[kGvWaves][MR];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int n0 = blk * R;
    const int nseg = (K + kGvSeg - 1) / kGvSeg;
    // Row of B (and of C) in slot r: n0 + r, or for a rotated product the
    // block's four pairs of one head, rows h D + q + r (r < 4) and
    // h D + D/2 + q + r - 4. An output's sums do not depend on its slot, so
    // each row gets the GEMV kernel's bits either way.
    // The geometry is read whether or not this product rotates: a read under
    // the product's flag put a branch and a scalar-load wait before every code
    // load.
    const bool rot = ROPE && rope;
    const int rbph = ROPE ? re->bph : 1, rD = ROPE ? re->D : 0, rhalf = ROPE ? re->half : 0;
    const int rh = rot ? blk / rbph : 0;
    const int rq = rot ? (blk - rh * rbph) * 4 : 0;
    const int lo = rot ? rh * rD + rq : n0;              // slots 0 .. 3: rows lo + r
    const int hi = rot ? rh * rD + rhalf + rq - 4 : n0;  // slots 4 .. 7: rows hi + r
    const auto row_of = [&](int r) { return (r < 4 ? lo : hi) + r; };

    // Loads: the lane's pieces of x (res) and w, then its rows of B. They are
    // issued without branches, so that waiting for the first ones does not
    // wait for the codes: a wave with no segment s (sg >= nseg) has every lane
    // past K, at K - 16, and its loads of that segment hit one line per row.
    bool kin[SEGS];
    int kc[SEGS];
    u32x4 xv[SEGS][MR][2], rv[SEGS][MR][2], wv[SEGS][2], bv[SEGS][R];
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
        const int k = (wave + s * kGvWaves) * kGvSeg + 16 * lane;
        kin[s] = k < K;
        kc[s] = kin[s] ? k : K - 16;
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const size_t off = static_cast<size_t>(min(m, M - 1)) * K + kc[s];
            xv[s][m][0] = ld16(na.x + off);
            xv[s][m][1] = ld16(na.x + off + 8);
            if (ADD) {
                rv[s][m][0] = ld16(na.res + off);
                rv[s][m][1] = ld16(na.res + off + 8);
            }
        }
        wv[s][0] = ld16(na.w + kc[s]);
        wv[s][1] = ld16(na.w + kc[s] + 8);
    }
#pragma unroll
    for (int s = 0; s < SEGS; ++s)
#pragma unroll
        for (int r = 0; r < R; ++r)
            bv[s][r] = ld16_stream(b + static_cast<size_t>(min(row_of(r), N - 1)) * K + kc[s]);
    __builtin_amdgcn_sched_barrier(0);

    // o = x, or the rounded sum x + res; squares of x, or of the unrounded
    // fp32 sum, as the row kernels take them. Lanes past K add nothing.
    double ssq[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) ssq[m] = 0.0;
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
        if (wave + s * kGvWaves >= nseg) continue;
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float s0, s1;
                    if (ADD) {
                        s0 = el_add<f16, 0>(xv[s][m][h][i], rv[s][m][h][i]);
                        s1 = el_add<f16, 1>(xv[s][m][h][i], rv[s][m][h][i]);
                        xv[s][m][h][i] = pack2<f16>(s0, s1);
                    } else {
                        s0 = el_get<f16, 0>(xv[s][m][h][i]);
                        s1 = el_get<f16, 1>(xv[s][m][h][i]);
                    }
                    const double d0 = kin[s] ? static_cast<double>(s0) : 0.0;
                    const double d1 = kin[s] ? static_cast<double>(s1) : 0.0;
                    ssq[m] = __builtin_fma(d0, d0, ssq[m]);
                    ssq[m] = __builtin_fma(d1, d1, ssq[m]);
                }
    }
    if (ADD && store) {
#pragma unroll
        for (int s = 0; s < SEGS; ++s)
#pragma unroll
            for (int m = 0; m < MR; ++m)
                if (kin[s] && m < M) {
                    uint16_t* ro = na.res_out + static_cast<size_t>(m) * K + kc[s];
                    st16(ro, xv[s][m][0]);
                    st16(ro + 8, xv[s][m][1]);
                }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        const double S = wave_sum_f64_dpp(ssq[m]);
        if (lane == 0) s_part[wave][m] = S;
    }
    __syncthreads();
    float rs[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        double S = s_part[0][m];
        for (int j = 1; j < kGvWaves; ++j) S += s_part[j][m];
        // Tree height: 16 SEGS terms in one lane, 6 across the wave, 3 across the waves.
        float ss;
        if (!ss_fast_resolve(S, 16 * SEGS + 10, ss)) {
            const float e = norm_row_ss_exact<ADD>(na, min(m, M - 1), K);
            if (e >= 0.0f) ss = e;
        }
        rs[m] = 1.0f / __builtin_sqrtf(ss / static_cast<float>(K) + na.eps);
    }

    // y = RN_f16(RN(o * r) * w): the GEMV's A, in registers.
    float acc[R][MR];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[r][m] = 0.0f;
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
        if (wave + s * kGvWaves >= nseg) continue;
        u32x4 av[MR][2];
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    av[m][h][i] = pack2<f16>(el_mul<f16, 0>(wv[s][h][i], el_mul<f16, 0>(xv[s][m][h][i], rs[m])),
                                             el_mul<f16, 1>(wv[s][h][i], el_mul<f16, 1>(xv[s][m][h][i], rs[m])));
        if (store) {
#pragma unroll
            for (int m = 0; m < MR; ++m)
                if (kin[s] && m < M) {
                    uint16_t* yo = na.normed + static_cast<size_t>(m) * K + kc[s];
                    st16(yo, av[m][0]);
                    st16(yo + 8, av[m][1]);
                }
        }
        gemv_segment<MR, R>(acc, av, bv[s], kin[s]);
    }
    if (!rot) {
        gemv_finish<MR, R>(acc, c, scale, M, N, n0);
        return;
    }
    // Rotated product: C = fp16(sum * scale) as the GEMV kernel rounds it, then
    // RoPE on the rounded pair, with cuda_rope_with_theta's angle, sincosf and
    // expression, rounded once more. Slot r's partner is r ^ 4 (thread
    // tid ^ 4 MR, in the first wave).
    constexpr int V = R * MR;
    const float v = gemv_reduce<MR, R>(acc);
    float x = 0.0f;
    int r = 0, m = 0, row = 0;
    if (tid < V) {
        r = tid / MR;
        m = tid % MR;
        row = row_of(r);
        x = to_f32<f16>(from_f32<f16>(v * scale[row]));
    }
    const float xp = __shfl_xor(x, 4 * MR, kWave);
    if (tid < V && m < M) {
        float sn, cs;
        sincosf(static_cast<float>(re->pos[m]) * re->inv_freq[rq + (r & 3)], &sn, &cs);
        const float y = r < 4 ? x * cs - xp * sn : xp * sn + x * cs;
        c[static_cast<size_t>(m) * N + row] = from_f32<f16>(y);
    }
}

template <int MR, int R, int SEGS, bool ADD>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_norm_shared_kernel(SharedSet s, NormArgs na, int M,
                                                                                int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int) {
        gemv_i8w_norm_block<MR, R, SEGS, ADD>(c, b, scale, na, M, n, K, blk, blockIdx.x == 0);
    });
}

// The same with RoPE on products 0 and 1 (q and k).
template <int MR, int SEGS>
__global__ __launch_bounds__(kGvWaves * kWave) void gemv_i8w_norm_rope_shared_kernel(SharedSet s, NormArgs na,
                                                                                     RopeEpi re, int M, int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int p) {
        gemv_i8w_norm_block<MR, 8, SEGS, false, true>(c, b, scale, na, M, n, K, blk, blockIdx.x == 0, p < 2, &re);
    });
}

template <int MR, int R>
int launch_gemv_shared(const SharedSet& set, int blocks, const uint16_t* a, int M, int K) {
    gemv_i8w_shared_kernel<MR, R><<<dim3(static_cast<unsigned>(blocks)), dim3(kGvWaves * kWave), 0, stream()>>>(
        set, a, M, K);
    NG_CHECK_LAUNCH("ng_gemm_int8_shared_a");
    return 0;
}

// Longest rows the fused norm kernels take: two segments per wave.
constexpr int kNormSharedMaxK = 2 * kGvWaves * kGvSeg;
// Most GEMV blocks of a fused norm launch. The fused kernel holds more
// registers than the GEMV kernel (5 waves per SIMD against 8 at one row):
// where the launch fits the GPU in about one round of blocks, folding the
// norm in saves its launch and its latency; with more blocks the launch is
// bound by the codes in flight, and the two calls are faster (measured on
// MI355X at Mistral-7B: q/k/v, 768 blocks, 7.2 against 8.3 us at one token;
// gate/up, 3584 blocks, 23.1 against 21.8 us). Only the GEMV shapes of one
// and two rows (8 rows of B per block) are folded: with four rows the fused
// kernel was slower at every block count measured (TinyLlama's q/k/v, 640
// blocks, 3 rows: 7.9 against 6.4 us).
constexpr int kNormSharedMaxBlocks = 1024;

template <int MR, int R, bool ADD>
int launch_gemv_norm_shared(const SharedSet& set, int blocks, const NormArgs& na, int M, int K) {
    const dim3 grid(static_cast<unsigned>(blocks)), block(kGvWaves * kWave);
    if (K <= kGvWaves * kGvSeg)
        gemv_i8w_norm_shared_kernel<MR, R, 1, ADD><<<grid, block, 0, stream()>>>(set, na, M, K);
    else
        gemv_i8w_norm_shared_kernel<MR, R, 2, ADD><<<grid, block, 0, stream()>>>(set, na, M, K);
    NG_CHECK_LAUNCH(ADD ? "ng_add_rmsnorm_gemm_int8_shared_a" : "ng_rmsnorm_gemm_int8_shared_a");
    return 0;
}

template <int MR, int R>
int launch_gemv(uint16_t* c, const uint16_t* a, const int8_t* b, const float* scale, int M, int N, int K) {
    const unsigned blocks = static_cast<unsigned>((N + R - 1) / R);
    gemv_i8w_kernel<MR, R><<<dim3(blocks), dim3(kGvWaves * kWave), 0, stream()>>>(c, a, b, scale, M, N, K);
    NG_CHECK_LAUNCH("cuda_gemm_int8");
    return 0;
}

// ---- split-K variant --------------------------------------------------------
// Up to 32 rows of A. For more than a few rows the kernel above reads A from L2
// once per 16 rows of B: at M = 32 that is 4 bytes of A per weight byte. Here a
// block of W waves owns 16 W rows of B and one of S slices of K; the A columns
// of each 128-k batch are staged once in LDS and shared by the block's waves
// (2M / (16 W) bytes of A per weight byte). W = 4, or 8 for K >= 8192 above 16
// rows (the down projection); 8 waves were slower at K = 4096, and 2 slower
// everywhere but N = 1024. The kernel of 33 to 128 rows does not pay here: its
// smallest tile is 32 rows, and at 8 rows gate/up took it 25.8 against 24.9 us.
//
// B is read in whole 128-byte lines: each load instruction of a wave covers
// 8 rows x 128 codes (8 lanes per row), two instructions a wave's 16 rows.
// Loading B straight into the MFMA layout instead (4 lanes per row, 64 bytes
// per row per instruction) streams about 25% slower on MI355X. The codes
// reach the MFMA layout through a per-wave LDS buffer: piece p (16 codes) of
// row r sits in slot 8r + (p xor r / 2), so the writes are contiguous and the
// reads conflict-free. (LDS on MI355X serves 256 bytes per clock from 64
// banks. Measured with access-pattern probes, 16-byte reads are conflict-free
// when the rows 0-7 of one lane group and the rows 8-15 of another fall in
// opposite halves of the banks; (p + r / 2) mod 8 breaks that and took two
// clocks per 16 lanes.)
//
// K is divided among blocks and inside them. The G groups of W waves of a
// block take turns of G consecutive batches (group g the batch g of each
// turn), each group with its own LDS copy of its batch of A; at the end the
// groups' sums are added through LDS in group order. With S > 1 each block
// stores those sums in `part` [S][M][N] and a second kernel adds the S slices
// in slice order. Either way the result does not depend on timing. (Having
// the last block of each tile add the slices instead needs an agent-scope
// release and acquire per block, which on MI355X write back and invalidate
// the whole L2: measured 3-5x slower.) Groups inside the block replace slices
// where there are enough tiles to fill the GPU with one slice: no partial
// sums in memory and no second launch.
constexpr int kBatch = 128;  // k per batch

// SW (ng_gemm_int8_silu_mul, one K slice): the block's first
// W/2 waves of each group take rows of the gate product and the last W/2 the
// same rows of the up product (8 W row pairs per block instead of 16 W rows of
// one product). A wave's sums depend only on its own 16 rows of B, which start
// at a multiple of 16 either way, so gate and up are the values of their own
// launches; the up waves hand their rounded values to the gate waves through
// LDS, which write gate, up and fp16(silu(gate) * up).
template <int MT, int W, int G, bool SW = false>
__device__ __forceinline__ void gemm_i8w_split_block(
    uint16_t* __restrict__ c, const uint16_t* __restrict__ a, const int8_t* __restrict__ b,
    const float* __restrict__ scale, float* __restrict__ part, int M, int N, int K, int S, int cps, int blk,
    const SwigluArgs* sw = nullptr) {
    static_assert(!SW || W % 2 == 0, "SW splits the waves of a group in two");
    // A batch of A in LDS: 256 bytes per row, padded by 32 (6% faster at 17-32
    // rows than an xor swizzle without conflicts).
    constexpr int kRowBytes = kBatch * 2 + 32;
    constexpr int kPieces = 16 * MT * 16;       // 16-byte pieces of A per batch
    constexpr int kThreads = G * W * kWave;
    static_assert((G * kPieces) % kThreads == 0, "A pieces must divide among the threads");
    static_assert(G == 1 || (G - 1) * W * MT * kWave * 16 <= 2 * G * 16 * MT * kRowBytes,
                  "the groups' sums must fit in the A buffers");
    __shared__ __align__(16) uint8_t lds_a[2][G][16 * MT * kRowBytes];
    __shared__ __align__(16) u32x4 lds_b[G * W][2 * kWave];

    const int sl = blk % S;
    const int tile = blk / S;

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int kg = wave / W;   // this wave's group: batch kg of each turn
    const int wv = wave % W;   // and its tile of 16 rows of B
    const int col = lane & 15;
    const int grp = lane >> 4;
    const int nbatch = (K + kBatch - 1) / kBatch;  // the last batch holds 64 k when K % 128 == 64
    const bool half_last = (K % kBatch) != 0;
    const int c0 = sl * cps;
    const int c1 = min(c0 + cps, nbatch);
    const bool upw = SW && wv >= W / 2;  // SW: this wave takes the up product's rows
    const int nw = SW ? tile * (8 * W) + 16 * (wv % (W / 2)) : tile * (16 * W) + 16 * wv;  // first row of B
    const int n = nw + col;                                 // row of B this lane multiplies
    if constexpr (SW) {
        b = upw ? sw->bu : sw->bg;
        scale = upw ? sw->su : sw->sg;
    }

    // A and B are read with buffer loads: B from this wave's first row (rows
    // past N clamp to the last one), A from its start, so that per-load
    // offsets are 32-bit instead of 64-bit addresses. Offsets are below 16 K
    // bytes for B and 2 M K bytes for A.
    const int nbase = min(nw, N - 1);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(b + static_cast<size_t>(nbase) * K), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a), 0, 0x7fffffff,
                                                                        0x00020000);
    uint32_t boff[2];
    int bpiece[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int r = 8 * j + (lane >> 3);
        bpiece[j] = (lane & 7) ^ (r >> 1);
        boff[j] = static_cast<uint32_t>((min(nw + r, N - 1) - nbase) * K);
    }
    constexpr int kP = G * kPieces / kThreads;
    uint32_t aoff[kP];
#pragma unroll
    for (int j = 0; j < kP; ++j) {
        const int pc = (j * kThreads + tid) % kPieces;
        aoff[j] = static_cast<uint32_t>(min(pc / 16, M - 1) * K * 2);
    }

    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Turns, two in flight: the loads of turn i + 1 (B into registers, A
    // into registers on their way to LDS) are issued before turn i is
    // multiplied; A alternates between two LDS buffers, so one barrier per
    // turn separates a buffer's writes from its reads and from its reuse two
    // turns later. A turn starting at batch `first` holds batches first ..
    // first + G - 1; those past the slice load its last batch (every load
    // stays unconditional) and are skipped by multiply.
    // A first: staging it into LDS then waits only for A, not for B.
    auto load = [&](u32x4 (&bv)[2], u32x4 (&ar)[kP], int first) {
#pragma unroll
        for (int j = 0; j < kP; ++j) {
            const int pc = j * kThreads + tid;
            const int cb = min(first + pc / kPieces, c1 - 1);
            const size_t kb = static_cast<size_t>(cb) * kBatch;
            int q = pc % 16;
            if (half_last && cb == nbatch - 1) q &= 7;  // k past K: load the batch's first 64 k again
            ar[j] = __builtin_amdgcn_raw_buffer_load_b128(ra, aoff[j] + static_cast<uint32_t>((kb + 8 * q) * 2), 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep A's loads ahead of B's
        // Pieces 4-7 of a half batch would lie past K: they load pieces 0-3
        // again (and are skipped by multiply).
        const int cb = min(first + kg, c1 - 1);
        const bool half = half_last && cb == nbatch - 1;
        const size_t kb = static_cast<size_t>(cb) * kBatch;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int pcs = half ? (bpiece[j] & 3) : bpiece[j];
            bv[j] = __builtin_amdgcn_raw_buffer_load_b128(rb, boff[j] + static_cast<uint32_t>(kb + 16 * pcs), 0, 2);
        }
    };
    auto stage = [&](int buf, const u32x4 (&ar)[kP]) {
#pragma unroll
        for (int j = 0; j < kP; ++j) {
            const int pc = j * kThreads + tid;
            const int g = pc / kPieces;
            const int row = (pc % kPieces) / 16;
            *reinterpret_cast<u32x4*>(lds_a[buf][g] + row * kRowBytes + 16 * (pc % 16)) = ar[j];
        }
    };
    auto multiply = [&](int buf, const u32x4 (&bv)[2], int first) {
        // This wave's codes into the MFMA layout. LDS operations of one wave
        // complete in order, so the reads see the writes, and the next batch's
        // writes come after these reads.
        lds_b[wave][lane] = bv[0];
        lds_b[wave][kWave + lane] = bv[1];
        __builtin_amdgcn_wave_barrier();
        const int cb = first + kg;
        const bool past = cb >= c1;                               // clamped batch: skipped
        const bool half = half_last && cb == nbatch - 1;          // its second 64 k lie past K
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            // A clamped batch, and the second half of a half batch, hold
            // reloaded codes and activations: skipped (wave-uniform), so that
            // an inf activation never meets a padding code (inf * 0 = NaN).
            if (past || (half && st == 1)) continue;
            const int p = 4 * st + grp;
            const u32x4 v = lds_b[wave][8 * col + (p ^ (col >> 1))];
            f16x8 b0, b1;
            codes16_to_operands(v, b0, b1);
            // All tiles' first halves, then their second halves: consecutive
            // MFMAs update different accumulators.
            u32x4 a0[MT], a1[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                // pieces 8 st + 2 grp and the next one of row 16 t + col
                const uint8_t* ap = lds_a[buf][kg] + (16 * t + col) * kRowBytes;
                const int q0 = 8 * st + 2 * grp;
                a0[t] = *reinterpret_cast<const u32x4*>(ap + 16 * q0);
                a1[t] = *reinterpret_cast<const u32x4*>(ap + 16 * (q0 + 1));
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a0[t]), b0, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a1[t]), b1, acc[t], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    };
    // The turn count is rounded up to even: an extra turn past the slice
    // is skipped by multiply. (Leaving the loop after an odd turn instead lets
    // the compiler sink the next turn's loads below the multiply.)
    const int nt = (c1 - c0 + G - 1) / G;
    u32x4 bv0[2], bv1[2];
    u32x4 ar0[kP], ar1[kP];
    load(bv0, ar0, c0);
    for (int i = 0; i < nt; i += 2) {
        stage(0, ar0);
        __syncthreads();
        load(bv1, ar1, c0 + G * (i + 1));
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, bv0, c0 + G * i);
        stage(1, ar1);
        __syncthreads();
        load(bv0, ar0, c0 + G * (i + 2));
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, bv1, c0 + G * (i + 1));
    }

    if (G > 1) {
        // Groups 1 .. G-1 hand their sums to group 0 through the A buffers
        // (free once every wave has passed this barrier), which adds them in
        // group order.
        __syncthreads();
        f32x4* red = reinterpret_cast<f32x4*>(&lds_a[0][0][0]);
        if (kg > 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t) red[(((kg - 1) * W + wv) * MT + t) * kWave + lane] = acc[t];
        }
        __syncthreads();
        // SW keeps every wave to the epilogue's barriers.
        if (!SW && kg > 0) return;
        if (kg == 0) {
#pragma unroll
            for (int g = 1; g < G; ++g)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] += red[(((g - 1) * W + wv) * MT + t) * kWave + lane];
        }
    }
    if constexpr (SW) {
        // gate, up and SwiGLU (one K slice): the up waves of group 0 store
        // their rounded values, the gate waves of group 0 combine.
        __syncthreads();  // the group sums' reads of the A buffers are done
        uint16_t* xch = reinterpret_cast<uint16_t*>(&lds_a[0][0][0]);  // [W/2][MT][4][64]
        const int wp = wv % (W / 2);
        if (kg == 0 && upw && n < N) {
            const float sc = scale[n];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) xch[((wp * MT + t) * 4 + e) * kWave + lane] = from_f32<f16>(acc[t][e] * sc);
        }
        __syncthreads();
        if (kg == 0 && !upw && n < N) {
            const float sc = scale[n];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = 16 * t + 4 * grp + e;
                    if (m < M) {
                        const size_t o = static_cast<size_t>(m) * N + n;
                        const uint16_t gv = from_f32<f16>(acc[t][e] * sc);
                        const uint16_t uv = xch[((wp * MT + t) * 4 + e) * kWave + lane];
                        sw->gate[o] = gv;
                        sw->up[o] = uv;
                        sw->out[o] = from_f32<f16>(swiglu_f32(to_f32<f16>(gv), to_f32<f16>(uv)));
                    }
                }
        }
        return;
    }
    if (S == 1) {
        if (n < N) {
            const float sc = scale[n];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = 16 * t + 4 * grp + e;
                    if (m < M) c[static_cast<size_t>(m) * N + n] = from_f32<f16>(acc[t][e] * sc);
                }
        }
        return;
    }
    if (n < N) {
        float* mine = part + static_cast<size_t>(sl) * M * N;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = 16 * t + 4 * grp + e;
                if (m < M) mine[static_cast<size_t>(m) * N + n] = acc[t][e];
            }
    }
}

template <int MT, int W, int G>
__global__ __launch_bounds__(G * W * kWave) void gemm_i8w_split_kernel(
    uint16_t* __restrict__ c, const uint16_t* __restrict__ a, const int8_t* __restrict__ b,
    const float* __restrict__ scale, float* __restrict__ part, int M, int N, int K, int S, int cps) {
    gemm_i8w_split_block<MT, W, G>(c, a, b, scale, part, M, N, K, S, cps, blockIdx.x);
}

// gate/up and SwiGLU on the split kernel (ng_gemm_int8_silu_mul from 3 rows):
// one K slice, blocks of 8 W row pairs.
template <int MT, int W, int G>
__global__ __launch_bounds__(G * W * kWave) void gemm_i8w_split_swiglu_kernel(SwigluArgs sa,
                                                                               const uint16_t* __restrict__ a,
                                                                               int M, int N, int K, int cps) {
    gemm_i8w_split_block<MT, W, G, true>(nullptr, a, nullptr, nullptr, nullptr, M, N, K, 1, cps, blockIdx.x, &sa);
}

// Products that share A on one split-kernel shape (ng_gemm_int8_shared_a):
// each product keeps its own slices of K and its own region of the
// partial-sum buffer, so its sums are those of its own launch.
template <int MT, int W, int G>
__global__ __launch_bounds__(G * W * kWave) void gemm_i8w_split_shared_kernel(SharedSet s, SplitSet sp,
                                                                               const uint16_t* __restrict__ a, int M,
                                                                               int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int p) {
        gemm_i8w_split_block<MT, W, G>(c, a, b, scale, pick4(p, sp.part[0], sp.part[1], sp.part[2], sp.part[3]), M,
                                       n, K, pick4(p, sp.S[0], sp.S[1], sp.S[2], sp.S[3]),
                                       pick4(p, sp.cps[0], sp.cps[1], sp.cps[2], sp.cps[3]), blk);
    });
}

// C[m, n] = fp16(scale[n] * sum over slices q = 0 .. S-1, in that order, of
// part[q][m][n]), S <= 8. Four outputs per thread when N % 4 == 0 (16-byte
// loads of the partial sums and scales, one 8-byte store), else one. Every
// slice is loaded before the first addition (slices past S reload slice 0),
// so the loads overlap: 1.3-1.5 us faster than a loop of dependent loads
// with 8 slices.
// The residual add after a product (ng_gemm_int8_add): out = fp16(C + res) on
// the rounded C, as cuda_add computes it. out may be C or res itself (each
// element is read and written by one thread, out last).
struct ResEpi {
    uint16_t* out;
    const uint16_t* res;
};

// Outputs i .. i + 3 (N % 4 == 0) and output t of the reduction, rounded.
__device__ __forceinline__ u32x2 reduce_slices4(const float* __restrict__ part, const float* __restrict__ scale,
                                                size_t mn, int N, int S, size_t i) {
    f32x4 pv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
        pv[q] = *reinterpret_cast<const f32x4*>(part + static_cast<size_t>(q < S ? q : 0) * mn + i);
    f32x4 v = pv[0];
#pragma unroll
    for (int q = 1; q < 8; ++q)
        if (q < S) v += pv[q];
    const f32x4 sc = *reinterpret_cast<const f32x4*>(scale + i % N);
    return u32x2{pack2<f16>(v[0] * sc[0], v[1] * sc[1]), pack2<f16>(v[2] * sc[2], v[3] * sc[3])};
}

__device__ __forceinline__ uint16_t reduce_slices1(const float* __restrict__ part, const float* __restrict__ scale,
                                                   size_t mn, int N, int S, size_t t) {
    float pv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) pv[q] = part[static_cast<size_t>(q < S ? q : 0) * mn + t];
    float v = pv[0];
#pragma unroll
    for (int q = 1; q < 8; ++q)
        if (q < S) v += pv[q];
    return from_f32<f16>(v * scale[t % N]);
}

template <bool VEC4, bool RES = false>
__device__ __forceinline__ void split_reduce_block(uint16_t* c, const float* __restrict__ part,
                                                   const float* __restrict__ scale, int M, int N, int S, int blk,
                                                   const ResEpi& ep = ResEpi{}) {
    const size_t mn = static_cast<size_t>(M) * N;
    const size_t t = static_cast<size_t>(blk) * 256 + threadIdx.x;
    if (VEC4) {
        const size_t i = 4 * t;
        if (i >= mn) return;
        const u32x2 out = reduce_slices4(part, scale, mn, N, S, i);
        if (RES) {
            const u32x2 rv = *reinterpret_cast<const u32x2*>(ep.res + i);
            *reinterpret_cast<u32x2*>(c + i) = out;
            u32x2 sum;
#pragma unroll
            for (int h = 0; h < 2; ++h)
                sum[h] = pack2<f16>(el_add<f16, 0>(out[h], rv[h]), el_add<f16, 1>(out[h], rv[h]));
            *reinterpret_cast<u32x2*>(ep.out + i) = sum;
        } else {
            *reinterpret_cast<u32x2*>(c + i) = out;
        }
    } else {
        if (t >= mn) return;
        const uint16_t cv = reduce_slices1(part, scale, mn, N, S, t);
        if (RES) {
            const float sum = to_f32<f16>(cv) + to_f32<f16>(ep.res[t]);
            c[t] = cv;
            ep.out[t] = from_f32<f16>(sum);
        } else {
            c[t] = cv;
        }
    }
}

template <bool VEC4, bool RES = false>
__global__ __launch_bounds__(256) void split_reduce_kernel(uint16_t* c, const float* __restrict__ part,
                                                           const float* __restrict__ scale, int M, int N, int S,
                                                           ResEpi ep = ResEpi{}) {
    split_reduce_block<VEC4, RES>(c, part, scale, M, N, S, blockIdx.x, ep);
}

// gate/up with several K slices and SwiGLU (ng_gemm_int8_silu_mul): each
// thread reduces its outputs of both products as split_reduce_block does,
// stores gate and up, then out = fp16(silu(gate) * up) (out may be gate or
// up itself: each element is written by one thread, out last).
template <bool VEC4>
__global__ __launch_bounds__(256) void split_reduce_swiglu_kernel(SwigluArgs sa, const float* __restrict__ pg,
                                                                  const float* __restrict__ pu, int M, int N,
                                                                  int S) {
    const size_t mn = static_cast<size_t>(M) * N;
    const size_t t = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (VEC4) {
        const size_t i = 4 * t;
        if (i >= mn) return;
        const u32x2 g = reduce_slices4(pg, sa.sg, mn, N, S, i);
        const u32x2 u = reduce_slices4(pu, sa.su, mn, N, S, i);
        u32x2 o;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            o[h] = pack2<f16>(swiglu_f32(el_get<f16, 0>(g[h]), el_get<f16, 0>(u[h])),
                              swiglu_f32(el_get<f16, 1>(g[h]), el_get<f16, 1>(u[h])));
        *reinterpret_cast<u32x2*>(sa.gate + i) = g;
        *reinterpret_cast<u32x2*>(sa.up + i) = u;
        *reinterpret_cast<u32x2*>(sa.out + i) = o;
    } else {
        if (t >= mn) return;
        const uint16_t g = reduce_slices1(pg, sa.sg, mn, N, S, t);
        const uint16_t u = reduce_slices1(pu, sa.su, mn, N, S, t);
        sa.gate[t] = g;
        sa.up[t] = u;
        sa.out[t] = from_f32<f16>(swiglu_f32(to_f32<f16>(g), to_f32<f16>(u)));
    }
}

// The reductions of the products of gemm_i8w_split_shared_kernel in one
// launch (blocks partitioned by product as in SharedSet).
template <bool VEC4>
__global__ __launch_bounds__(256) void split_reduce_shared_kernel(SharedSet s, SplitSet sp, int M) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t*, const float* scale, int n, int blk, int p) {
        split_reduce_block<VEC4>(c, pick4(p, sp.part[0], sp.part[1], sp.part[2], sp.part[3]), scale, M, n,
                                 pick4(p, sp.S[0], sp.S[1], sp.S[2], sp.S[3]), blk);
    });
}


// ---- prefill variant (M > 128) ----------------------------------------------
// Many rows of A: the product is bound by the matrix cores (2 M flop per
// weight byte), so a block computes a BM x BN tile of C with WM x WN waves over
// steps of 64 k, and everything else has to hide under the MFMAs:
//   * A (fp16) and the codes of B go from memory straight into LDS
//     (buffer_load ... lds, 16 bytes per lane), NST steps deep: no registers,
//     no conversion and no LDS store on the way in. A step is waited for two or
//     more steps after its loads were issued;
//   * B stays int8 in LDS (half the LDS bytes of fp16) and is converted to
//     exact fp16 integers on its way from LDS into the MFMAs, the next column
//     of 32 rows of B under the MFMAs of the current one; each code is
//     converted by the WM waves that read it;
//   * v_mfma_f32_32x32x16_f16 with the weights as first operand: a lane then
//     holds 4 consecutive n of one row of C. Lane l supplies row l % 32 of each
//     operand; MFMA (P, j) of a step (P, j in {0, 1}) takes k = 32 P + 16 (l /
//     32) + 8 j .. + 7, so that one 16-byte read of codes feeds two MFMAs;
//   * the fragments of the next 16 k are read while the current ones multiply,
//     across steps too: the one barrier of a step stands before its last
//     quarter, whose fragments are already in registers;
//   * LDS rows of A are 128 bytes, 16-byte piece q of row r at q xor ((r / 2)
//     mod 8); rows of B are 64 bytes, piece q at q xor ((r / 4) mod 4). The lanes
//     that a 16-byte read serves together (measured: 0-3, 12-15, 20-27 and
//     4-11, 16-19, 28-31 of each half wave) then touch all 64 banks once;
//   * rows past M or N repeat the last one and are not stored; k past K (K % 64
//     != 0) repeat k below K and are zeroed in both operands in a last step of
//     its own (an inf times a zero code would give NaN);
//   * the tile is stored through LDS in whole 16-byte pieces of rows of C;
//   * tiles are handed out XCD by XCD: block b takes tile (b mod 8) * (tiles /
//     8) + b / 8, grouped kPfGroupM rows of tiles at a time, so that the tiles
//     of one XCD (and of its L2) share rows of A and of B;
//   * with S > 1 the K steps are split into S slices (slice-major over the
//     tiles); each block stores its fp32 sums in `part` [S][M][N] and the
//     reduction adds the slices in slice order.
// Every output is the sum over k in one order whatever the tile shape, so only
// S (a function of M, N and K alone) shows in the bits. Measured on MI355X, in
// turn with the kernel this replaces (A and B through registers, B stored to LDS
// as fp16, two LDS buffers): a whole layer at 333 tokens of Llama-2-7B 220
// against 344 us, at 1024 tokens of Mistral-7B 468 against 574. In that last
// layer's kernel trace (weights cold): q/k/v 62 us, o 44, gate/up with SwiGLU 222
// (1.08 PFLOP/s), down 113 and 18 for its reduction. What bounds it on
// 256 x 256 tiles (1024 x 28672, K = 4096: 206 us, 1.17 PFLOP/s): the power limit
// with the matrix cores 64% busy (1.75 GHz). The MFMAs alone (no loads, no LDS
// reads) took 130 us, without the LDS reads 164, without the loads into LDS 182,
// without converting codes 193. Four waves of 128 x 128 on the same tile: 220.
constexpr int kPfBK = 64;
constexpr int kPfGroupM = 8;

typedef float f32x16 __attribute__((ext_vector_type(16)));

// 16 bytes per lane from (voff + soff) of a buffer to LDS at lds + 16 lane.
// Written out because the compiler waits for all outstanding loads (vmcnt(0))
// before any LDS read that follows its builtin; the kernel waits by count. The
// load has no register result. s_nop: the wait state between a write of m0 and a
// load that reads it. m0 is declared as written, so that the compiler sets it
// again for uses of its own; it warns that it keeps nothing in a reserved register
// across the statement, which is what is meant.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff),
                 "s"(r), "s"(soff)
                 : "memory", "m0");
}

// Likewise, non-temporal.
__device__ __forceinline__ void load_lds16_nt(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(lds), "v"(voff),
                 "s"(r), "s"(soff)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// At most N of this wave's vector memory operations still outstanding.
template <int N>
__device__ __forceinline__ void wait_vmem() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// This wave's LDS reads are in its registers, then the block's barrier; no
// memory access moves across it.
__device__ __forceinline__ void lds_read_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 8 codes (two dwords) as exact fp16 integers.
__device__ __forceinline__ f16x8 codes8_to_operand(uint32_t lo, uint32_t hi) {
    const u32x4 x = {codes_to_f16x2<0x04010400u>(lo), codes_to_f16x2<0x04030402u>(lo),
                     codes_to_f16x2<0x04010400u>(hi), codes_to_f16x2<0x04030402u>(hi)};
    return __builtin_bit_cast(f16x8, x);
}

// What follows the product of a launch with one K slice: nothing, the
// residual add (out, res), or SwiGLU (SW: the tile's columns 0 .. BN / 2 - 1
// are gate's, the others up's).
struct TileEpi {
    uint16_t* out;        // residual add or SwiGLU; null: none
    const uint16_t* res;  // residual add
};

// Whether rows of C (and of what else the epilogue touches) are whole 16-byte pieces.
template <bool SW>
__device__ __forceinline__ bool out_vec(const uint16_t* c, int N, const TileEpi& ep, const SwigluArgs* sw) {
    const auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return N % 8 == 0 && on16(SW ? sw->gate : c) && (!SW || on16(sw->up)) && (ep.out == nullptr || on16(ep.out)) &&
           (ep.res == nullptr || on16(ep.res));
}

// Elements o .. o + 7 of C (n_ok of them in the row) with what follows: v as
// rounded to fp16 (SW: gate, with up in u). out may be an operand itself: each
// element is read and written by one thread, out last.
template <bool SW>
__device__ __forceinline__ void store_out8(uint16_t* c, size_t o, int n_ok, const u32x4& v, const u32x4& u, bool vec,
                                           const TileEpi& ep, const SwigluArgs* sw) {
    const auto store = [&](uint16_t* p, const u32x4& x) {
        if (vec) {
            st16(p + o, x);
        } else {
            for (int e = 0; e < 8; ++e)
                if (e < n_ok) p[o + e] = lane16(x, e);
        }
    };
    u32x4 y;
    if constexpr (SW) {
#pragma unroll
        for (int h = 0; h < 4; ++h)
            y[h] = pack2<f16>(swiglu_f32(el_get<f16, 0>(v[h]), el_get<f16, 0>(u[h])),
                              swiglu_f32(el_get<f16, 1>(v[h]), el_get<f16, 1>(u[h])));
        store(sw->gate, v);
        store(sw->up, u);
        store(ep.out, y);
    } else if (ep.out == nullptr) {
        store(c, v);
    } else {
        u32x4 x;
        if (vec) {
            x = ld16(ep.res + o);
        } else {
            for (int h = 0; h < 4; ++h)
                x[h] = (2 * h < n_ok ? ep.res[o + 2 * h] : 0u) | ((2 * h + 1 < n_ok ? ep.res[o + 2 * h + 1] : 0u) << 16);
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) y[h] = pack2<f16>(el_add<f16, 0>(v[h], x[h]), el_add<f16, 1>(v[h], x[h]));
        store(c, v);
        store(ep.out, y);
    }
}

// SERIAL: a block takes all K slices of its tile (S = 1; cps: a slice's steps),
// one after the other, and adds each sum to those before it as the reduction
// does: the bits of a launch with a block per slice, without its partial sums.
template <int BM, int BN, int WM, int WN, int NST, bool SW, bool SERIAL = false>
__device__ __forceinline__ void gemm_i8w_tile_block(
    uint16_t* c, const uint16_t* __restrict__ a, const int8_t* __restrict__ b, const float* __restrict__ scale,
    float* __restrict__ part, int M, int N, int K, int tiles_m, int tiles_n, int S, int cps, int blk,
    const TileEpi& ep, const SwigluArgs* sw = nullptr) {
    constexpr int NW = WM * WN;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;   // a wave's 32 x 32 tiles
    constexpr int kAI = BM / 8 / NW, kBI = BN / 16 / NW;  // loads of 1 KiB per wave and step
    constexpr int kABytes = BM * 128, kStage = kABytes + BN * 64;
    constexpr int kLoads = kAI + kBI;
    constexpr int kRow = BN * 2 + 16;  // a row of the tile of C in LDS, padded
    static_assert(TM * WM * 32 == BM && TN * WN * 32 == BN, "tiles must divide among the waves");
    static_assert(kAI * 8 * NW == BM && kBI * 16 * NW == BN, "loads must divide among the waves");
    static_assert(!SW || BN / 2 % 16 == 0, "a load of B lies in gate or in up");
    __shared__ __align__(1024) uint8_t lds[NST * kStage > BM * kRow ? NST * kStage : BM * kRow];
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds));
    constexpr int BNC = SW ? BN / 2 : BN;  // columns of one matrix C in the tile

    const int ntiles = tiles_m * tiles_n;
    int t = blk;
    if ((ntiles * S) % 8 == 0) t = (t % 8) * (ntiles * S / 8) + t / 8;
    const int sl = t / ntiles;
    t -= sl * ntiles;
    const int per_group = kPfGroupM * tiles_n;
    const int grp0 = (t / per_group) * kPfGroupM;
    const int gm = min(kPfGroupM, tiles_m - grp0);
    const int tm = grp0 + (t % per_group) % gm;
    const int tn = (t % per_group) / gm;
    const int m0 = tm * BM, n0 = tn * BNC;

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wm = wave / WN, wn = wave % WN;
    const int grp = lane >> 5;

    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a + static_cast<size_t>(m0) * K), 0,
        static_cast<int>(min(static_cast<long long>(M - m0) * K * 2, 0x7fffffffll)), 0x00020000);
    const auto rsrc_b = [&](const int8_t* p) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<int8_t*>(p + static_cast<size_t>(n0) * K), 0,
            static_cast<int>(min(static_cast<long long>(N - n0) * K, 0x7fffffffll)), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rsb = rsrc_b(SW ? sw->bg : b), rsu = rsrc_b(SW ? sw->bu : b);

    // Load j of a step fills 1 KiB of LDS in lane order: 8 rows of A (lane l:
    // row l / 8, slot l % 8) or 16 rows of B (row l / 4, slot l % 4). The
    // swizzle is in which piece a lane fetches. Rows past M or N repeat the last.
    const auto a_row = [&](int j) { return (wave * kAI + j) * 8 + (lane >> 3); };
    const auto a_piece = [&](int j) { return (lane & 7) ^ ((a_row(j) >> 1) & 7); };
    const auto b_row = [&](int j) { return (wave * kBI + j) * 16 + (lane >> 2); };
    const int b_piece = (lane & 3) ^ ((lane >> 4) & 3);
    uint32_t av[kAI], bv[kBI];
#pragma unroll
    for (int j = 0; j < kAI; ++j) av[j] = static_cast<uint32_t>(min(a_row(j), M - 1 - m0) * K * 2 + 16 * a_piece(j));
#pragma unroll
    for (int j = 0; j < kBI; ++j)
        bv[j] = static_cast<uint32_t>(min(SW ? b_row(j) % BNC : b_row(j), N - 1 - n0) * K + 16 * b_piece);
    const int nk = (K + kPfBK - 1) / kPfBK;
    const int krem = K % kPfBK;  // k of a partial last step (a multiple of 16)
    // Loads j0 .. j1 - 1 (A's, then B's) of a step into stage st.
    const auto load = [&](int step, int st, int j0, int j1) {
        const uint32_t base = lds0 + static_cast<uint32_t>(st * kStage);
        const uint32_t k0 = static_cast<uint32_t>(step * kPfBK);
        // Pieces past K of a partial last step fetch the step's first piece.
        // (Selects: with a branch for whole steps the loop was 4-7% slower.)
        const bool part_step = krem != 0 && step == nk - 1;
#pragma unroll
        for (int j = 0; j < kAI; ++j) {
            if (j < j0 || j >= j1) continue;
            const uint32_t v = part_step && 8 * a_piece(j) >= krem ? av[j] - 16 * a_piece(j) : av[j];
            load_lds16(rsa, base + static_cast<uint32_t>((wave * kAI + j) * 1024), v, 2 * k0);
        }
#pragma unroll
        for (int j = 0; j < kBI; ++j) {
            if (kAI + j < j0 || kAI + j >= j1) continue;
            const uint32_t v = part_step && 16 * b_piece >= krem ? bv[j] - 16 * b_piece : bv[j];
            const bool up = SW && (wave * kBI + j) * 16 >= BNC;
            load_lds16(up ? rsu : rsb, base + static_cast<uint32_t>(kABytes + (wave * kBI + j) * 1024), v, k0);
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    const int ar = wm * TM * 32 + (lane & 31), br = wn * TN * 32 + (lane & 31);
    const uint32_t aoff = static_cast<uint32_t>(ar * 128 + (((2 * grp) ^ ((ar >> 1) & 7)) << 4));
    const uint32_t boff = static_cast<uint32_t>(kABytes + br * 64 + ((grp ^ ((br >> 2) & 3)) << 4));
    // Fragments of A for MFMA (q / 2, q % 2), and codes of B for MFMAs (P, 0) and (P, 1).
    const auto read_a = [&](int st, int q, u32x4 (&f)[TM]) {
        const uint8_t* p = lds + st * kStage + (aoff ^ ((4 * (q >> 1) + (q & 1)) << 4));
#pragma unroll
        for (int i = 0; i < TM; ++i) f[i] = *reinterpret_cast<const u32x4*>(p + i * 32 * 128);
    };
    const auto read_b = [&](int st, int P, u32x4 (&f)[TN]) {
        const uint8_t* p = lds + st * kStage + (boff ^ (P << 5));
#pragma unroll
        for (int j = 0; j < TN; ++j) f[j] = *reinterpret_cast<const u32x4*>(p + j * 32 * 64);
    };
    // The MFMAs of column j with its weights w; the next column's codes are
    // converted into w under them.
    f16x8 w;
    const auto column = [&](const u32x4 (&f)[TM], int j, uint32_t next_lo, uint32_t next_hi) {
        const f16x8 next = codes8_to_operand(next_lo, next_hi);
#pragma unroll
        for (int i = 0; i < TM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, __builtin_bit_cast(f16x8, f[i]), acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (10 + TM - 1) / TM, 0);
        }
        w = next;
    };
    // Columns j0 .. j1 - 1 of MFMA (., J) from the codes cb; after the last
    // column comes column 0 of MFMA (., NJ) from ncb.
    const auto columns = [&](const u32x4 (&f)[TM], const u32x4 (&cb)[TN], int J, const u32x4 (&ncb)[TN], int NJ,
                             int j0, int j1) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if (j < j0 || j >= j1) continue;
            const u32x4 nc = j + 1 < TN ? cb[j + 1 < TN ? j + 1 : 0] : ncb[0];
            const int o = 2 * (j + 1 < TN ? J : NJ);
            column(f, j, nc[o], nc[o + 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    const int c0 = SERIAL ? 0 : sl * cps, c1 = SERIAL ? nk : min(nk, c0 + cps);
    const int n = c1 - c0;                            // steps of this block
    const int full = c1 == nk && krem ? n - 1 : n;    // of them whole ones
    u32x4 fa[2][TM], cb[2][TN];
#pragma unroll
    for (int s = 0; s < NST; ++s)
        if (s < n) load(c0 + s, s, 0, kLoads);
    if (n >= NST) wait_vmem<(NST - 1) * kLoads>();
    else wait_vmem<0>();
    lds_read_barrier();
    read_a(0, 0, fa[0]);
    read_b(0, 0, cb[0]);
    w = codes8_to_operand(cb[0][0][0], cb[0][0][1]);
    int st = 0;
    // Step c0 + i's last quarter and step c0 + i + 1's first two issue the
    // loads of step c0 + i + NST, a third each, between two columns of MFMAs:
    // issued in one go behind the barrier they held the MFMAs up (256 x 256 at
    // 1024 x 28672, K = 4096: 206 against 215 us; one by one between all
    // columns: 210).
    constexpr int kThird = (kLoads + 2) / 3, kEarly = TN > 1 ? 1 : 0;
    // STEADY: steps whose loads all exist, without a branch in the body.
    const auto step = [&](int i, auto steady) {
        constexpr bool STEADY = decltype(steady)::value;
        const int nx = st + 1 == NST ? 0 : st + 1, prev = st == 0 ? NST - 1 : st - 1;
        const bool more = STEADY || (i > 0 && i - 1 + NST < n);  // loads left of step i - 1 + NST
        read_a(st, 1, fa[1]);
        read_b(st, 1, cb[1]);
        columns(fa[0], cb[0], 0, cb[0], 1, 0, 1);
        if (more) load(c0 + i - 1 + NST, prev, kThird, 2 * kThird);
        columns(fa[0], cb[0], 0, cb[0], 1, 1, TN);
        read_a(st, 2, fa[0]);
        columns(fa[1], cb[0], 1, cb[1], 0, 0, 1);
        if (more) load(c0 + i - 1 + NST, prev, 2 * kThird, kLoads);
        columns(fa[1], cb[0], 1, cb[1], 0, 1, TN);
        read_a(st, 3, fa[1]);
        columns(fa[0], cb[1], 0, cb[1], 1, 0, TN);
        // Step i + 1 is in LDS once every wave has waited for its own loads of
        // it; stage st is free once every wave has read its last fragments.
        if (STEADY || i + NST <= n) wait_vmem<(NST - 2) * kLoads>();
        else wait_vmem<0>();
        lds_read_barrier();
        columns(fa[1], cb[1], 1, cb[0], 0, 0, kEarly);
        read_b(nx, 0, cb[0]);
        read_a(nx, 0, fa[0]);
        if (STEADY || i + NST < n) load(c0 + i + NST, st, 0, kThird);
        columns(fa[1], cb[1], 1, cb[0], 0, kEarly, TN);
        st = nx;
    };
    int i0 = 0;
    if (full > 0) step(i0++, std::false_type{});
    [[maybe_unused]] f32x16 sum[SERIAL ? TM : 1][SERIAL ? TN : 1] = {};  // of the slices before
    if constexpr (SERIAL) {
        for (int end = cps; end < n; end += cps) {
            const int stop = min(end, full);
            for (; i0 + NST < n && i0 < stop; ++i0) step(i0, std::true_type{});
            for (; i0 < stop; ++i0) step(i0, std::false_type{});
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    sum[i][j] += acc[i][j];
                    acc[i][j] = f32x16{};
                }
        }
    }
    for (; i0 + NST < n && i0 < full; ++i0) step(i0, std::true_type{});
    for (; i0 < full; ++i0) step(i0, std::false_type{});
    if (full < n) {
        // The partial last step: k past K zeroed in both operands.
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool kin = 32 * (q >> 1) + 16 * grp + 8 * (q & 1) < krem;
            read_a(st, q, fa[0]);
            read_b(st, q >> 1, cb[0]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
                if (!kin) fa[0][i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                w = codes8_to_operand(cb[0][j][2 * (q & 1)], cb[0][j][2 * (q & 1) + 1]);
                if (!kin) w = __builtin_bit_cast(f16x8, u32x4{0u, 0u, 0u, 0u});
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, __builtin_bit_cast(f16x8, fa[0][i]),
                                                                       acc[i][j], 0, 0, 0);
            }
        }
    }

    if constexpr (SERIAL) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j] + acc[i][j];
    }
    // acc[i][j][4 q + e] is C[m0 + wm TM 32 + 32 i + l % 32][n0 + wn TN 32 + 32 j + 8 q + 4 (l / 32) + e].
    if (S > 1) {
        float* mine = part + static_cast<size_t>(sl) * M * N;
        const bool vec = N % 4 == 0;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m0 + wm * TM * 32 + 32 * i + (lane & 31);
            if (m >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int nn = n0 + wn * TN * 32 + 32 * j + 8 * q + 4 * grp;
                    const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    float* o = mine + static_cast<size_t>(m) * N + nn;
                    if (vec) {
                        if (nn < N) *reinterpret_cast<f32x4*>(o) = v;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (nn + e < N) o[e] = v[e];
                    }
                }
        }
        return;
    }
    lds_read_barrier();  // the stages are free
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int nl = wn * TN * 32 + 32 * j + 8 * q + 4 * grp;
            const float* sc = SW ? (nl < BNC ? sw->sg : sw->su) : scale;
            float s[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = sc[min(n0 + (SW ? nl % BNC : nl) + e, N - 1)];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                *reinterpret_cast<u32x2*>(lds + (wm * TM * 32 + 32 * i + (lane & 31)) * kRow + 2 * nl) =
                    u32x2{pack2<f16>(acc[i][j][4 * q] * s[0], acc[i][j][4 * q + 1] * s[1]),
                          pack2<f16>(acc[i][j][4 * q + 2] * s[2], acc[i][j][4 * q + 3] * s[3])};
        }
    __syncthreads();
    constexpr int kPieces = BNC / 8;  // 16-byte pieces of a row of one matrix C
    const bool vec = out_vec<SW>(c, N, ep, sw);
    for (int p = tid; p < BM * kPieces; p += NW * kWave) {
        const int r = p / kPieces, q = p % kPieces;
        const int m = m0 + r, nn = n0 + 8 * q;
        if (m >= M || nn >= N) continue;
        const uint8_t* row = lds + r * kRow + 16 * q;
        const u32x4 v = *reinterpret_cast<const u32x4*>(row);
        const u32x4 u = *reinterpret_cast<const u32x4*>(row + (SW ? 2 * BNC : 0));
        store_out8<SW>(c, static_cast<size_t>(m) * N + nn, N - nn, v, u, vec, ep, sw);
    }
}

// One or more products that share A (ng_gemm_int8_shared_a): each keeps its
// own tiles, K slices and partial-sum region. In SplitSet, `tiles` holds the
// product's tiles along N and `TT` its tiles along M. ep follows the product of
// a launch of one with one K slice (out may be c or res itself: each element
// is read and written by one thread, out last).
template <int BM, int BN, int WM, int WN, int NST, bool SERIAL>
__global__ __launch_bounds__(WM * WN * kWave, 1) void gemm_i8w_tile_kernel(SharedSet s, SplitSet sp,
                                                                           const uint16_t* __restrict__ a, int M,
                                                                           int K, TileEpi ep) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int p) {
        gemm_i8w_tile_block<BM, BN, WM, WN, NST, false, SERIAL>(
            c, a, b, scale, pick4(p, sp.part[0], sp.part[1], sp.part[2], sp.part[3]), M, n, K,
            pick4(p, sp.TT[0], sp.TT[1], sp.TT[2], sp.TT[3]),
            pick4(p, sp.tiles[0], sp.tiles[1], sp.tiles[2], sp.tiles[3]),
            pick4(p, sp.S[0], sp.S[1], sp.S[2], sp.S[3]), pick4(p, sp.cps[0], sp.cps[1], sp.cps[2], sp.cps[3]), blk,
            ep);
    });
}

// gate, up and SwiGLU (ng_gemm_int8_silu_mul) with one K slice: a block's tile
// is BN / 2 columns of gate and the same columns of up. Each output's sum over k
// is its own launch's, so gate and up keep their bits.
template <int BM, int BN, int WM, int WN, int NST>
__global__ __launch_bounds__(WM * WN * kWave, 1) void gemm_i8w_tile_swiglu_kernel(SwigluArgs sa,
                                                                                  const uint16_t* __restrict__ a,
                                                                                  int M, int N, int K, int tiles_m,
                                                                                  int tiles_n, int cps) {
    const TileEpi ep{sa.out, nullptr};
    gemm_i8w_tile_block<BM, BN, WM, WN, NST, true>(nullptr, a, nullptr, nullptr, nullptr, M, N, K, tiles_m, tiles_n, 1,
                                                   cps, blockIdx.x, ep, &sa);
}

// ---- 33 to 128 rows of A ------------------------------------------------------
// Here the weights still have to be read once, but a block that streams its
// rows of B also reads its K slice of A from L2, and both have to be in flight
// ahead of the matrix cores. One tile of all rows of A x BN rows of B per block:
//   * stages of WK x 64 k, NST of them, go straight into LDS as in the prefill
//     kernel, NST - 1 steps ahead: 80 to 128 KiB in flight per CU (one block, or
//     two of the small tiles) and one barrier per step (the kernel this replaces
//     staged both through registers one step ahead);
//   * the WK groups of WN waves multiply different 64 k of a stage, each wave
//     all rows of A by 32 rows of B, so a fragment of A feeds as many MFMAs as
//     the tile is wide and B is converted once; the groups' sums meet in LDS at
//     the end, in group order;
//   * B is loaded, and lies in LDS, in 128-byte pieces of rows (128 k, two
//     groups): whole lines; 16-byte piece q of row r at q xor ((r / 2) mod 8), as
//     for A;
//   * S slices of K (a function of M, N and K) where one slice leaves most CUs
//     idle, added in slice order by the reduction; with one slice the epilogues
//     of the prefill kernel. Gate and up with SwiGLU load B non-temporally (at 64
//     rows 29.2 against 31.2 us); with K slices that was 2-8% slower.
// Measured on MI355X against that kernel, reductions included: q/k/v of
// Mistral-7B at 64 rows 16.0 against 22.7 us, o 11.2 against 12.0, gate/up with
// SwiGLU 32.4 against 39.0; at 128 rows 21.7 against 29.7, 14.1 against 17.1, 46.3
// against 67.3, down 31.2 against 32.1; gate/up of TinyLlama at 64 rows 11.2
// against 18.1; k/v alone (N = 1024) 7.2 against 7.5, three products of 4096 rows
// of B at 33 and 64 rows 18.0 against 20.6 and 21.6 against 25.9. Up to 6% slower at 33 -
// 64 rows: one wide product of K >= 5120 whose blocks of 64 rows of B take most of
// the GPU's CUs (13824 x 5120 at 64 rows 25.9 against 24.7), since a CU then runs 4
// waves; two of them, or one with SwiGLU, are faster.
// Bound at 64 rows: gate/up move 117 MB of weights in 32 us (3.7 TB/s) and A 224
// times from L2 (as much again); 8 or 16 us calls are launch, first loads and the
// reduction.
// SERIAL: a block takes both K slices of its tile (S = 1; cps: the first one's
// steps), one after the other, and adds the second sum to the first as the
// reduction does: the bits of a launch with a block per slice, without its partial sums.
template <int BM, int BN, int WN, int WK, int NST, bool SW, bool SERIAL = false>
__device__ __forceinline__ void gemm_i8w_ring_block(uint16_t* c, const uint16_t* __restrict__ a,
                                                    const int8_t* __restrict__ b, const float* __restrict__ scale,
                                                    float* __restrict__ part, int Mall, int N, int K, int S,
                                                    int tiles, int cps, int TT, int blk, const TileEpi& ep,
                                                    const SwigluArgs* sw = nullptr) {
    constexpr int NW = WN * WK;
    constexpr int TM = BM / 32;
    constexpr int kA64 = BM * 128, kB128 = BN * 128;  // bytes of A of 64 k, of B of 128 k
    constexpr int kABytes = WK * kA64, kStage = kABytes + WK / 2 * kB128;
    constexpr int kAI = kABytes / 1024 / NW, kBI = WK / 2 * kB128 / 1024 / NW, kLoads = kAI + kBI;
    constexpr int kRow = BN * 4 + 16;  // a row of a group's fp32 sums in LDS, padded
    constexpr int kSums = WK * BM * kRow;
    constexpr int BNC = SW ? BN / 2 : BN;
    static_assert(BN == 32 * WN && WK % 2 == 0 && BM % 32 == 0, "tile shape");
    static_assert(kAI * NW * 1024 == kABytes && kBI * NW * 2048 == WK * kB128, "loads must divide among the waves");
    __shared__ __align__(1024) uint8_t lds[NST * kStage > kSums ? NST * kStage : kSums];
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds));
    // With TT > 1 row tiles, the TT blocks of a unit (a tile and slice) sit on
    // one XCD (ids 8 apart), so that they read its rows of B from one L2.
    int unit = blk, m0 = 0;
    if (TT > 1) {
        const int i = blk / 8;
        m0 = BM * (i % TT);
        unit = i / TT * 8 + blk % 8;
        if (unit >= tiles * S) return;
    }
    const int M = Mall - m0;  // rows from this tile's first on
    const int sl = unit % S, n0 = unit / S * BNC;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int kg = wave / WN, wn = wave % WN;
    const int grp = lane >> 5;

    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a + static_cast<size_t>(m0) * K), 0, static_cast<int>(min(static_cast<long long>(M) * K * 2, 0x7fffffffll)), 0x00020000);
    const auto rsrc_b = [&](const int8_t* p) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<int8_t*>(p + static_cast<size_t>(n0) * K), 0,
            static_cast<int>(min(static_cast<long long>(N - n0) * K, 0x7fffffffll)), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rsb = rsrc_b(SW ? sw->bg : b), rsu = rsrc_b(SW ? sw->bu : b);
    // Load j of a step: 8 rows of A of one group's 64 k, or 8 rows of B of two
    // groups' 128 k; lane l row l / 8, slot l % 8. Rows past M or N repeat the last.
    const auto a_group = [&](int j) { return (wave * kAI + j) / (BM / 8); };
    const auto b_pair = [&](int j) { return (wave * kBI + j) / (BN / 8); };
    const auto a_row = [&](int j) { return (wave * kAI + j) % (BM / 8) * 8 + (lane >> 3); };
    const auto b_row = [&](int j) { return (wave * kBI + j) % (BN / 8) * 8 + (lane >> 3); };
    const auto piece = [&](int r) { return (lane & 7) ^ ((r >> 1) & 7); };
    uint32_t av[kAI], bv[kBI];
#pragma unroll
    for (int j = 0; j < kAI; ++j)
        av[j] = static_cast<uint32_t>(min(a_row(j), M - 1) * K * 2 + 128 * a_group(j) + 16 * piece(a_row(j)));
#pragma unroll
    for (int j = 0; j < kBI; ++j)
        bv[j] = static_cast<uint32_t>(min(SW ? b_row(j) % BNC : b_row(j), N - 1 - n0) * K + 128 * b_pair(j) +
                                      16 * piece(b_row(j)));
    const int nk = (K + 64 * WK - 1) / (64 * WK);
    const int kparts = K / 64 - (nk - 1) * WK;  // 64-k parts of the last step (K % 64 == 0)
    const auto load = [&](int step, int st) {
        const uint32_t base = lds0 + static_cast<uint32_t>(st * kStage);
        const uint32_t k0 = static_cast<uint32_t>(step * 64 * WK);
        // Parts past K of the last step fetch the step's first part.
        const bool cut = kparts < WK && step == nk - 1;
#pragma unroll
        for (int j = 0; j < kBI; ++j) {
            const int in_pair = piece(b_row(j)) >> 2;
            const uint32_t v =
                cut && 2 * b_pair(j) + in_pair >= kparts ? bv[j] - 128 * b_pair(j) - 64 * in_pair : bv[j];
            const bool up = SW && (wave * kBI + j) % (BN / 8) * 8 >= BNC;
            const uint32_t to = base + static_cast<uint32_t>(kABytes + (wave * kBI + j) * 1024);
            if (SW) load_lds16_nt(up ? rsu : rsb, to, v, k0);
            else load_lds16(rsb, to, v, k0);
        }
#pragma unroll
        for (int j = 0; j < kAI; ++j) {
            const uint32_t v = cut && a_group(j) >= kparts ? av[j] - 128 * a_group(j) : av[j];
            load_lds16(rsa, base + static_cast<uint32_t>((wave * kAI + j) * 1024), v, 2 * k0);
        }
    };

    f32x16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    const int ar = lane & 31, br = wn * 32 + (lane & 31);
    const uint32_t aoff = static_cast<uint32_t>(kg * kA64 + ar * 128 + (((2 * grp) ^ ((ar >> 1) & 7)) << 4));
    const uint32_t boff = static_cast<uint32_t>(kABytes + kg / 2 * kB128 + br * 128 +
                                                (((4 * (kg & 1) + grp) ^ ((br >> 1) & 7)) << 4));

    const int c0 = SERIAL ? 0 : sl * cps, c1 = SERIAL ? nk : min(nk, c0 + cps), n = c1 - c0;
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
        if (s < n) load(c0 + s, s);
    // MFMA (P, j) of the group's 64 k as in the prefill kernel: fragments of A
    // for q = 2 P + j, codes of B for both j.
    u32x4 fa[4][TM], cb[2];
    const auto read = [&](int st) {
        const uint8_t* base = lds + st * kStage;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q % 2 == 0) cb[q / 2] = *reinterpret_cast<const u32x4*>(base + (boff ^ (q << 4)));
            const uint8_t* p = base + (aoff ^ ((4 * (q >> 1) + (q & 1)) << 4));
#pragma unroll
            for (int m = 0; m < TM; ++m) fa[q][m] = *reinterpret_cast<const u32x4*>(p + m * 32 * 128);
        }
    };
    const auto multiply = [&]() {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f16x8 w = codes8_to_operand(cb[q >> 1][2 * (q & 1)], cb[q >> 1][2 * (q & 1) + 1]);
#pragma unroll
            for (int m = 0; m < TM; ++m)
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, __builtin_bit_cast(f16x8, fa[q][m]), acc[m], 0, 0, 0);
        }
    };
    // Whole steps; a last one that not every group has a part of follows the
    // loop (a branch around the loop's MFMAs cost gate at 64 rows 3 of 23 us).
    const int full = c1 == nk && kparts < WK ? n - 1 : n;
    int st = 0;
    const auto step = [&](int i, auto steady) {
        constexpr bool STEADY = decltype(steady)::value;
        // This wave's loads of step i have landed; after the barrier every
        // wave's have, and every wave has read step i - 1, whose stage the
        // loads of step i + NST - 1 then take.
        if (STEADY || i + NST - 1 <= n) wait_vmem<(NST - 2) * kLoads>();
        else wait_vmem<0>();
        lds_read_barrier();
        read(st);
        __builtin_amdgcn_sched_barrier(0);
        if (STEADY || i + NST - 1 < n) load(c0 + i + NST - 1, st == 0 ? NST - 1 : st - 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        __builtin_amdgcn_sched_barrier(0);
        st = st + 1 == NST ? 0 : st + 1;
    };
    int i0 = 0;
    [[maybe_unused]] f32x16 first[SERIAL ? TM : 1];  // the first slice's sums
    const bool two = SERIAL && cps < n;
    if constexpr (SERIAL) {
        if (two) {
            for (; i0 + NST - 1 < n && i0 < cps; ++i0) step(i0, std::true_type{});
            for (; i0 < cps; ++i0) step(i0, std::false_type{});
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            first[i] = acc[i];
            acc[i] = f32x16{};
        }
    }
    for (; i0 + NST - 1 < n && i0 < full; ++i0) step(i0, std::true_type{});
    for (; i0 < full; ++i0) step(i0, std::false_type{});
    if (full < n) {
        wait_vmem<0>();
        lds_read_barrier();
        if (kg < kparts) {
            read(st);
            multiply();
        }
    }
    lds_read_barrier();  // the stages are free (their last loads were waited for)

    // acc[i][4 q + e] is this group's sum for row 32 i + l % 32, column 32 wn + 8 q + 4 (l / 32) + e.
    if constexpr (!SERIAL) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4*>(lds + (kg * BM + 32 * i + (lane & 31)) * kRow + 4 * (32 * wn + 8 * q + 4 * grp)) =
                    f32x4{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
        __syncthreads();
    }
    // Eight columns from `col` of row r, groups added in order.
    const auto sums8 = [&](int r, int col, float (&v)[8]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 x = *reinterpret_cast<const f32x4*>(lds + r * kRow + 4 * col + 16 * h);
#pragma unroll
            for (int g = 1; g < WK; ++g) x += *reinterpret_cast<const f32x4*>(lds + (g * BM + r) * kRow + 4 * col + 16 * h);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * h + e] = x[e];
        }
    };
    constexpr int kPieces = BNC / 8;
    [[maybe_unused]] float head[8];  // of this thread's piece: the first slice
    if constexpr (SERIAL) {
        static_assert(BM * kPieces == NW * kWave, "one piece per thread");
        const auto put = [&](const f32x16 (&x)[TM]) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4*>(lds + (kg * BM + 32 * i + (lane & 31)) * kRow +
                                              4 * (32 * wn + 8 * q + 4 * grp)) =
                        f32x4{x[i][4 * q], x[i][4 * q + 1], x[i][4 * q + 2], x[i][4 * q + 3]};
            __syncthreads();
        };
        if (two) {
            put(first);
            sums8(tid / kPieces, 8 * (tid % kPieces), head);
            __syncthreads();
        }
        put(acc);
    }
    const bool vec = S > 1 ? N % 4 == 0 : out_vec<SW>(c, N, ep, sw);
    for (int p = tid; p < BM * kPieces; p += NW * kWave) {
        const int r = p / kPieces, q = p % kPieces, nn = n0 + 8 * q;
        if (r >= M || nn >= N) continue;
        float v[8];
        sums8(r, 8 * q, v);
        if constexpr (SERIAL) {
            if (two) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = head[e] + v[e];
            }
        }
        if (S > 1) {
            float* o = part + (static_cast<size_t>(sl) * Mall + m0 + r) * N + nn;
            if (vec) {
                *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
                if (nn + 4 < N) *reinterpret_cast<f32x4*>(o + 4) = f32x4{v[4], v[5], v[6], v[7]};
            } else {
                for (int e = 0; e < 8; ++e)
                    if (nn + e < N) o[e] = v[e];
            }
            continue;
        }
        const auto scaled = [&](const float* sc) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= sc[min(nn + e, N - 1)];
            return pack8<f16>(v);
        };
        const u32x4 x = scaled(SW ? sw->sg : scale);
        u32x4 u = x;
        if constexpr (SW) {
            sums8(r, BNC + 8 * q, v);
            u = scaled(sw->su);
        }
        store_out8<SW>(c, static_cast<size_t>(m0 + r) * N + nn, N - nn, x, u, vec, ep, sw);
    }
}

// A product alone: plain arguments, which are in registers when its waves
// start (o at 64 rows 9.6 us without its reduction, 10.0 through the argument sets
// of the shared form).
template <int BM, int BN, int WN, int WK, int NST>
__global__ __launch_bounds__(WN * WK * kWave, 1) void gemm_i8w_ring_kernel(
    uint16_t* c, const uint16_t* __restrict__ a, const int8_t* __restrict__ b, const float* __restrict__ scale,
    float* __restrict__ part, int M, int N, int K, int S, int tiles, int cps, int TT, TileEpi ep) {
    gemm_i8w_ring_block<BM, BN, WN, WK, NST, false>(c, a, b, scale, part, M, N, K, S, tiles, cps, TT, blockIdx.x, ep);
}

// Products that share A, as gemm_i8w_tile_kernel.
template <int BM, int BN, int WN, int WK, int NST, bool SERIAL>
__global__ __launch_bounds__(WN * WK * kWave, 1) void gemm_i8w_ring_shared_kernel(SharedSet s, SplitSet sp,
                                                                                  const uint16_t* __restrict__ a,
                                                                                  int M, int K) {
    shared_dispatch(s, [&](uint16_t* c, const int8_t* b, const float* scale, int n, int blk, int p) {
        gemm_i8w_ring_block<BM, BN, WN, WK, NST, false, SERIAL>(
            c, a, b, scale, pick4(p, sp.part[0], sp.part[1], sp.part[2], sp.part[3]), M, n, K,
            pick4(p, sp.S[0], sp.S[1], sp.S[2], sp.S[3]), pick4(p, sp.tiles[0], sp.tiles[1], sp.tiles[2], sp.tiles[3]),
            pick4(p, sp.cps[0], sp.cps[1], sp.cps[2], sp.cps[3]), pick4(p, sp.TT[0], sp.TT[1], sp.TT[2], sp.TT[3]),
            blk, TileEpi{nullptr, nullptr});
    });
}

// gate, up and SwiGLU with one K slice, as gemm_i8w_tile_swiglu_kernel.
template <int BM, int BN, int WN, int WK, int NST>
__global__ __launch_bounds__(WN * WK * kWave, 1) void gemm_i8w_ring_swiglu_kernel(SwigluArgs sa,
                                                                                  const uint16_t* __restrict__ a,
                                                                                  int M, int N, int K, int tiles,
                                                                                  int cps, int TT) {
    const TileEpi ep{sa.out, nullptr};
    gemm_i8w_ring_block<BM, BN, WN, WK, NST, true>(nullptr, a, nullptr, nullptr, nullptr, M, N, K, 1, tiles, cps, TT,
                                                   blockIdx.x, ep, &sa);
}

// ---- hipBLASLt path ----------------------------------------------------------
constexpr size_t kLtWorkspace = size_t(32) << 20;

#define NG_LT_CHECK(call)                                                                      \
    do {                                                                                       \
        hipblasStatus_t ng_st_ = (call);                                                       \
        if (ng_st_ != HIPBLAS_STATUS_SUCCESS) {                                                \
            fprintf(stderr, "neurogrid-amd: %s:%d: hipBLASLt status %d\n", __FILE__, __LINE__, \
                    static_cast<int>(ng_st_));                                                 \
            return -1;                                                                         \
        }                                                                                      \
    } while (0)

struct Plan {
    hipblasLtMatmulDesc_t desc = nullptr;
    hipblasLtMatrixLayout_t lw = nullptr, lx = nullptr, ly = nullptr;
    hipblasLtMatmulAlgo_t algo{};
    size_t ws = 0;
};

// Buffers of one (device, stream) pair: the library workspace, the fp16 copy
// of the weights, and the split-K partial sums. Work on one
// stream is ordered, so reusing them from call to call on that stream is safe;
// another stream gets its own.
struct StreamBuffers {
    void* ws = nullptr;
    size_t ws_bytes = 0;
    void* deq = nullptr;
    size_t deq_bytes = 0;
    void* part = nullptr;
    size_t part_bytes = 0;
};

using PlanKey = std::tuple<int, int, int, int, bool, bool, int>;  // device, M, K, N, transpose_a, transpose_b, ldc

std::mutex g_mu;
std::map<int, hipblasLtHandle_t> g_handles;
std::map<PlanKey, Plan> g_plans;
std::set<PlanKey> g_lt_refused;   // shapes hipBLASLt has no algorithm for, or refused
std::map<std::pair<int, hipStream_t>, StreamBuffers> g_buffers;
// Buffers replaced by larger ones. A HIP graph that captured an earlier call
// still names the old buffer, so it is kept until gemm_release().
std::vector<void*> g_retired;

int capturing(hipStream_t s, bool* out) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    NG_HIP_CHECK(hipStreamIsCapturing(s, &st));
    *out = st != hipStreamCaptureStatusNone;
    return 0;
}

// Make *p hold at least `need` bytes. Growing while the stream is being
// captured is refused: allocation cannot be captured. The old buffer is
// retired, not freed, so that graphs captured before the growth stay valid;
// a new buffer is at least twice the old one, which bounds what is retired by
// the final size. Caller holds g_mu.
int grow(hipStream_t s, void** p, size_t* have, size_t need) {
    if (need <= *have) return 0;
    bool cap = false;
    if (capturing(s, &cap) != 0) return -1;
    NG_REQUIRE(!cap, "cuda_gemm: the stream is being captured and a buffer of %zu bytes must be allocated first; "
                     "make one call of this shape on the stream before capture", need);
    const size_t bytes = need > 2 * *have ? need : 2 * *have;
    void* fresh = nullptr;
    NG_HIP_CHECK(hipMalloc(&fresh, bytes));
    if (*p != nullptr) g_retired.push_back(*p);
    *p = fresh;
    *have = bytes;
    return 0;
}

// Plan for row-major C[M,N] = op(A) @ op(B), the rows of C ldc elements
// apart (ldc = N unless C is a column block of a wider matrix). hipBLASLt is
// column-major: the row-major matrices are their transposes, so it computes
// C^T = op(B)^T op(A)^T with B as its first operand (the same swap as
// matmul.cu:90-147).
int get_plan(int dev, int M, int K, int N, bool ta, bool tb, const Plan** out, int ldc = 0) {
    if (ldc == 0) ldc = N;
    const PlanKey key{dev, M, K, N, ta, tb, ldc};
    auto it = g_plans.find(key);
    if (it != g_plans.end()) {
        *out = &it->second;
        return 0;
    }
    auto h = g_handles.find(dev);
    if (h == g_handles.end()) {
        hipblasLtHandle_t handle = nullptr;
        NG_LT_CHECK(hipblasLtCreate(&handle));
        h = g_handles.emplace(dev, handle).first;
    }
    Plan p;
    NG_LT_CHECK(hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F));
    const int32_t op_w = tb ? HIPBLAS_OP_T : HIPBLAS_OP_N;
    const int32_t op_x = ta ? HIPBLAS_OP_T : HIPBLAS_OP_N;
    NG_LT_CHECK(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &op_w, sizeof(op_w)));
    NG_LT_CHECK(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &op_x, sizeof(op_x)));
    if (tb) NG_LT_CHECK(hipblasLtMatrixLayoutCreate(&p.lw, HIP_R_16F, K, N, K));
    else NG_LT_CHECK(hipblasLtMatrixLayoutCreate(&p.lw, HIP_R_16F, N, K, N));
    if (ta) NG_LT_CHECK(hipblasLtMatrixLayoutCreate(&p.lx, HIP_R_16F, M, K, M));
    else NG_LT_CHECK(hipblasLtMatrixLayoutCreate(&p.lx, HIP_R_16F, K, M, K));
    NG_LT_CHECK(hipblasLtMatrixLayoutCreate(&p.ly, HIP_R_16F, N, M, ldc));
    hipblasLtMatmulPreference_t pref = nullptr;
    NG_LT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
    const uint64_t ws = kLtWorkspace;
    NG_LT_CHECK(hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws,
                                                      sizeof(ws)));
    hipblasLtMatmulHeuristicResult_t res{};
    int found = 0;
    const hipblasStatus_t st =
        hipblasLtMatmulAlgoGetHeuristic(h->second, p.desc, p.lw, p.lx, p.ly, p.ly, pref, 1, &res, &found);
    hipblasLtMatmulPreferenceDestroy(pref);
    NG_LT_CHECK(st);
    NG_REQUIRE(found > 0, "cuda_gemm: hipBLASLt has no kernel for M=%d K=%d N=%d", M, K, N);
    p.algo = res.algo;
    p.ws = res.workspaceSize;
    *out = &g_plans.emplace(key, p).first->second;
    return 0;
}

// C = op(A) @ op(B) through hipBLASLt. With q != nullptr, B is first
// dequantized from the int8 codes q and their scales into this stream's fp16
// copy (matmul.cu:205-236), and the copy is the B of the product.
int gemm_lt(void* c, const void* a, const void* b, const void* q, const void* scale, int M, int K, int N, bool ta,
            bool tb) {
    int dev = 0;
    NG_HIP_CHECK(hipGetDevice(&dev));
    const hipStream_t s = stream();
    std::lock_guard<std::mutex> lock(g_mu);
    const Plan* p = nullptr;
    if (get_plan(dev, M, K, N, ta, tb, &p) != 0) return -1;
    StreamBuffers* sb = &g_buffers[{dev, s}];
    if (grow(s, &sb->ws, &sb->ws_bytes, p->ws) != 0) return -1;
    if (q != nullptr &&
        grow(s, &sb->deq, &sb->deq_bytes, static_cast<size_t>(K) * static_cast<size_t>(N) * 2) != 0)
        return -1;
    if (q != nullptr) {
        const int r = tb ? cuda_dequantize_weights(sb->deq, q, scale, N, K, 1)
                         : cuda_dequantize_weights(sb->deq, q, scale, K, N, 0);
        if (r != 0) return r;
        b = sb->deq;
    }
    const float alpha = 1.0f, beta = 0.0f;
    NG_LT_CHECK(hipblasLtMatmul(g_handles[dev], p->desc, &alpha, b, p->lw, a, p->lx, &beta, c, p->ly, c, p->ly,
                                &p->algo, sb->ws, p->ws, s));
    return 0;
}

// cuda_gemm_int8 from kLtMinM rows of A on, in the engine's layout (B int8
// [N, K], one scale per row): the reference's composition, dequantize then
// multiply (matmul.cu:205-236), through gemm_lt. It keeps a K x N fp16 copy
// of the weights in this (device, stream)'s buffer, grown to the largest
// weight seen (117 MB for a 14336 x 4096 projection), where the reference
// allocates and frees one per call. Measured on MI355X at M = 4096 for
// Mistral-7B's projections, eager calls back to back: 108-116 us for q/o against
// 116-125 us for the fused prefill kernel, 371 against 410 for gate or up, 337
// against 373 for down, 47 against 42 for k/v (not worth a rule of its own).
// Between 512 and 4096 rows the composition is not measured,
// so the fused kernel keeps those sizes. Returns 1 when hipBLASLt has no
// algorithm for the shape or refuses the call (remembered for the shape),
// having written nothing but the fp16 buffer: the caller then runs the fused
// prefill kernel.
constexpr int kLtMinM = 4096;

int gemm_lt_rows(void* c, const void* a, const void* q, const void* scale, int M, int K, int N) {
    int dev = 0;
    NG_HIP_CHECK(hipGetDevice(&dev));
    const hipStream_t s = stream();
    std::lock_guard<std::mutex> lock(g_mu);
    const PlanKey key{dev, M, K, N, false, true, N};
    if (g_lt_refused.count(key)) return 1;
    const Plan* p = nullptr;
    if (get_plan(dev, M, K, N, false, true, &p) != 0) {
        g_lt_refused.insert(key);
        return 1;
    }
    StreamBuffers* sb = &g_buffers[{dev, s}];
    if (grow(s, &sb->ws, &sb->ws_bytes, p->ws) != 0 ||
        grow(s, &sb->deq, &sb->deq_bytes, static_cast<size_t>(K) * static_cast<size_t>(N) * 2) != 0)
        return -1;
    const int r = cuda_dequantize_weights(sb->deq, q, scale, N, K, 1);
    if (r != 0) return r;
    const float alpha = 1.0f, beta = 0.0f;
    const hipblasStatus_t st = hipblasLtMatmul(g_handles[dev], p->desc, &alpha, sb->deq, p->lw, a, p->lx, &beta, c,
                                               p->ly, c, p->ly, &p->algo, sb->ws, p->ws, s);
    if (st != HIPBLAS_STATUS_SUCCESS) {
        // hipBLASLt's heuristic can name an algorithm that the call then
        // refuses (an internal error, status 6, at 4096 x 14336 x 512): the
        // shape goes to the fused kernel from now on, this call included.
        fprintf(stderr, "neurogrid-amd: hipBLASLt status %d at M=%d K=%d N=%d; using the fused kernel\n",
                static_cast<int>(st), M, K, N);
        g_lt_refused.insert(key);
        return 1;
    }
    return 0;
}

// The buffer of a split-K launch's `need` bytes of fp32 partial sums: `scratch`
// when the caller brings one (refused when too small), else this (device,
// stream)'s buffer, grown on demand with `lock` (g_mu) taken; the caller
// keeps the lock until both kernels are enqueued, so that calls from other
// host threads on the same stream cannot slip a launch between them.
int partial_buffer(hipStream_t s, size_t need, float* scratch, size_t scratch_bytes,
                   std::unique_lock<std::mutex>& lock, float** out) {
    if (scratch != nullptr) {
        NG_REQUIRE(need <= scratch_bytes,
                   "ng_gemm_int8_noalloc: the partial sums of the slices of K need %zu bytes, more than the "
                   "%zu-byte scratch; call cuda_gemm_int8 instead", need, scratch_bytes);
        *out = scratch;
        return 0;
    }
    int dev = 0;
    NG_HIP_CHECK(hipGetDevice(&dev));
    lock.lock();
    StreamBuffers* sb = &g_buffers[{dev, s}];
    if (grow(s, &sb->part, &sb->part_bytes, need) != 0) return -1;
    *out = static_cast<float*>(sb->part);
    return 0;
}

// Whether partial_buffer can give `need` bytes on stream s: not when they would
// have to be allocated while it is captured.
bool partial_room(hipStream_t s, size_t need) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (need <= g_buffers[{dev, s}].part_bytes) return true;
    }
    bool cap = false;
    return capturing(s, &cap) == 0 && !cap;
}

// C = fp16(scale[n] * sum of the S slices of part), slices added in order.
int launch_reduce(hipStream_t s, uint16_t* c, const float* part, const float* scale, int M, int N, int S,
                  const ResEpi* ep = nullptr) {
    const size_t mn = static_cast<size_t>(M) * N;
    const dim3 b4(static_cast<unsigned>((mn / 4 + 255) / 256)), b1(static_cast<unsigned>((mn + 255) / 256));
    const bool vec4 = N % 4 == 0 && aligned16(scale) && aligned8(c) && (!ep || (aligned8(ep->out) && aligned8(ep->res)));
    if (ep) {
        if (vec4) split_reduce_kernel<true, true><<<b4, dim3(256), 0, s>>>(c, part, scale, M, N, S, *ep);
        else split_reduce_kernel<false, true><<<b1, dim3(256), 0, s>>>(c, part, scale, M, N, S, *ep);
    } else {
        if (vec4) split_reduce_kernel<true><<<b4, dim3(256), 0, s>>>(c, part, scale, M, N, S);
        else split_reduce_kernel<false><<<b1, dim3(256), 0, s>>>(c, part, scale, M, N, S);
    }
    NG_CHECK_LAUNCH("cuda_gemm_int8");
    return 0;
}

// Slices of K for a split launch of `tiles` tiles of B:
// enough for about 256 blocks (512 for K >= 8192; with G groups in the
// block, 192 blocks of twice the waves), at most 8, each of at least two
// turns, none empty; cps batches of 128 k per slice.
void split_slices(int tiles, int G, int K, int& S, int& cps) {
    const int nbatch = (K + kBatch - 1) / kBatch;
    const int target = G > 1 ? 192 : K >= 8192 ? 512 : 256;
    S = (target + tiles - 1) / tiles;
    S = max(1, min(S, min(8, nbatch / (2 * G))));
    cps = (nbatch + S - 1) / S;
    S = (nbatch + cps - 1) / cps;
}

template <int MT, int W, int G>
int launch_split(uint16_t* c, const uint16_t* a, const int8_t* b, const float* scale, int M, int N, int K,
                 float* scratch, size_t scratch_bytes, const ResEpi* ep = nullptr) {
    const int tiles = (N + 16 * W - 1) / (16 * W);
    int S = 0, cps = 0;
    split_slices(tiles, G, K, S, cps);
    // With S > 1 the partial-sum buffer is this stream's: the lock is held
    // until both kernels are enqueued, so calls from other host threads on the
    // same stream cannot slip a launch between them.
    const hipStream_t s = stream();
    float* part = nullptr;
    std::unique_lock<std::mutex> lock(g_mu, std::defer_lock);
    const size_t need = static_cast<size_t>(S) * M * N * sizeof(float);
    if (S > 1 && partial_buffer(s, need, scratch, scratch_bytes, lock, &part) != 0) return -1;
    gemm_i8w_split_kernel<MT, W, G><<<dim3(static_cast<unsigned>(tiles * S)), dim3(G * W * kWave), 0, s>>>(
        c, a, b, scale, part, M, N, K, S, cps);
    NG_CHECK_LAUNCH("cuda_gemm_int8");
    if (S > 1) return launch_reduce(s, c, part, scale, M, N, S, ep);
    return ep ? cuda_add(ep->out, c, ep->res, static_cast<size_t>(M) * N) : 0;
}

// The GEMV kernel gemm_i8w runs for a product on the weight-streaming path:
// 1 (one row of A, 8 rows of B per block), 2 (two rows of A, 8 of B), 3 (up
// to four rows of A, 4 of B), or 0 for the MFMA kernels. The GEMV kernel
// takes M <= 4 and K % 16 == 0, except M = 3, 4 with K or N of 8192 or more
// and K % 64 == 0, where the split kernel is faster.
int gemv_shape(int M, int K, int N) {
    const bool big = K >= 8192 || N >= 8192;
    if (M > 4 || K % 16 != 0 || (M >= 3 && big && K % kChunk == 0)) return 0;
    return M == 1 ? 1 : M == 2 ? 2 : 3;
}

// The split kernel's launch shape <MT, W, G> that gemm_i8w takes up to 32
// rows of A when the GEMV kernel does not, or kSmallM for the small-M MFMA kernel:
//   K >= 8192 (down): 8 waves per block above 16 rows;
//   N >= 12288 at smaller K (gate/up): 192 or more tiles of 64 rows fill the
//   GPU with one slice of K, split between two groups of 4 waves per block;
//   M <= 16 with K and N below 8192: the small-M MFMA kernel.
enum SplitConfig { kSmallM, kSplit281, kSplit242, kSplit241, kSplit142, kSplit141 };
SplitConfig split_config(int M, int K, int N) {
    const bool big = K >= 8192 || N >= 8192;
    const bool deep = K >= 8192;
    const bool wide = !deep && N >= 12288;
    if (M > 16) return deep ? kSplit281 : wide ? kSplit242 : kSplit241;
    if (big) return wide ? kSplit142 : kSplit141;
    return kSmallM;
}

// ng_gemm_int8_shared_a's paths of the products on the prefill kernel and on
// the 33 - 128 row kernel.
constexpr int kPathPrefill = 40, kPathRing2 = 41, kPathRing4 = 42;
constexpr int kRingMinM = 33;

void ring_slices(int M, int N, int K, int& wk, int& S, int& cps);
int gemm_ring(int count, void* const* c, const void* a, const void* const* b, const void* const* scales, const int* n,
              int M, int K, float* scratch = nullptr, size_t scratch_bytes = 0, const ResEpi* ep = nullptr,
              const SwigluArgs* sw = nullptr);

// The launch shape gemm_i8w takes for a product on the weight-streaming
// path, for ng_gemm_int8_shared_a: the GEMV shapes 1-3 above, 4 for the
// small-M MFMA kernel, 10 + c for split shape c, kPathRing2 or kPathRing4 by the
// groups of the 33 - 128 row kernel.
int shared_path(int M, int K, int N) {
    const int gv = gemv_shape(M, K, N);
    if (gv != 0) return gv;
    if (M >= kRingMinM) {
        int wk = 0, S = 0, cps = 0;
        ring_slices(M, N, K, wk, S, cps);
        return wk == 2 ? kPathRing2 : kPathRing4;
    }
    const SplitConfig sc = split_config(M, K, N);
    return sc == kSmallM ? 4 : 10 + static_cast<int>(sc);
}

// Kernel and tile shape by M, K and N, from sweeps on MI355X over K x N in
// {4096 x 4096, 4096 x 1024, 4096 x 14336, 14336 x 4096} and M from 1 to 128:
// the GEMV kernel up to M = 4 (8 rows of B per block for M <= 2, 4 for M = 3,
// 4: 23-33% faster than the MFMA kernels at M = 1), the split kernel from
// M = 17 on and from M = 3 on with K or N of 8192 or more (at M = 4: 13.4 vs
// 14.8 us for gate/up, 13.7 vs 15.5 us for down), the ring kernel from M = 33
// on, otherwise the MFMA kernel that reads A from L2 directly.
// With ep, the residual add after the product follows: in the split-K
// reduction's epilogue where the launch has several K slices, in the ring
// kernel's where it has one, else as cuda_add.
int gemm_i8w(void* c, const void* a, const void* b, const void* scale, int M, int K, int N,
             float* scratch = nullptr, size_t scratch_bytes = 0, const ResEpi* ep = nullptr) {
    auto* cp = static_cast<uint16_t*>(c);
    auto* ap = static_cast<const uint16_t*>(a);
    auto* bp = static_cast<const int8_t*>(b);
    auto* sp = static_cast<const float*>(scale);
    const auto then_add = [&](int r) {
        return r != 0 || !ep ? r : cuda_add(ep->out, c, ep->res, static_cast<size_t>(M) * N);
    };
    switch (gemv_shape(M, K, N)) {
        case 1: return then_add(launch_gemv<1, 8>(cp, ap, bp, sp, M, N, K));
        case 2: return then_add(launch_gemv<2, 8>(cp, ap, bp, sp, M, N, K));
        case 3: return then_add(launch_gemv<4, 4>(cp, ap, bp, sp, M, N, K));
        default: break;
    }
    if (M >= kRingMinM) return gemm_ring(1, &c, a, &b, &scale, &N, M, K, scratch, scratch_bytes, ep);
    switch (split_config(M, K, N)) {
        case kSplit281: return launch_split<2, 8, 1>(cp, ap, bp, sp, M, N, K, scratch, scratch_bytes, ep);
        case kSplit242: return launch_split<2, 4, 2>(cp, ap, bp, sp, M, N, K, scratch, scratch_bytes, ep);
        case kSplit241: return launch_split<2, 4, 1>(cp, ap, bp, sp, M, N, K, scratch, scratch_bytes, ep);
        case kSplit142: return launch_split<1, 4, 2>(cp, ap, bp, sp, M, N, K, scratch, scratch_bytes, ep);
        case kSplit141: return launch_split<1, 4, 1>(cp, ap, bp, sp, M, N, K, scratch, scratch_bytes, ep);
        default: return then_add(launch_i8w<1, 1, 8, 4>(cp, ap, bp, sp, M, N, K));
    }
}

// The prefill kernel takes transpose_b, K % 16 == 0 and 16-byte aligned A and B.
bool use_prefill(const void* a, const void* b, int M, int K, int N, bool transpose_b) {
    return transpose_b && K % 16 == 0 && aligned16(a) && aligned16(b) &&
           static_cast<long long>(M) * K * 2 < (1ll << 31) && static_cast<long long>(N) * K < (1ll << 31);
}

// Per-product plan of a shared split-K launch: K slices, batches per slice,
// tiles along N and along M, and blocks.
struct SharedPlan {
    int S[kMaxShared], cps[kMaxShared], tn[kMaxShared], tm[kMaxShared];
    long long blocks[kMaxShared];
};

// Floats of partial sums of a launch of `count` products, the regions of those
// with K slices one after the other, each on 16 bytes; the starts in `at`.
size_t partial_floats(int count, const int* n, int M, const int* S, size_t* at = nullptr) {
    size_t end = 0;
    for (int i = 0; i < count; ++i) {
        if (S[i] == 1) continue;
        const size_t start = (end + 3) / 4 * 4;
        if (at != nullptr) at[i] = start;
        end = start + static_cast<size_t>(S[i]) * M * n[i];
    }
    return end;
}

// Products that share A on one split-K kernel shape: one launch of the kernel
// (`launch(set, sp, blocks, stream)`), then one of the reduction for the products with
// more than one slice of K, each product with its own slices and its own
// region of the stream's partial-sum buffer (the lock is held until both
// kernels are enqueued, as in launch_split).
// With sw (gate and up, both with several K slices, as count 2), the
// reduction is split_reduce_swiglu_kernel's; otherwise it returns 1 before
// launching anything. With ep (a product alone), the residual add follows in
// its reduction; scratch is a partial-sum buffer that the caller brings.
template <typename L>
int run_shared_split(int count, void* const* c, const void* const* b, const void* const* scales, const int* n,
                     int M, int K, const SharedPlan& pl, L&& launch, const SwigluArgs* sw = nullptr,
                     float* scratch = nullptr, size_t scratch_bytes = 0, const ResEpi* ep = nullptr) {
    if (sw && !(count == 2 && n[0] == n[1] && pl.S[0] > 1 && pl.S[1] == pl.S[0])) return 1;
    size_t at[kMaxShared] = {};
    const size_t floats = partial_floats(count, n, M, pl.S, at);
    const hipStream_t st = stream();
    float* part = nullptr;
    std::unique_lock<std::mutex> lock(g_mu, std::defer_lock);
    if (floats > 0 && partial_buffer(st, floats * sizeof(float), scratch, scratch_bytes, lock, &part) != 0) return -1;
    SharedSet set{}, rset{};
    SplitSet sp{};
    long long blocks = 0, rblocks = 0;
    bool vec4_all = true, vec4_any = false;
    for (int i = 0; i < kMaxShared; ++i) {
        const int j = i < count ? i : 0;  // unused slots repeat product 0 and are never selected
        set.c[i] = rset.c[i] = static_cast<uint16_t*>(c[j]);
        set.b[i] = rset.b[i] = static_cast<const int8_t*>(b[j]);
        set.scale[i] = rset.scale[i] = static_cast<const float*>(scales[j]);
        set.n[i] = rset.n[i] = n[j];
        sp.S[i] = pl.S[j];
        sp.tiles[i] = pl.tn[j];
        sp.cps[i] = pl.cps[j];
        sp.TT[i] = pl.tm[j];
        sp.part[i] = nullptr;
        set.first[i] = i < count ? static_cast<int>(blocks) : INT_MAX;
        rset.first[i] = i < count ? static_cast<int>(rblocks) : INT_MAX;
        if (i >= count) continue;
        blocks += pl.blocks[i];
        if (pl.S[i] > 1) {
            sp.part[i] = part + at[i];
            const bool v4 = n[i] % 4 == 0 && aligned16(scales[i]) && aligned8(c[i]);
            vec4_all = vec4_all && v4;
            vec4_any = vec4_any || v4;
            const long long mn = static_cast<long long>(M) * n[i];
            rblocks += v4 ? (mn / 4 + 255) / 256 : (mn + 255) / 256;
        }
        NG_REQUIRE(blocks < (1ll << 31) && rblocks < (1ll << 31), "ng_gemm_int8_shared_a: too many rows of B");
    }
    launch(set, sp, static_cast<unsigned>(blocks), st);
    NG_CHECK_LAUNCH("ng_gemm_int8_shared_a");
    if (sw) {
        const bool v4 = n[0] % 4 == 0 && aligned16(sw->sg) && aligned16(sw->su) && aligned8(sw->gate) &&
                        aligned8(sw->up) && aligned8(sw->out);
        const long long mn = static_cast<long long>(M) * n[0];
        const unsigned sb = static_cast<unsigned>(v4 ? (mn / 4 + 255) / 256 : (mn + 255) / 256);
        if (v4)
            split_reduce_swiglu_kernel<true><<<dim3(sb), dim3(256), 0, st>>>(*sw, sp.part[0], sp.part[1], M, n[0],
                                                                             pl.S[0]);
        else
            split_reduce_swiglu_kernel<false><<<dim3(sb), dim3(256), 0, st>>>(*sw, sp.part[0], sp.part[1], M, n[0],
                                                                              pl.S[0]);
        NG_CHECK_LAUNCH("ng_gemm_int8_silu_mul");
        return 0;
    }
    if (rblocks == 0) return 0;
    if (count == 1) return launch_reduce(st, set.c[0], part, set.scale[0], M, n[0], pl.S[0], ep);
    if (vec4_all || !vec4_any) {
        if (vec4_all)
            split_reduce_shared_kernel<true><<<dim3(static_cast<unsigned>(rblocks)), dim3(256), 0, st>>>(rset, sp, M);
        else
            split_reduce_shared_kernel<false><<<dim3(static_cast<unsigned>(rblocks)), dim3(256), 0, st>>>(rset, sp, M);
        NG_CHECK_LAUNCH("ng_gemm_int8_shared_a");
        return 0;
    }
    // Products whose reductions take different forms: one reduction each.
    for (int i = 0; i < count; ++i)
        if (pl.S[i] > 1 && launch_reduce(st, static_cast<uint16_t*>(c[i]), sp.part[i],
                                         static_cast<const float*>(scales[i]), M, n[i], pl.S[i]) != 0)
            return -1;
    return 0;
}

// Tile shapes of the prefill kernel, <BM, BN, 2, 4, NST>, and the time of a
// launch on each on MI355X, in us: fixed, plus for each step of 64 k of a block
// lo with few blocks on the GPU, rising from a share `knee` of the 256 CUs to hi
// at one block for each (the clock falls as the matrix cores fill), and more for
// every full round of a launch of several. Fitted to 544 launches of
// M = 130 - 3000 at N = 1024 - 28672, K = 2048 - 14336 with 1 - 8 slices on every
// shape; taken by it a launch is at most 10% (0.5% on average) above the fastest
// of all shapes and slices. The 192 row tiles are for M that 128 and 256 divide
// badly (gate/up of 333 rows, 4096 -> 2 x 14336: 90 us, 107 on 256 x 256; of 190
// rows 57, 70 on 128 x 256) and in slices for down (900 x 4096 x 14336: 116 us
// in three, 138 on 128 x 256). Also measured and slower than the best of these
// wherever they could be taken: 64 x 256, 64 x 64, 128 x 128 with 4 waves or 6
// stages, and 4 x 2 waves on 256 x 128.
struct TileShape {
    int BM, BN;
    double fixed, lo, hi, knee, more;
};
constexpr TileShape kTileShapes[] = {
    {256, 256, 9.1, 1.097, 1.534, 0.49, 1.694}, {192, 256, 8.4, 0.899, 1.236, 0.56, 1.353},
    {256, 128, 7.3, 0.653, 0.906, 0.47, 0.994}, {128, 256, 7.3, 0.714, 0.969, 0.61, 1.025},
    {192, 128, 6.4, 0.507, 0.732, 0.45, 0.792}, {128, 128, 5.3, 0.425, 0.587, 0.54, 0.527},
    {64, 128, 4.4, 0.324, 0.398, 0.58, 0.349}};
constexpr int kTileShapeCount = 7, kTileSerialFirst = 2;

// CUs of the device that the times were fitted on. Not the present device's: slices,
// and with them the bits, would then depend on how it is partitioned.
constexpr int kTileCus = 256;

// Time of a launch of `blocks` blocks of `steps` steps each on average.
double tile_time(const TileShape& ts, long long blocks, double steps) {
    const long long full = blocks / kTileCus;
    const double rest = static_cast<double>(blocks % kTileCus) / kTileCus;
    double step;
    if (full == 0) step = ts.lo + (rest > ts.knee ? (ts.hi - ts.lo) * (rest - ts.knee) / (1.0 - ts.knee) : 0.0);
    else if (rest == 0.0) step = full == 1 ? ts.hi : ts.more * full;
    else step = ts.more * full + ts.lo + (ts.more - ts.lo) * rest;
    return ts.fixed + step * steps;
}

long long tile_blocks(const TileShape& ts, int M, int N) {
    return ((static_cast<long long>(M) + ts.BM - 1) / ts.BM) * ((static_cast<long long>(N) + ts.BN - 1) / ts.BN);
}

// K slices of a product on the prefill kernel: a function of M, N and K alone,
// so that a product has the same bits in every launch that it is part of.
// The S <= 8 of least time over the tile shapes, each slice of 8 steps or more
// and the partial sums within the fixed array of ng_gemm_int8_noalloc, the
// reduction counted as 3 us and 0.3 us a MB of partial sums; more than one only
// where it saves 2% (333 x 4096 x 14336: 57 us with four slices, 83 with one;
// 130 x 4096 x 4096 19 us with two, 25 with one).
void prefill_slices(int M, int N, int K, int& S, int& cps) {
    const int nk = (K + kPfBK - 1) / kPfBK;
    double one = 0.0, best = 0.0;
    S = 1;
    cps = nk;
    long long tiles[kTileShapeCount];
    for (int k = 0; k < kTileShapeCount; ++k) tiles[k] = tile_blocks(kTileShapes[k], M, N);
    for (int s = 1; s <= 8; ++s) {
        const int per = (nk + s - 1) / s, ss = (nk + per - 1) / per;
        const double bytes = static_cast<double>(ss) * M * N * sizeof(float);
        if (s > 1 && (per < 8 || ss < s || bytes > static_cast<double>(kNoAllocScratchBytes))) continue;
        const double steps = static_cast<double>(nk) / ss;
        double t = 0.0;
        for (int k = 0; k < kTileShapeCount; ++k) {
            const double v = tile_time(kTileShapes[k], tiles[k] * ss, steps);
            if (t == 0.0 || v < t) t = v;
        }
        if (ss > 1) t += 3.0 + 0.3e-6 * bytes;
        if (s == 1) one = best = t;
        if (s > 1 && t < 0.98 * one && t < best) {
            best = t;
            S = ss;
            cps = per;
        }
    }
}

template <int BM, int BN, int WM, int WN, int NST, bool SERIAL = false>
int launch_tiles(int count, void* const* c, const uint16_t* a, const void* const* b, const void* const* scales,
                 const int* n, int M, int K, SharedPlan& pl, float* scratch, size_t scratch_bytes, const ResEpi* ep,
                 const SwigluArgs* sw) {
    const dim3 block(WM * WN * kWave);
    if (sw && pl.S[0] == 1) {
        const int tm = (M + BM - 1) / BM, tn = (n[0] + BN / 2 - 1) / (BN / 2);
        gemm_i8w_tile_swiglu_kernel<BM, BN, WM, WN, NST><<<dim3(static_cast<unsigned>(tm) * tn), block, 0, stream()>>>(
            *sw, a, M, n[0], K, tm, tn, pl.cps[0]);
        NG_CHECK_LAUNCH("ng_gemm_int8_silu_mul");
        return 0;
    }
    for (int i = 0; i < count; ++i) {
        pl.tm[i] = (M + BM - 1) / BM;
        pl.tn[i] = (n[i] + BN - 1) / BN;
        pl.blocks[i] = static_cast<long long>(pl.tm[i]) * pl.tn[i] * pl.S[i];
    }
    const TileEpi te{ep && pl.S[0] == 1 ? ep->out : nullptr, ep && pl.S[0] == 1 ? ep->res : nullptr};
    return run_shared_split(count, c, b, scales, n, M, K, pl,
                            [&](const SharedSet& set, const SplitSet& sp, unsigned blocks, hipStream_t st) {
                                gemm_i8w_tile_kernel<BM, BN, WM, WN, NST, SERIAL>
                                    <<<dim3(blocks), block, 0, st>>>(set, sp, a, M, K, te);
                            },
                            sw, scratch, scratch_bytes, ep);
}

// Products that share A on the prefill kernel, in one launch (plus one of the
// reduction where a product has K slices), on the tile shape of least time for
// all of them. ep (a product alone): the residual add after it. sw (gate and
// up): SwiGLU after them.
// Of several products narrow ones have slices that pay alone but not beside a
// wide one, whose blocks fill the GPU meanwhile: there a block takes all slices
// of its tile, with the same bits, where that is the faster estimate, on the
// shapes whose second set of sums fits in registers (q/k/v of 4096, 1024 and
// 1024 rows, K = 4096, with k and v in 4 slices: 512 rows 38 against 48 us, 700
// rows 45 against 55; with slices of 2, 8 and 8 at 190 rows 27 against 26). A
// launch under capture that finds no buffer for its partial sums does the same
// (not with sw: 1 is returned before launching anything).
int gemm_tiles(int count, void* const* c, const void* a, const void* const* b, const void* const* scales,
               const int* n, int M, int K, float* scratch = nullptr, size_t scratch_bytes = 0,
               const ResEpi* ep = nullptr, const SwigluArgs* sw = nullptr) {
    const auto* ap = static_cast<const uint16_t*>(a);
    SharedPlan pl{};
    const int nk = (K + kPfBK - 1) / kPfBK;
    int longest = 0;
    for (int i = 0; i < count; ++i) {
        prefill_slices(M, n[i], K, pl.S[i], pl.cps[i]);
        longest = max(longest, pl.cps[i]);
    }
    const size_t part_bytes = sizeof(float) * partial_floats(count, n, M, pl.S);
    const double reduce = part_bytes > 0 ? 3.0 + 0.3e-6 * part_bytes : 0.0;
    const bool room = part_bytes == 0 || scratch != nullptr || partial_room(stream(), part_bytes);
    if (sw && !room) return 1;
    // The shape of least time, with a block per slice and with all slices in one.
    const auto best = [&](bool serial, int first, double& least) {
        int shape = first;
        for (int k = first; k < kTileShapeCount; ++k) {
            long long blocks = 0, steps = 0;
            for (int i = 0; i < count; ++i) {
                const long long tiles = tile_blocks(kTileShapes[k], M, n[i]);
                blocks += serial ? tiles : tiles * pl.S[i];
                steps += tiles * nk;
            }
            double t = tile_time(kTileShapes[k], blocks, static_cast<double>(steps) / blocks);
            if (!serial) t = reduce + std::max(t, kTileShapes[k].fixed + kTileShapes[k].lo * longest);
            if (k == first || t < least) {
                least = t;
                shape = k;
            }
        }
        return shape;
    };
    double least = 0.0;
    const int shape = best(false, 0, least);
    if (!sw && part_bytes > 0 && (count > 1 || !room)) {
        double least_serial = 0.0;
        const int serial = best(true, kTileSerialFirst, least_serial);
        if (!room || 1.02 * least_serial < least) {
            for (int i = 0; i < count; ++i) pl.S[i] = 1;
#define NG_TILES(BM, BN, NST) return launch_tiles<BM, BN, 2, 4, NST, true>(count, c, ap, b, scales, n, M, K, pl, scratch, scratch_bytes, ep, sw)
            switch (serial) {
                case 2: NG_TILES(256, 128, 3);
                case 3: NG_TILES(128, 256, 4);
                case 4: NG_TILES(192, 128, 3);
                case 5: NG_TILES(128, 128, 3);
                default: NG_TILES(64, 128, 4);
            }
#undef NG_TILES
        }
    }
#define NG_TILES(BM, BN, NST) \
    return launch_tiles<BM, BN, 2, 4, NST>(count, c, ap, b, scales, n, M, K, pl, scratch, scratch_bytes, ep, sw)
    switch (shape) {
        case 0: NG_TILES(256, 256, 3);
        case 1: NG_TILES(192, 256, 3);
        case 2: NG_TILES(256, 128, 3);
        case 3: NG_TILES(128, 256, 4);
        case 4: NG_TILES(192, 128, 3);
        case 5: NG_TILES(128, 128, 3);
        default: NG_TILES(64, 128, 4);
    }
#undef NG_TILES
}

// The 33 - 128 row kernel's 64-k groups of a block and K slices of a product,
// by its M, N and K alone (they show in the bits; tile sizes do not). Times in us.
//   Groups: four up to 64 rows; two for wide products (gate/up), whose tiles are
//   128 wide, for the longest K, and above 64 rows, where four leave room for two
//   stages only - but four for short K, on small tiles (K and N of 2048 at 128
//   rows 5.8, with two 8.9).
//   Slices: one for wide products and short K, whose reduction costs more than it
//   gains; else for about 128 blocks of 64 rows of B, at K >= 8192 twice (above 64
//   rows four times) that. N = 2048 up to K = 4096 two only: three such products
//   fill the GPU with them (at 33 rows 13.8, with four each 16.5). K of 16384 and
//   more by 8192 rows of B and more three or four (28672 x 8192 at 64 rows 52.9,
//   with two on narrower tiles 62). Narrow products (k/v) would leave most of the
//   GPU idle: slices of 1024 k (above 64 rows and below N = 1024 of 512) up to
//   about one small tile for each CU (N = 512, K = 4096 at 96 rows 6.8, with four
//   8.6).
constexpr int kRingWideN = 10240;
constexpr int kRingNarrowN = 1024;

void ring_slices(int M, int N, int K, int& wk, int& S, int& cps) {
    const int tiles = (N + 63) / 64, rows = (M + 31) / 32;
    const bool wide = N >= kRingWideN, narrow = N <= kRingNarrowN, shallow = K <= 2048;
    const bool longest = K >= 16384 && N >= 8192;
    wk = wide || (M > 64 ? !(shallow && K >= 512 && N <= 4096) : longest) ? 2 : 4;
    const int nk = (K + 64 * wk - 1) / (64 * wk);
    if (wide || shallow) S = 1;
    else if (longest && M <= 64) S = K > 16384 ? 4 : 3;
    else if (K >= 8192) S = min((M > 64 ? 512 : 256) / tiles, 8);
    else if (!narrow) S = min(128 / tiles, M > 64 ? K / 1024 : K > 4096 || N > 2048 || N <= 1792 ? 4 : 2);
    else S = min(min(8, 256 / (rows * (M > 64 ? tiles : (N + 31) / 32))), K / (M > 64 && N < kRingNarrowN ? 512 : 1024));
    S = max(S, 1);
    cps = (nk + S - 1) / S;
    S = (nk + cps - 1) / cps;
}

template <int BM, int BN, int WK, int NST, bool SERIAL = false>
int launch_ring(int count, void* const* c, const uint16_t* a, const void* const* b, const void* const* scales,
                const int* n, int M, int K, SharedPlan& pl, float* scratch, size_t scratch_bytes, const ResEpi* ep,
                const SwigluArgs* sw) {
    constexpr int WN = BN / 32;
    const dim3 block(WN * WK * kWave);
    const int TT = (M + BM - 1) / BM;
    const auto blocks_of = [&](long long units) { return TT > 1 ? (units + 7) / 8 * 8 * TT : units; };
    if constexpr (!SERIAL) {
        if (sw && pl.S[0] == 1) {
            const int tiles = (n[0] + BN / 2 - 1) / (BN / 2);
            gemm_i8w_ring_swiglu_kernel<BM, BN, WN, WK, NST>
                <<<dim3(static_cast<unsigned>(blocks_of(tiles))), block, 0, stream()>>>(*sw, a, M, n[0], K, tiles,
                                                                                        pl.cps[0], TT);
            NG_CHECK_LAUNCH("ng_gemm_int8_silu_mul");
            return 0;
        }
    }
    for (int i = 0; i < count; ++i) {
        pl.tm[i] = TT;
        pl.tn[i] = (n[i] + BN - 1) / BN;
        pl.blocks[i] = blocks_of(static_cast<long long>(pl.tn[i]) * pl.S[i]);
    }
    const TileEpi te{ep && pl.S[0] == 1 ? ep->out : nullptr, ep && pl.S[0] == 1 ? ep->res : nullptr};
    return run_shared_split(count, c, b, scales, n, M, K, pl,
                            [&](const SharedSet& set, const SplitSet& sp, unsigned blocks, hipStream_t st) {
                                if constexpr (!SERIAL) {
                                    if (count == 1) {
                                        gemm_i8w_ring_kernel<BM, BN, WN, WK, NST><<<dim3(blocks), block, 0, st>>>(
                                            set.c[0], a, set.b[0], set.scale[0], sp.part[0], M, set.n[0], K, sp.S[0],
                                            sp.tiles[0], sp.cps[0], TT, te);
                                        return;
                                    }
                                }
                                gemm_i8w_ring_shared_kernel<BM, BN, WN, WK, NST, SERIAL>
                                    <<<dim3(blocks), block, 0, st>>>(set, sp, a, M, K);
                            },
                            sw, scratch, scratch_bytes, ep);
}

// Products that share A at 33 to 128 rows and take the same groups; other
// arguments as gemm_tiles. Tile by the number of blocks: the widest that still
// gives every CU one, and rows of A cut into tiles of 32 too where that takes
// fewer rounds of blocks. Measured in us, four groups: K = 4096 at 64 rows, N =
// 1024 6.8 on 32 x 32 and 8.3 on 64 x 32, N = 4096 11.4 on 32 x 64 and 13.1 on 64 x
// 64; slices of 1024 k or less pay too little for that (N = 8192, K = 1024 at 33
// rows 5.6 on 64 x 32, 6.1 on 32 x 64). Two groups up to 64 rows: 64 x 64, six
// stages deep or, two blocks per CU, three (N = 11008, K = 4096: 17.4 and 18.3 at 33
// rows, 19.9 and 19.6 at 64), up to a block for each CU or where nearly two fit it
// (N = 32000, K = 4096 at 33 rows 33.3, on 64 x 128 36.0), 64 x 128 between and for
// SwiGLU. Above 64 rows 32 x 64 in one round, or in two of short slices (N = 1024,
// K = 4096 at 96 rows 7.9, on eight stages of it 8.3), then wider.
// A set whose sliced products take more than one round has both slices of a tile
// in one block (SERIAL: three products of 4096 rows of B, K = 4096, at 33, 48 and 64
// rows 18, 19 and 21; with a block per slice 24, 24 and 26). Several products on a
// stream under capture whose buffer holds the partial sums of each but not of all
// of them: one launch each (with sw 1 is returned before launching anything), as
// separate calls.
int gemm_ring(int count, void* const* c, const void* a, const void* const* b, const void* const* scales, const int* n,
              int M, int K, float* scratch, size_t scratch_bytes, const ResEpi* ep, const SwigluArgs* sw) {
    const auto* ap = static_cast<const uint16_t*>(a);
    SharedPlan pl{};
    int wk = 0;
    const int rows32 = (M + 31) / 32;
    long long b32 = 0, b64 = 0, b128 = 0;
    int most = 1, longest = 0;  // slices of a product, steps of a slice
    for (int i = 0; i < count; ++i) {
        ring_slices(M, n[i], K, wk, pl.S[i], pl.cps[i]);
        most = max(most, pl.S[i]);
        longest = max(longest, pl.cps[i]);
        b32 += (static_cast<long long>(n[i]) + 31) / 32 * pl.S[i];
        b64 += (static_cast<long long>(n[i]) + 63) / 64 * pl.S[i];
        b128 += (static_cast<long long>(n[i]) + 127) / 128 * pl.S[i];
    }
    const bool serial = count > 1 && !sw && M <= 64 && wk == 4 && most == 2 && b64 > 256;
    const size_t floats = serial ? 0 : partial_floats(count, n, M, pl.S);
    if (count > 1 && floats > 0 && !partial_room(stream(), floats * sizeof(float))) {
        if (sw) return 1;
        for (int i = 0; i < count; ++i)
            if (gemm_ring(1, c + i, a, b + i, scales + i, n + i, M, K) != 0) return -1;
        return 0;
    }
    const auto rounds = [](long long blocks) { return (blocks + 255) / 256; };  // at a block per CU
#define NG_RING(BM, BN, WK, NST) \
    return launch_ring<BM, BN, WK, NST>(count, c, ap, b, scales, n, M, K, pl, scratch, scratch_bytes, ep, sw)
    if (wk == 4) {
        if (b32 * rows32 <= 256) NG_RING(32, 32, 4, 3);
        if (longest <= 4 && b32 <= 256 && M <= 64) NG_RING(64, 32, 4, 4);
        if (count > 1 && most >= 4 && b32 * rows32 <= 512) NG_RING(32, 32, 4, 3);
        if (7 * rounds(b64 * rows32) < 10 * rounds(b64 * ((M + 63) / 64))) NG_RING(32, 64, 4, 4);
        if (serial) {
            for (int i = 0; i < count; ++i) pl.S[i] = 1;
            return launch_ring<64, 64, 4, 3, true>(count, c, ap, b, scales, n, M, K, pl, scratch, scratch_bytes, ep, sw);
        }
        NG_RING(64, 64, 4, 3);
    }
    if (M <= 64) {
        if (!sw && b64 <= 256 && M <= 48 && K > 2048) NG_RING(64, 64, 2, 6);
        if (!sw && (b64 <= 256 || (b64 <= 512 && (b64 > 448 ? K <= 4096 : count == 1 && K <= 1024)))) NG_RING(64, 64, 2, 3);
        NG_RING(64, 128, 2, 4);
    }
    if (b64 * rows32 <= (most >= 4 ? 512 : 256)) NG_RING(32, 64, 2, 4);
    if (b64 <= 128) NG_RING(64, 64, 2, 6);
    if (b128 >= 160) {
        if (M <= 96) NG_RING(96, 128, 2, 3);
        NG_RING(128, 128, 2, 3);
    }
    if (M <= 96) NG_RING(96, 64, 2, 5);
    NG_RING(128, 64, 2, 4);
#undef NG_RING
}

int gemm_prefill(void* c, const void* a, const void* b, const void* scale, int M, int K, int N,
                 float* scratch = nullptr, size_t scratch_bytes = 0, const ResEpi* ep = nullptr) {
    return gemm_tiles(1, &c, a, &b, &scale, &N, M, K, scratch, scratch_bytes, ep);
}

// The weight-streaming path takes transpose_b, M <= kMaxFusedM, 16-byte aligned
// A and B, and K % 64 == 0 (K % 16 == 0 for M <= 4).
bool use_i8w(const void* a, const void* b, int M, int K, int N, bool transpose_b) {
    if (!transpose_b || M > kMaxFusedM || !aligned16(a) || !aligned16(b)) return false;
    return K % kChunk == 0 || (M <= 4 && K % 16 == 0);
}

// Device address of `scratch` on device `dev`, looked up with that device
// current on first use and kept per device (each device holds its own copy of
// the array at its own address).
constexpr int kMaxDevices = 64;
std::atomic<float*> g_scratch[kMaxDevices];

int scratch_ptr(int dev, float** out) {
    NG_REQUIRE(dev >= 0 && dev < kMaxDevices, "ng_gemm_int8_noalloc: device %d out of range", dev);
    float* p = g_scratch[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        void* addr = nullptr;
        NG_HIP_CHECK(hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)));
        NG_REQUIRE(addr != nullptr, "ng_gemm_int8_noalloc: no device address for the scratch array");
        p = static_cast<float*>(addr);
        g_scratch[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return 0;
}

}  // namespace

int gemm_scratch_init(int dev) {
    float* p = nullptr;
    return scratch_ptr(dev, &p);
}

void gemm_release() {
    std::lock_guard<std::mutex> lock(g_mu);
    for (auto& kv : g_plans) {
        Plan& p = kv.second;
        hipblasLtMatrixLayoutDestroy(p.lw);
        hipblasLtMatrixLayoutDestroy(p.lx);
        hipblasLtMatrixLayoutDestroy(p.ly);
        hipblasLtMatmulDescDestroy(p.desc);
    }
    g_plans.clear();
    g_lt_refused.clear();
    for (auto& kv : g_buffers) {
        for (void* b : {kv.second.ws, kv.second.deq, kv.second.part})
            if (b != nullptr) (void)hipFree(b);
    }
    g_buffers.clear();
    for (void* b : g_retired) (void)hipFree(b);
    g_retired.clear();
    for (auto& kv : g_handles) hipblasLtDestroy(kv.second);
    g_handles.clear();
    // A device reset (cuda_shutdown) releases the module's device globals:
    // look the scratch array up again after the next initialisation.
    for (auto& p : g_scratch) p.store(nullptr, std::memory_order_release);
}

}  // namespace ng

using namespace ng;

extern "C" int cuda_gemm_fp16(void* c, const void* a, const void* b, int M, int K, int N, bool transpose_a,
                              bool transpose_b) {
    NG_REQUIRE(c && a && b, "cuda_gemm_fp16: null pointer");
    NG_REQUIRE(M > 0 && K > 0 && N > 0, "cuda_gemm_fp16: M=%d K=%d N=%d must be > 0", M, K, N);
    return gemm_lt(c, a, b, nullptr, nullptr, M, K, N, transpose_a, transpose_b);
}

extern "C" int cuda_gemm_int8(void* c, const void* a, const void* b, const void* scale, int M, int K, int N,
                              bool transpose_b) {
    NG_REQUIRE(c && a && b && scale, "cuda_gemm_int8: null pointer");
    NG_REQUIRE(M > 0 && K > 0 && N > 0, "cuda_gemm_int8: M=%d K=%d N=%d must be > 0", M, K, N);
    if (use_i8w(a, b, M, K, N, transpose_b)) return gemm_i8w(c, a, b, scale, M, K, N);
    if (use_prefill(a, b, M, K, N, transpose_b)) {
        if (M >= kLtMinM) {
            const int r = gemm_lt_rows(c, a, b, scale, M, K, N);
            if (r <= 0) return r;
        }
        return gemm_prefill(c, a, b, scale, M, K, N);
    }
    return gemm_lt(c, a, nullptr, b, scale, M, K, N, false, transpose_b);
}

// The fused paths of cuda_gemm_int8 with no allocation: their only buffer,
// the split-K partial sums, lives in this library's fixed `scratch` array of
// the current device. Same kernels, same launch shapes and so the same bits as
// cuda_gemm_int8 below kLtMinM rows of A; from kLtMinM rows on it keeps the
// fused prefill kernel, where cuda_gemm_int8 runs the dequantize + hipBLASLt
// composition. Every call on a device shares that device's
// array: calls that overlap on one GPU (other streams, other host threads)
// race on it. The kernels write every partial sum before the reduction
// reads it, so nothing needs clearing between calls.
extern "C" int ng_gemm_int8_noalloc(void* c, const void* a, const void* b, const void* scale, int M, int K, int N,
                                    bool transpose_b) {
    NG_REQUIRE(c && a && b && scale, "ng_gemm_int8_noalloc: null pointer");
    NG_REQUIRE(M > 0 && K > 0 && N > 0, "ng_gemm_int8_noalloc: M=%d K=%d N=%d must be > 0", M, K, N);
    const bool stream_path = use_i8w(a, b, M, K, N, transpose_b);
    NG_REQUIRE(stream_path || use_prefill(a, b, M, K, N, transpose_b),
               "ng_gemm_int8_noalloc: M=%d K=%d N=%d transpose_b=%d is outside the paths that run without "
               "allocating (transpose_b, K %% 16 == 0 (K %% 64 == 0 for 4 < M <= %d), 16-byte aligned A and B); "
               "call cuda_gemm_int8 instead", M, K, N, static_cast<int>(transpose_b), kMaxFusedM);
    int dev = 0;
    NG_HIP_CHECK(hipGetDevice(&dev));
    float* part = nullptr;
    if (scratch_ptr(dev, &part) != 0) return -1;
    if (stream_path) return gemm_i8w(c, a, b, scale, M, K, N, part, kNoAllocScratchBytes);
    return gemm_prefill(c, a, b, scale, M, K, N, part, kNoAllocScratchBytes);
}

// The split kernel's shared form: slices and blocks as launch_split.
template <int MT, int W, int G>
int launch_split_shared(int count, void* const* c, const uint16_t* a, const void* const* b,
                        const void* const* scales, const int* n, int M, int K,
                        const SwigluArgs* sw = nullptr) {
    SharedPlan pl{};
    for (int i = 0; i < count; ++i) {
        pl.tn[i] = (n[i] + 16 * W - 1) / (16 * W);
        split_slices(pl.tn[i], G, K, pl.S[i], pl.cps[i]);
        pl.blocks[i] = static_cast<long long>(pl.tn[i]) * pl.S[i];
    }
    return run_shared_split(count, c, b, scales, n, M, K, pl,
                            [&](const SharedSet& set, const SplitSet& sp, unsigned blocks, hipStream_t st) {
                                gemm_i8w_split_shared_kernel<MT, W, G>
                                    <<<dim3(blocks), dim3(G * W * kWave), 0, st>>>(set, sp, a, M, K);
                            }, sw);
}

// One group of products that take the same launch shape `path` (see
// shared_path), in one launch of that kernel's shared form; shapes without a
// shared form, and groups of one, are one cuda_gemm_int8 call per product.
int shared_group(int path, int count, void* const* c, const void* a, const void* const* b,
                 const void* const* scales, const int* n, int M, int K) {
    const auto* ap = static_cast<const uint16_t*>(a);
    if (count > 1) {
        switch (path) {
            case 10 + kSplit141: return launch_split_shared<1, 4, 1>(count, c, ap, b, scales, n, M, K);
            case 10 + kSplit241: return launch_split_shared<2, 4, 1>(count, c, ap, b, scales, n, M, K);
            case 10 + kSplit142: return launch_split_shared<1, 4, 2>(count, c, ap, b, scales, n, M, K);
            case 10 + kSplit242: return launch_split_shared<2, 4, 2>(count, c, ap, b, scales, n, M, K);
            case kPathRing2:
            case kPathRing4: return gemm_ring(count, c, ap, b, scales, n, M, K);
            case kPathPrefill: return gemm_tiles(count, c, ap, b, scales, n, M, K);
            default: break;
        }
    }
    if (count == 1 || path <= 0 || path >= 10) {
        for (int i = 0; i < count; ++i) {
            const int r = cuda_gemm_int8(c[i], a, b[i], scales[i], M, K, n[i], true);
            if (r != 0) return r;
        }
        return 0;
    }
    const int R = path == 3 ? 4 : path == 4 ? 16 : 8;  // rows of B per block
    SharedSet set{};
    long long blocks = 0;
    for (int i = 0; i < kMaxShared; ++i) {
        const int j = i < count ? i : 0;  // unused slots repeat product 0 and are never selected
        set.c[i] = static_cast<uint16_t*>(c[j]);
        set.b[i] = static_cast<const int8_t*>(b[j]);
        set.scale[i] = static_cast<const float*>(scales[j]);
        set.n[i] = n[j];
        set.first[i] = i < count ? static_cast<int>(blocks) : INT_MAX;
        if (i < count) blocks += (n[i] + R - 1) / R;
        NG_REQUIRE(blocks < (1ll << 31), "ng_gemm_int8_shared_a: too many rows of B");
    }
    const int nb = static_cast<int>(blocks);
    switch (path) {
        case 1: return launch_gemv_shared<1, 8>(set, nb, ap, M, K);
        case 2: return launch_gemv_shared<2, 8>(set, nb, ap, M, K);
        case 3: return launch_gemv_shared<4, 4>(set, nb, ap, M, K);
        default:
            gemm_i8w_shared_kernel<1, 1, 8, 4><<<dim3(static_cast<unsigned>(nb)), dim3(8 * kWave), 0, stream()>>>(
                set, ap, M, K);
            NG_CHECK_LAUNCH("ng_gemm_int8_shared_a");
            return 0;
    }
}

// Products that share A (the engine's q/k/v and gate/up projections): they
// are grouped by the launch shape gemm_i8w would take for each, and each group
// runs in one launch of that kernel's shared form (plus one launch of the
// reduction where K slices have blocks of their own). Up to 32 rows each
// product's blocks are exactly its own launch's; above, the tile may be another
// (no bit depends on it). Products that take no kernel of the library's are one
// cuda_gemm_int8 call each, and so are those of a set whose partial sums have no
// room while a graph is captured. Either way the results are cuda_gemm_int8's,
// bit for bit.
extern "C" int ng_gemm_int8_shared_a(int count, void* const* c, const void* a, const void* const* b,
                                     const void* const* scales, const int* n, int M, int K) {
    NG_REQUIRE(c && a && b && scales && n, "ng_gemm_int8_shared_a: null pointer");
    NG_REQUIRE(count >= 1 && count <= kMaxShared, "ng_gemm_int8_shared_a: count=%d must be in [1, %d]", count,
               kMaxShared);
    NG_REQUIRE(M > 0 && K > 0, "ng_gemm_int8_shared_a: M=%d K=%d must be > 0", M, K);
    int path[kMaxShared];
    for (int i = 0; i < count; ++i) {
        NG_REQUIRE(c[i] && b[i] && scales[i], "ng_gemm_int8_shared_a: null pointer in product %d", i);
        NG_REQUIRE(n[i] > 0, "ng_gemm_int8_shared_a: n[%d]=%d must be > 0", i, n[i]);
        // cuda_gemm_int8's fused prefill kernel runs below kLtMinM rows of A
        path[i] = use_i8w(a, b[i], M, K, n[i], true) ? shared_path(M, K, n[i])
                  : M < kLtMinM && use_prefill(a, b[i], M, K, n[i], true) ? kPathPrefill
                                                                          : 0;
    }
    bool done[kMaxShared] = {};
    for (int i = 0; i < count; ++i) {
        if (done[i]) continue;
        void* gc[kMaxShared];
        const void* gb[kMaxShared];
        const void* gs[kMaxShared];
        int gn[kMaxShared], g = 0;
        for (int j = i; j < count; ++j) {
            if (done[j] || path[j] != path[i] || (path[i] <= 0 && j != i)) continue;
            gc[g] = c[j];
            gb[g] = b[j];
            gs[g] = scales[j];
            gn[g] = n[j];
            ++g;
            done[j] = true;
        }
        const int r = shared_group(path[i], g, gc, a, gb, gs, gn, M, K);
        if (r != 0) return r;
    }
    return 0;
}

// [p, p + pn) and [q, q + qn) share a byte.
static bool overlaps(const void* p, size_t pn, const void* q, size_t qn) {
    const auto a = reinterpret_cast<uintptr_t>(p), b = reinterpret_cast<uintptr_t>(q);
    return a < b + qn && b < a + pn;
}

// RMSNorm (ADD: residual add + RMSNorm) of A, then the products that share
// the normalised A: one launch of gemv_i8w_norm_shared_kernel when every
// product takes the same GEMV shape of one or two rows, K <= 8192, the launch
// has at most kNormSharedMaxBlocks blocks and no output overlaps an input (the kernel's
// blocks read the inputs while the first one stores); otherwise the norm
// entry point followed by ng_gemm_int8_shared_a.
// The same bits either way. With rs, RoPE (ng_rope_qk_with_theta, style 0)
// follows on products 0 and 1 in place; the fused launch then also needs D a
// multiple of 8 (four rotation pairs per block of 8 rows of B), the three
// outputs apart from each other and the positions apart from every output.
struct RopeSpec {
    const int* pos;
    int nq, nkv, D;
    float theta;
};

template <bool ADD>
static int norm_shared(const char* name, int count, void* normed, void* res_out, void* const* c, const void* x,
                       const void* res, const void* w, float eps, const void* const* b, const void* const* scales,
                       const int* n, int M, int K, const RopeSpec* rs = nullptr) {
    NG_REQUIRE(normed && x && w && c && b && scales && n && (!ADD || (res && res_out)), "%s: null pointer", name);
    NG_REQUIRE(count >= 1 && count <= kMaxShared, "%s: count=%d must be in [1, %d]", name, count, kMaxShared);
    NG_REQUIRE(M > 0 && K > 0, "%s: M=%d K=%d must be > 0", name, M, K);
    const size_t rows = static_cast<size_t>(M) * K * 2;
    int path = -1;
    const size_t wb = static_cast<size_t>(K) * 2;
    // Nothing the blocks read may share a byte with what the first block
    // writes (normed, residual_out) or what any block writes (c).
    const auto clear_of_writes = [&](const void* p, size_t pn) {
        return !overlaps(p, pn, normed, rows) && (!ADD || !overlaps(p, pn, res_out, rows));
    };
    bool apart = clear_of_writes(x, rows) && clear_of_writes(w, wb) &&
                 (!ADD || (clear_of_writes(res, rows) && !overlaps(res_out, rows, normed, rows)));
    for (int i = 0; i < count; ++i) {
        NG_REQUIRE(c[i] && b[i] && scales[i], "%s: null pointer in product %d", name, i);
        NG_REQUIRE(n[i] > 0, "%s: n[%d]=%d must be > 0", name, i, n[i]);
        const int pi = use_i8w(normed, b[i], M, K, n[i], true) ? gemv_shape(M, K, n[i]) : 0;
        path = (path == -1 || path == pi) ? pi : 0;
        const size_t cb = static_cast<size_t>(M) * n[i] * 2;
        apart = apart && clear_of_writes(b[i], static_cast<size_t>(n[i]) * K) &&
                clear_of_writes(scales[i], static_cast<size_t>(n[i]) * 4) && clear_of_writes(c[i], cb) &&
                !overlaps(c[i], cb, x, rows) && !overlaps(c[i], cb, w, wb) && (!ADD || !overlaps(c[i], cb, res, rows));
    }
    if (rs) {
        const size_t pb = static_cast<size_t>(M) * 4;
        apart = apart && !overlaps(rs->pos, pb, normed, rows) && (!ADD || !overlaps(rs->pos, pb, res_out, rows));
        for (int i = 0; i < count; ++i) {
            const size_t cb = static_cast<size_t>(M) * n[i] * 2;
            apart = apart && !overlaps(rs->pos, pb, c[i], cb);
            for (int j = i + 1; j < count; ++j) apart = apart && !overlaps(c[i], cb, c[j], static_cast<size_t>(M) * n[j] * 2);
        }
    }
    // GEMV blocks of the fused launch (rows of B per block as the GEMV kernel's).
    const int R = 8;
    long long blocks = 0;
    for (int i = 0; i < count; ++i) blocks += (n[i] + R - 1) / R;
    const bool fused = (path == 1 || path == 2) && apart && K <= kNormSharedMaxK && blocks <= kNormSharedMaxBlocks &&
                       aligned16(x) && aligned16(w) && aligned16(normed) &&
                       (!ADD || (aligned16(res) && aligned16(res_out))) &&
                       (!rs || (rs->D % 8 == 0 && rs->D <= 2 * kRopeEpiMaxHalf));
    if (!fused) {
        int r = ADD ? cuda_add_rmsnorm(normed, res_out, x, res, w, M, K, eps) : cuda_rmsnorm(normed, x, w, M, K, eps);
        if (r == 0) r = ng_gemm_int8_shared_a(count, c, normed, b, scales, n, M, K);
        if (r == 0 && rs)
            r = ng_rope_qk_with_theta(c[0], c[0], c[1], c[1], rs->pos, 1, M, rs->nq, rs->nkv, rs->D, 0, rs->theta);
        return r;
    }
    SharedSet set{};
    int first = 0;
    for (int i = 0; i < kMaxShared; ++i) {
        const int j = i < count ? i : 0;  // unused slots repeat product 0 and are never selected
        set.c[i] = static_cast<uint16_t*>(c[j]);
        set.b[i] = static_cast<const int8_t*>(b[j]);
        set.scale[i] = static_cast<const float*>(scales[j]);
        set.n[i] = n[j];
        set.first[i] = i < count ? first : INT_MAX;
        if (i < count) first += (n[i] + R - 1) / R;
    }
    const NormArgs na{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(res), static_cast<const uint16_t*>(w),
                      static_cast<uint16_t*>(normed), static_cast<uint16_t*>(res_out), eps};
    if constexpr (!ADD) {
        if (rs) {
            RopeEpi re{};
            re.pos = rs->pos;
            re.D = rs->D;
            re.half = rs->D / 2;
            re.bph = rs->D / 8;
            fill_inv_freq(rs->theta, rs->D, re.inv_freq);
            const dim3 grid(static_cast<unsigned>(first)), block(kGvWaves * kWave);
            const bool one = K <= kGvWaves * kGvSeg;
            if (path == 1) {
                if (one) gemv_i8w_norm_rope_shared_kernel<1, 1><<<grid, block, 0, stream()>>>(set, na, re, M, K);
                else gemv_i8w_norm_rope_shared_kernel<1, 2><<<grid, block, 0, stream()>>>(set, na, re, M, K);
            } else {
                if (one) gemv_i8w_norm_rope_shared_kernel<2, 1><<<grid, block, 0, stream()>>>(set, na, re, M, K);
                else gemv_i8w_norm_rope_shared_kernel<2, 2><<<grid, block, 0, stream()>>>(set, na, re, M, K);
            }
            NG_CHECK_LAUNCH(name);
            return 0;
        }
    }
    if (path == 1) return launch_gemv_norm_shared<1, 8, ADD>(set, first, na, M, K);
    return launch_gemv_norm_shared<2, 8, ADD>(set, first, na, M, K);
}

extern "C" int ng_rmsnorm_gemm_int8_shared_a(int count, void* normed, void* const* c, const void* x,
                                             const void* norm_weight, float eps, const void* const* b,
                                             const void* const* scales, const int* n, int M, int K) {
    return norm_shared<false>("ng_rmsnorm_gemm_int8_shared_a", count, normed, nullptr, c, x, nullptr, norm_weight, eps,
                              b, scales, n, M, K);
}

extern "C" int ng_add_rmsnorm_gemm_int8_shared_a(int count, void* normed, void* residual_out, void* const* c,
                                                 const void* x, const void* residual_in, const void* norm_weight,
                                                 float eps, const void* const* b, const void* const* scales,
                                                 const int* n, int M, int K) {
    return norm_shared<true>("ng_add_rmsnorm_gemm_int8_shared_a", count, normed, residual_out, c, x, residual_in,
                             norm_weight, eps, b, scales, n, M, K);
}

extern "C" int ng_rmsnorm_qkv_rope_int8(void* normed, void* q, void* k, void* v, const void* x,
                                        const void* norm_weight, float eps, const void* const* b,
                                        const void* const* scales, const int* positions, int M, int hidden,
                                        int num_q_heads, int num_kv_heads, int head_dim, float rope_theta) {
    const char* name = "ng_rmsnorm_qkv_rope_int8";
    NG_REQUIRE(q && k && v && positions && b && scales, "%s: null pointer", name);
    NG_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && head_dim > 0 && head_dim % 2 == 0 && head_dim <= 256,
               "%s: num_q_heads=%d num_kv_heads=%d head_dim=%d (even, at most 256)", name, num_q_heads, num_kv_heads,
               head_dim);
    NG_REQUIRE(static_cast<long long>(num_q_heads) * head_dim < (1ll << 31) &&
                   static_cast<long long>(num_kv_heads) * head_dim < (1ll << 31),
               "%s: too many rows of B", name);
    void* c[3] = {q, k, v};
    const int n[3] = {num_q_heads * head_dim, num_kv_heads * head_dim, num_kv_heads * head_dim};
    const RopeSpec rs{positions, num_q_heads, num_kv_heads, head_dim, rope_theta};
    return norm_shared<false>(name, 3, normed, nullptr, c, x, nullptr, norm_weight, eps, b, scales, n, M, hidden, &rs);
}

// The split kernel's SwiGLU form: the launch shape <MT, W, G> that
// split_config gives each of gate and up, when it takes one K slice (the
// wide two-group shapes); 1 when it does not, so that the caller runs the
// two calls.
template <int MT, int W, int G>
int launch_split_swiglu(const SwigluArgs& sa, const uint16_t* a, int M, int N, int K) {
    const int tn = (N + 16 * W - 1) / (16 * W);  // tiles of one product's own launch
    int S = 0, cps = 0;
    split_slices(tn, G, K, S, cps);
    if (S != 1) return 1;
    const unsigned blocks = static_cast<unsigned>((N + 8 * W - 1) / (8 * W));
    gemm_i8w_split_swiglu_kernel<MT, W, G><<<dim3(blocks), dim3(G * W * kWave), 0, stream()>>>(sa, a, M, N, K, cps);
    NG_CHECK_LAUNCH("ng_gemm_int8_silu_mul");
    return 0;
}

// gate/up with several K slices on a one-group split shape: the shared launch
// (partial sums only) and split_reduce_swiglu_kernel; 1 for other shapes.
static int swiglu_sliced(const SwigluArgs& sa, const uint16_t* a, int M, int K, int N) {
    void* c[2] = {sa.gate, sa.up};
    const void* b[2] = {sa.bg, sa.bu};
    const void* sc[2] = {sa.sg, sa.su};
    const int n[2] = {N, N};
    switch (shared_path(M, K, N)) {
        case 10 + kSplit141: return launch_split_shared<1, 4, 1>(2, c, a, b, sc, n, M, K, &sa);
        case 10 + kSplit241: return launch_split_shared<2, 4, 1>(2, c, a, b, sc, n, M, K, &sa);
        default: return 1;
    }
}

static int swiglu_split(const SwigluArgs& sa, const uint16_t* a, int M, int K, int N) {
    switch (split_config(M, K, N)) {
        case kSplit242: return launch_split_swiglu<2, 4, 2>(sa, a, M, N, K);
        case kSplit142: return launch_split_swiglu<1, 4, 2>(sa, a, M, N, K);
        default: return 1;
    }
}

// gate/up (cuda_gemm_int8 on one A, as ng_gemm_int8_shared_a) and SwiGLU
// (cuda_silu_mul), when no output overlaps an input or another output (out
// may be gate or up exactly): one launch of gemv_i8w_swiglu_kernel when both
// products take the GEMV kernel; one of the SwiGLU form of the split kernel (up
// to 32 rows), the ring kernel (33 to 128) or the tile kernel (below kLtMinM) when
// they take that kernel with one K slice; the kernel's shared launch and
// split_reduce_swiglu_kernel when they have several; otherwise the two calls.
// The same bits either way.
extern "C" int ng_gemm_int8_silu_mul(void* out, void* gate, void* up, const void* a, const void* b_gate,
                                     const void* scale_gate, const void* b_up, const void* scale_up, int M, int K,
                                     int N) {
    NG_REQUIRE(out && gate && up && a && b_gate && scale_gate && b_up && scale_up, "ng_gemm_int8_silu_mul: null pointer");
    NG_REQUIRE(M > 0 && K > 0 && N > 0, "ng_gemm_int8_silu_mul: M=%d K=%d N=%d must be > 0", M, K, N);
    const size_t cb = static_cast<size_t>(M) * N * 2, ab = static_cast<size_t>(M) * K * 2;
    const size_t bb = static_cast<size_t>(N) * K, sb = static_cast<size_t>(N) * 4;
    const int path = use_i8w(a, b_gate, M, K, N, true) && use_i8w(a, b_up, M, K, N, true) ? gemv_shape(M, K, N) : 0;
    bool apart = !overlaps(gate, cb, up, cb) && (out == gate || out == up || (!overlaps(out, cb, gate, cb) &&
                                                                              !overlaps(out, cb, up, cb)));
    for (const void* o : {out, gate, up})
        apart = apart && !overlaps(o, cb, a, ab) && !overlaps(o, cb, b_gate, bb) && !overlaps(o, cb, b_up, bb) &&
                !overlaps(o, cb, scale_gate, sb) && !overlaps(o, cb, scale_up, sb);
    const SwigluArgs sa{static_cast<uint16_t*>(out), static_cast<uint16_t*>(gate), static_cast<uint16_t*>(up),
                        static_cast<const int8_t*>(b_gate), static_cast<const int8_t*>(b_up),
                        static_cast<const float*>(scale_gate), static_cast<const float*>(scale_up)};
    if (path < 1 && apart && use_i8w(a, b_gate, M, K, N, true) && use_i8w(a, b_up, M, K, N, true)) {
        if (M >= kRingMinM) {
            void* c[2] = {gate, up};
            const void* b[2] = {b_gate, b_up};
            const void* sc[2] = {scale_gate, scale_up};
            const int n[2] = {N, N};
            const int r = gemm_ring(2, c, a, b, sc, n, M, K, nullptr, 0, nullptr, &sa);
            if (r <= 0) return r;
        } else {
            int r = swiglu_split(sa, static_cast<const uint16_t*>(a), M, K, N);
            if (r == 1) r = swiglu_sliced(sa, static_cast<const uint16_t*>(a), M, K, N);
            if (r <= 0) return r;
        }
    } else if (path < 1 && apart && M < kLtMinM && use_prefill(a, b_gate, M, K, N, true) &&
               use_prefill(a, b_up, M, K, N, true) && !use_i8w(a, b_gate, M, K, N, true)) {
        void* c[2] = {gate, up};
        const void* b[2] = {b_gate, b_up};
        const void* sc[2] = {scale_gate, scale_up};
        const int n[2] = {N, N};
        const int r = gemm_tiles(2, c, a, b, sc, n, M, K, nullptr, 0, nullptr, &sa);
        if (r <= 0) return r;
    }
    if (path < 1 || !apart) {
        void* c[2] = {gate, up};
        const void* b[2] = {b_gate, b_up};
        const void* sc[2] = {scale_gate, scale_up};
        const int n[2] = {N, N};
        const int r = ng_gemm_int8_shared_a(2, c, a, b, sc, n, M, K);
        if (r != 0) return r;
        return cuda_silu_mul(out, gate, up, static_cast<size_t>(M) * N);
    }
    const auto ap = static_cast<const uint16_t*>(a);
    const dim3 block(kGvWaves * kWave);
    if (path == 3) {
        gemv_i8w_swiglu_kernel<4, 4><<<dim3(static_cast<unsigned>((N + 3) / 4)), block, 0, stream()>>>(sa, ap, M, N, K);
    } else if (path == 2) {
        gemv_i8w_swiglu_kernel<2, 8><<<dim3(static_cast<unsigned>((N + 7) / 8)), block, 0, stream()>>>(sa, ap, M, N, K);
    } else {
        gemv_i8w_swiglu_kernel<1, 8><<<dim3(static_cast<unsigned>((N + 7) / 8)), block, 0, stream()>>>(sa, ap, M, N, K);
    }
    NG_CHECK_LAUNCH("ng_gemm_int8_silu_mul");
    return 0;
}

// A product (cuda_gemm_int8 with transpose_b) and the residual add after it
// (cuda_add(out, c, residual)): when no output overlaps an input or the other
// output (out may be c or the residual exactly), one launch of
// gemv_i8w_add_kernel on the GEMV kernel's shapes, and on cuda_gemm_int8's
// other fused paths (the weight-streaming kernels up to 128 rows, the prefill
// kernel below kLtMinM) the add in the reduction of the K slices, or with one K
// slice in the epilogue of the ring and the tile kernel (up to 32 rows after the
// product as cuda_add); otherwise the two calls. The same bits either way.
extern "C" int ng_gemm_int8_add(void* out, void* c, const void* a, const void* b, const void* scale,
                                const void* residual, int M, int K, int N) {
    NG_REQUIRE(out && c && a && b && scale && residual, "ng_gemm_int8_add: null pointer");
    NG_REQUIRE(M > 0 && K > 0 && N > 0, "ng_gemm_int8_add: M=%d K=%d N=%d must be > 0", M, K, N);
    const size_t cb = static_cast<size_t>(M) * N * 2, ab = static_cast<size_t>(M) * K * 2;
    const size_t bb = static_cast<size_t>(N) * K, sb = static_cast<size_t>(N) * 4;
    const int path = use_i8w(a, b, M, K, N, true) ? gemv_shape(M, K, N) : 0;
    bool apart = !overlaps(c, cb, residual, cb) &&
                 (out == c || out == residual || (!overlaps(out, cb, c, cb) && !overlaps(out, cb, residual, cb)));
    for (const void* o : {out, c})
        apart = apart && !overlaps(o, cb, a, ab) && !overlaps(o, cb, b, bb) && !overlaps(o, cb, scale, sb);
    if (path < 1 || !apart) {
        // cuda_gemm_int8's own fused paths (the weight-streaming kernels up to
        // 128 rows of A, the prefill kernel below kLtMinM): the add in the
        // split-K reduction or the epilogue.
        const ResEpi ep{static_cast<uint16_t*>(out), static_cast<const uint16_t*>(residual)};
        if (apart && use_i8w(a, b, M, K, N, true)) return gemm_i8w(c, a, b, scale, M, K, N, nullptr, 0, &ep);
        if (apart && M < kLtMinM && use_prefill(a, b, M, K, N, true))
            return gemm_prefill(c, a, b, scale, M, K, N, nullptr, 0, &ep);
        const int r = cuda_gemm_int8(c, a, b, scale, M, K, N, true);
        if (r != 0) return r;
        return cuda_add(out, c, residual, static_cast<size_t>(M) * N);
    }
    const auto o16 = static_cast<uint16_t*>(out);
    const auto c16 = static_cast<uint16_t*>(c);
    const auto r16 = static_cast<const uint16_t*>(residual);
    const auto ap = static_cast<const uint16_t*>(a);
    const auto bp = static_cast<const int8_t*>(b);
    const auto sp = static_cast<const float*>(scale);
    const dim3 block(kGvWaves * kWave);
    if (path == 3) {
        gemv_i8w_add_kernel<4, 4><<<dim3(static_cast<unsigned>((N + 3) / 4)), block, 0, stream()>>>(
            o16, c16, r16, ap, bp, sp, M, N, K);
    } else if (path == 2) {
        gemv_i8w_add_kernel<2, 8><<<dim3(static_cast<unsigned>((N + 7) / 8)), block, 0, stream()>>>(
            o16, c16, r16, ap, bp, sp, M, N, K);
    } else {
        gemv_i8w_add_kernel<1, 8><<<dim3(static_cast<unsigned>((N + 7) / 8)), block, 0, stream()>>>(
            o16, c16, r16, ap, bp, sp, M, N, K);
    }
    NG_CHECK_LAUNCH("ng_gemm_int8_add");
    return 0;
}
