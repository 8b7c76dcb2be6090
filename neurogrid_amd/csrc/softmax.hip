// softmax.hip - row softmax over fp16 rows (ABI completeness; not on the
// per-layer path). y_i = RN_f16(exp(x_i - m) / sum_j exp(x_j - m)) with m the
// true row maximum. The reference kernel (gpu/cuda/kernels.cu:580-631) shifts
// by one thread's partial maximum instead; softmax is shift-invariant, so the
// results agree wherever the reference's exponentials do not overflow.
//
// Rows of up to 65536 elements in whole 16-byte vectors stay in registers: a
// block of 1, 4 or 16 waves per row, every vector requested before any is used,
// one exponential per element, the quotient by the correctly rounded reciprocal
// and one correction step (3 operations instead of about 10 for a division).
// Longer rows (whose exponentials do not fit) are read three times, by 1024
// threads in 16-byte vectors, all others element by element. Bound: few rows
// (sampling) leave one block per CU, whose exponentials and quotients take the
// time: 64 rows of 32000 take 8.2 us on MI355X back to back in a graph, against
// 63.5 us read three times by 256 threads per row.
#include "ng_common.hpp"

namespace ng {

constexpr int kSmThreads = 256;

// Sum and maximum over the block, in every thread; s holds a float per wave.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* s) {
    v = MAX ? wave_max_f32(v) : wave_sum_f32(v);
    const int nw = blockDim.x / kWave;
    if (nw == 1) return v;
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    v = s[0];
    for (int j = 1; j < nw; ++j) v = MAX ? fmaxf(v, s[j]) : v + s[j];
    __syncthreads();
    return v;
}

// v / s, correctly rounded for the normal quotients of this kernel, given inv = RN(1 / s).
__device__ __forceinline__ float quotient(float v, float s, float inv) {
    const float z = v * inv;
    return __builtin_fmaf(__builtin_fmaf(z, -s, v), inv, z);
}

// Vector i of a thread is vector threadIdx.x + i THREADS of the row.
template <int V, int THREADS>
__global__ __launch_bounds__(THREADS) void softmax_vec_kernel(uint16_t* out, const uint16_t* in, int cols) {
    __shared__ float s_red[THREADS / kWave];
    const size_t off = static_cast<size_t>(blockIdx.x) * cols;
    const int nv = cols / 8;
    u32x4 x[V];
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = ld16_stream(in + off + 8 * min(static_cast<int>(threadIdx.x) + i * THREADS, nv - 1));
    float m = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < V; ++i) {  // a vector past the row repeats its last one
        float f[8];
        unpack8<f16>(x[i], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, f[e]);
    }
    m = block_reduce<true>(m, s_red);
    float ex[V][8];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        if (static_cast<int>(threadIdx.x) + i * THREADS >= nv) continue;
        unpack8<f16>(x[i], ex[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ex[i][e] = expf(ex[i][e] - m);
            s += ex[i][e];
        }
    }
    s = block_reduce<false>(s, s_red);
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int k = static_cast<int>(threadIdx.x) + i * THREADS;
        if (k >= nv) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) ex[i][e] = quotient(ex[i][e], s, inv);
        st16_stream(out + off + 8 * k, pack8<f16>(ex[i]));
    }
}

__global__ __launch_bounds__(1024) void softmax_long_kernel(uint16_t* out, const uint16_t* in, int cols) {
    __shared__ float s_red[1024 / kWave];
    const size_t off = static_cast<size_t>(blockIdx.x) * cols;
    const int nv = cols / 8;
    float m = -__builtin_inff(), s = 0.0f, f[8];
#pragma unroll 4
    for (int k = threadIdx.x; k < nv; k += 1024) {
        unpack8<f16>(ld16(in + off + 8 * k), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, f[e]);
    }
    m = block_reduce<true>(m, s_red);
    for (int k = threadIdx.x; k < nv; k += 1024) {
        unpack8<f16>(ld16(in + off + 8 * k), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) s += expf(f[e] - m);
    }
    s = block_reduce<false>(s, s_red);
    const float inv = 1.0f / s;
    for (int k = threadIdx.x; k < nv; k += 1024) {
        unpack8<f16>(ld16(in + off + 8 * k), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = quotient(expf(f[e] - m), s, inv);
        st16_stream(out + off + 8 * k, pack8<f16>(f));
    }
}

__global__ __launch_bounds__(kSmThreads) void softmax_kernel(uint16_t* out, const uint16_t* in, int cols) {
    __shared__ float s_red[kSmThreads / kWave];
    const size_t off = static_cast<size_t>(blockIdx.x) * cols;
    const uint16_t* x = in + off;
    uint16_t* y = out + off;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;

    float m = -__builtin_inff();
    for (int i = threadIdx.x; i < cols; i += kSmThreads) m = fmaxf(m, to_f32<f16>(x[i]));
    m = wave_max_f32(m);
    if (lane == 0) s_red[wid] = m;
    __syncthreads();
    m = s_red[0];
    for (int j = 1; j < kSmThreads / kWave; ++j) m = fmaxf(m, s_red[j]);
    __syncthreads();

    float s = 0.0f;
    for (int i = threadIdx.x; i < cols; i += kSmThreads) s += expf(to_f32<f16>(x[i]) - m);
    s = wave_sum_f32(s);
    if (lane == 0) s_red[wid] = s;
    __syncthreads();
    s = 0.0f;
    for (int j = 0; j < kSmThreads / kWave; ++j) s += s_red[j];

    for (int i = threadIdx.x; i < cols; i += kSmThreads) y[i] = from_f32<f16>(expf(to_f32<f16>(x[i]) - m) / s);
}

}  // namespace ng

using namespace ng;

extern "C" int cuda_softmax(void* output, const void* input, int num_rows, int row_size) {
    NG_REQUIRE(output && input, "cuda_softmax: null pointer");
    NG_REQUIRE(num_rows > 0 && row_size > 0, "cuda_softmax: num_rows=%d row_size=%d must be > 0", num_rows,
               row_size);
    auto* y = static_cast<uint16_t*>(output);
    const auto* x = static_cast<const uint16_t*>(input);
    const dim3 grid(num_rows);
    // A launch takes fewer than 2^32 threads: from 2^22 rows on no 1024 to a row.
    const bool wide = num_rows < (1 << 22);
    if (row_size % 8 == 0 && aligned16(output) && aligned16(input) && (row_size <= 8192 || wide)) {
        // One wave for rows of up to 512 elements, four up to 8192, sixteen
        // above: a block of 16 waves pays for its barriers and for threads with
        // no vector (4096 rows of 2056: 11.2 us with 4 waves, 29.2 with 16; of
        // 8192: 22.3 and 36.4; 64 rows of 4096: 3.5 and 4.1).
        if (row_size <= 512) softmax_vec_kernel<1, 64><<<grid, dim3(64), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 2048) softmax_vec_kernel<1, 256><<<grid, dim3(256), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 4096) softmax_vec_kernel<2, 256><<<grid, dim3(256), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 8192) softmax_vec_kernel<4, 256><<<grid, dim3(256), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 16384) softmax_vec_kernel<2, 1024><<<grid, dim3(1024), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 32768) softmax_vec_kernel<4, 1024><<<grid, dim3(1024), 0, stream()>>>(y, x, row_size);
        else if (row_size <= 65536) softmax_vec_kernel<8, 1024><<<grid, dim3(1024), 0, stream()>>>(y, x, row_size);
        else softmax_long_kernel<<<grid, dim3(1024), 0, stream()>>>(y, x, row_size);
    } else {
        softmax_kernel<<<grid, dim3(kSmThreads), 0, stream()>>>(y, x, row_size);
    }
    NG_CHECK_LAUNCH("cuda_softmax");
    return 0;
}
