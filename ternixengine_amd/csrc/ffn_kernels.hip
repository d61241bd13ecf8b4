// ffn_kernels.hip -- the float steps around the ternary matmuls of a BitNet-style feed-forward block
// on gfx950: RMSNorm (optionally fused with the int8 activation quantisation that feeds the
// up-projection) and SwiGLU.
//
// Semantics follow the reference's CPU routines (src/simd_math.cpp): RMSNorm
//   out[i] = in[i] * inv * w[i],  inv = 1 / sqrt(sum(in^2) / size + eps)          (:7-12, :14-38)
// and SwiGLU over interleaved pairs out[i] = silu(in[2i]) * in[2i+1],
//   silu(g) = g / (1 + exp(-g))                                                     (:40-46).
// The sum of squares is a parallel tree here (the reference sums sequentially, or in 8 AVX2 lanes),
// so results agree to float rounding, not bit for bit -- the reference's own test tolerance between
// its scalar and AVX2 versions is 1e-4 relative (tests/test_simd_math.cpp:17-27).
// One workgroup per row for RMSNorm, the row in registers; a flat grid for SwiGLU, an HBM stream.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "row_stats.h"
#include "ternary_kernels.h"

namespace ternix_hip {
namespace {

__global__ __launch_bounds__(256) void rmsnorm_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                      float eps, float* __restrict__ out, int8_t* __restrict__ Q,
                                                      float* __restrict__ row_scale, int K) {
    __shared__ float red[4];
    const int m = blockIdx.x;
    const float* x = X + (size_t)m * (size_t)K;
    const float inv = row_rms_inv(x, K, eps, red);
    if (Q == nullptr) {
        float* o = out + (size_t)m * (size_t)K;
        for (int k = threadIdx.x; k < K; k += 256) o[k] = row_value(x, W, inv, k);
        return;
    }
    // Fused quantisation of the normalised row (the rule of quantize_rows_kernel).
    const float a = fmaxf(row_absmax(x, W, inv, K, red), 1e-5f);
    const float s = 127.0f / a;
    if (threadIdx.x == 0) row_scale[m] = a / 127.0f;
    int8_t* q = Q + (size_t)m * (size_t)K;
    for (int k = threadIdx.x; k < K; k += 256) q[k] = (int8_t)quantize_value(row_value(x, W, inv, k), s);
}

// The same with the row held in registers, K <= 256 * NV.  What bounds a row is latency: the strided loops
// above wait for memory once per 256 elements in each of three passes over the row; here all of the
// row's loads (and the weights') are in flight at once and the row is read once.  Thread t holds elements t,
// t + 256, ... as those loops visit them, so every sum has the same order and the results the same bits.
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_reg_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                          float eps, float* __restrict__ out, int8_t* __restrict__ Q,
                                                          float* __restrict__ row_scale, int K) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x;
    const float* x = X + (size_t)m * (size_t)K;
    float v[NV], g[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int k = tid + 256 * u;
        v[u] = k < K ? x[k] : 0.0f;
        g[u] = k < K ? W[k] : 0.0f;
    }
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (256 * u < K) ss = fmaf(v[u], v[u], ss);  // elements past the row are zeros and add nothing
    const float inv = 1.0f / sqrtf(row_block_sum(ss, red) / (float)K + eps);
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (256 * u < K) v[u] = v[u] * inv * g[u];
    if (Q == nullptr) {
        float* o = out + (size_t)m * (size_t)K;
#pragma unroll
        for (int u = 0; u < NV; ++u)
            if (tid + 256 * u < K) o[tid + 256 * u] = v[u];
        return;
    }
    float amax = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (tid + 256 * u < K) amax = fmaxf(amax, fabsf(v[u]));
    const float a = fmaxf(row_block_max(amax, red), 1e-5f);
    const float s = 127.0f / a;
    if (tid == 0) row_scale[m] = a / 127.0f;
    int8_t* q = Q + (size_t)m * (size_t)K;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (tid + 256 * u < K) q[tid + 256 * u] = (int8_t)quantize_value(v[u], s);
}

__global__ __launch_bounds__(256) void swiglu_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                     size_t pairs) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pairs) return;
    const float g = in[2 * i], u = in[2 * i + 1];
    out[i] = (g / (1.0f + expf(-g))) * u;
}

}  // namespace

hipError_t launch_rmsnorm(const float* X, const float* W, float eps, float* out, int8_t* Q, float* row_scale, int M,
                          int K, hipStream_t st) {
    if (M == 0) return hipSuccess;
    const dim3 grid((unsigned)M), block(256);
    // Up to 16384 elements the row stays in registers (64 a lane, its weights 64 more).  On MI355X, warm, RMSNorm
    // + quantise, us before -> after: 1x2560 6.1 -> 3.2, 32x2560 6.5 -> 3.5, 64x11008 20.0 -> 8.7,
    // 1024x2560 7.5 -> 4.8, 2048x4096 18.1 -> 9.4, 2048x16384 74.5 -> 42.1.
#define TX_RMS(kern) hipLaunchKernelGGL(kern, grid, block, 0, st, X, W, eps, out, Q, row_scale, K)
    if (K <= 1024) TX_RMS(rmsnorm_reg_kernel<4>);
    else if (K <= 2048) TX_RMS(rmsnorm_reg_kernel<8>);
    else if (K <= 4096) TX_RMS(rmsnorm_reg_kernel<16>);
    else if (K <= 8192) TX_RMS(rmsnorm_reg_kernel<32>);
    else if (K <= 16384) TX_RMS(rmsnorm_reg_kernel<64>);
    else TX_RMS(rmsnorm_kernel);
#undef TX_RMS
    return hipGetLastError();
}

hipError_t launch_swiglu(const float* in, float* out, size_t pairs, hipStream_t st) {
    if (pairs == 0) return hipSuccess;
    hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, st, in, out, pairs);
    return hipGetLastError();
}

}  // namespace ternix_hip
