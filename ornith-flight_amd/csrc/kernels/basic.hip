// SPDX-License-Identifier: MIT
//
// fp32 element-wise and small dense kernels behind the gpu.h backend API.
// Compiled with -ffp-contract=off: every mul/add below rounds separately, in
// the order written, like the reference CPU backend (gpu.c:104-238).
#include "common.h"
#include "launch.h"

namespace {

__global__ void k_fill(float *p, float v, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

__global__ void k_silu(float *out, const float *x, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        float v = x[i];
        out[i] = v / (1.0f + expf(-v));
    }
}

__global__ void k_silu_mul(float *out, const float *g, const float *u, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        float v = g[i];
        out[i] = (v / (1.0f + expf(-v))) * u[i];
    }
}

__global__ void k_add(float *out, const float *a, const float *b, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] + b[i];
}

// Streaming read of n16 16-byte words (grid-stride, 8 loads in flight per
// thread), folded with xor into one word per thread so the loads are live.
__global__ void __launch_bounds__(256) k_stream_read(const uint4 *__restrict__ p, size_t n16,
                                                     uint32_t *__restrict__ out)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0;
    for (; i + 7 * stride < n16; i += 8 * stride) {
        uint4 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[i + j * stride];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc ^= v[j].x ^ v[j].y ^ v[j].z ^ v[j].w;
    }
    for (; i < n16; i += stride) {
        const uint4 v = p[i];
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = acc;
}

inline int blocks_for(size_t n, int bs) { return (int)((n + (size_t)bs - 1) / (size_t)bs); }

}  // namespace

// out: ORNK_STREAM_GRID * 256 words.
extern "C" int ornk_stream_read(const void *p, size_t bytes, uint32_t *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_stream_read, dim3(ORNK_STREAM_GRID), dim3(256), 0, s,
                       reinterpret_cast<const uint4 *>(p), bytes / 16, out);
    return hipGetLastError();
}

extern "C" int ornk_fill_f32(float *p, float v, size_t n, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    size_t nb = (n + 255) / 256;
    int grid = nb > 65536 ? 65536 : (int)nb;
    hipLaunchKernelGGL(k_fill, dim3(grid), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

extern "C" int ornk_silu(float *out, const float *x, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_silu, dim3(blocks_for((size_t)n, 256)), dim3(256), 0, s, out, x, n);
    return hipGetLastError();
}

extern "C" int ornk_silu_mul(float *out, const float *g, const float *u, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_silu_mul, dim3(blocks_for((size_t)n, 256)), dim3(256), 0, s, out, g, u, n);
    return hipGetLastError();
}

extern "C" int ornk_add(float *out, const float *a, const float *b, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_add, dim3(blocks_for((size_t)n, 256)), dim3(256), 0, s, out, a, b, n);
    return hipGetLastError();
}
