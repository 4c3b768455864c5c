// SPDX-License-Identifier: MIT
//
// The dense products and the rmsnorm of the gpu.h backend API and of the MoE
// forward.  Compiled with -ffp-contract=off: every mul/add below rounds
// separately, in the order written, like the reference CPU backend
// (gpu.c:104-156).  A code object of its own, loaded when one of them first
// runs, and not part of basic.hip's, which every context loads: the one-token
// forward moves by up to 0.5 us with what is loaded beside its kernels.
#include "common.h"
#include "launch.h"

namespace {

inline int blocks_for(size_t n, int bs) { return (int)((n + (size_t)bs - 1) / (size_t)bs); }

// gpu.c:104-115: C[i][j] = sum_k A[i][k] * B[k][j], a sequential fp32 sum
// from 0.0f with k ascending and separately rounded products, so results are
// bit-identical to the CPU backend.  A thread owns NC adjacent columns for MT
// rows; with RS = 2 the work group's upper two waves take the next MT rows of
// the lower two's columns, whose B values they then find in the CU's cache.
// A is staged in LDS in chunks of MM_KC columns (every lane reads the same
// words: broadcast).  The rows of A for the next 4 k's are read from LDS, and
// B's next MM_U loads issued, before the products of the current ones, so the
// multiply and add per product are what is left to wait for.  Rows past M are
// zero in LDS and never stored.
//
// What bounds it: HBM up to 4 rows (2.03 GB at K = 2048, N = 248,320: 325 us,
// 6.3 TB/s), the vector issue slots above (16 rows: 254 M wave instructions,
// 441 us).  Before, with one LDS read per product group right before its use,
// 16 rows took 530-630 us there, and 16 / 4 / 1 rows at N = 32,768 took 293 /
// 241 / 117 us; now 149 / 88 / 68.
constexpr int MM_KC = 256, MM_U = 8;

template <int NC>
struct MmVec;
template <>
struct MmVec<1> { typedef float T; };
template <>
struct MmVec<2> { typedef float T __attribute__((ext_vector_type(2))); };
template <>
struct MmVec<4> { typedef v4f T; };

template <int MT, int NC, int RS>
__global__ void __launch_bounds__(256) k_matmul(float *__restrict__ C, const float *__restrict__ A,
                                                  const float *__restrict__ B, int M, int N, int K)
{
    typedef typename MmVec<NC>::T bvec;
    constexpr int TC = 256 / RS;
    __shared__ __align__(16) float As[MT * RS][MM_KC + 4];
    const int j = (blockIdx.x * TC + (threadIdx.x % TC)) * NC;  // first column of this thread
    const int r0 = RS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TC) * MT : 0;
    const int ib = blockIdx.y * MT * RS;  // first row of the work group
    const bool live = j < N;  // NC > 1 only when N % NC == 0
    const bvec *b = reinterpret_cast<const bvec *>(B + (live ? j : 0));
    const size_t ldb = (size_t)N / NC;
    float acc[MT][NC];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[i][c] = 0.0f;
    auto at = [](const bvec &v, int c) -> float {
        if constexpr (NC == 1) return v;
        else return v[c];
    };
    bvec b0[MM_U], b1[MM_U];
    auto load_b = [&](bvec(&r)[MM_U], int k) {  // k past the last whole turn: re-read row 0, unused
        const bvec *p = b + (k + MM_U <= K ? (size_t)k * ldb : 0);
        const size_t st = k + MM_U <= K ? ldb : 0;
#pragma unroll
        for (int u = 0; u < MM_U; ++u) r[u] = p[u * st];
    };
    if (K > 0) load_b(b0, 0);  // K = 0: B may hold nothing
    for (int k0 = 0; k0 < K; k0 += MM_KC) {
        const int kc = K - k0 < MM_KC ? K - k0 : MM_KC;
        __syncthreads();  // the previous chunk is consumed
        for (int e = threadIdx.x; e < MT * RS * MM_KC; e += 256) {
            const int i = e / MM_KC, k = e - i * MM_KC;
            As[i][k] = (ib + i < M && k < kc) ? A[(size_t)(ib + i) * K + k0 + k] : 0.0f;
        }
        __syncthreads();
        v4f a0[MT], a1[MT];
        auto load_a = [&](v4f(&r)[MT], int k) {  // within the padded row, also past kc
#pragma unroll
            for (int i = 0; i < MT; ++i) r[i] = *reinterpret_cast<const v4f *>(&As[r0 + i][k]);
        };
        auto mac4 = [&](const v4f(&ar)[MT], const bvec *br) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int c = 0; c < NC; ++c) acc[i][c] += ar[i][u] * at(br[u], c);
        };
        auto turn = [&](bvec(&cur)[MM_U], bvec(&nxt)[MM_U], int k) {
            load_b(nxt, k0 + k + MM_U);
            load_a(a1, k + 4);
            __builtin_amdgcn_sched_barrier(0);
            mac4(a0, cur);
            __builtin_amdgcn_sched_barrier(0);
            load_a(a0, k + 8 < MM_KC ? k + 8 : 0);
            __builtin_amdgcn_sched_barrier(0);
            mac4(a1, cur + 4);
            __builtin_amdgcn_sched_barrier(0);
        };
        load_a(a0, 0);
        const int kw = kc - kc % MM_U;
        int k = 0;
        for (; k + 2 * MM_U <= kw; k += 2 * MM_U) {
            turn(b0, b1, k);
            turn(b1, b0, k + MM_U);
        }
        if (k < kw) {  // an odd turn, in the last chunk alone
            turn(b0, b1, k);
            k += MM_U;
        }
        for (; k < kc; ++k) {
            const bvec bk = b[(size_t)(k0 + k) * ldb];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[i][c] += As[r0 + i][k] * at(bk, c);
        }
    }
    if (!live) return;
#pragma unroll
    for (int i = 0; i < MT; ++i)
        if (ib + r0 + i < M)
#pragma unroll
            for (int c = 0; c < NC; ++c) C[(size_t)(ib + r0 + i) * N + j + c] = acc[i][c];
}

// gpu.c:144-156 per row: ss is the reference's sequential fp32 sum of the
// fp32 products x[i]*x[i], i ascending, then out = w * (x * inv_rms).  The
// products are formed by all threads into LDS (dim floats of dynamic shared
// memory); one lane then adds them in order (orn_lds_seq_sum32), so only the
// chain of adds is serial and the roundings are the reference's.
__global__ void __launch_bounds__(256) k_rmsnorm(float *out, const float *x, const float *w, int dim)
{
    extern __shared__ __align__(16) float s_p[];
    __shared__ float inv_s;
    const float *xr = x + (size_t)blockIdx.x * dim;
    float *orow = out + (size_t)blockIdx.x * dim;
    // Vector path (dim a multiple of 4, at most 16384): a thread's x and w
    // are loaded in one round trip, before the first product.
    const bool vec = (dim & 3) == 0 && dim <= 16 * 1024;
    const int n4 = dim >> 2;
    v4f xv[16], wv[16];
    if (vec) {
        const v4f *x4 = reinterpret_cast<const v4f *>(xr);
        const v4f *w4 = reinterpret_cast<const v4f *>(w);
        v4f *p4 = reinterpret_cast<v4f *>(s_p);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = (int)threadIdx.x + 256 * j;
            if (i < n4) {
                xv[j] = x4[i];
                wv[j] = w4[i];
            }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = (int)threadIdx.x + 256 * j;
            if (i < n4) p4[i] = xv[j] * xv[j];
        }
    } else {
        for (int i = threadIdx.x; i < dim; i += blockDim.x) {
            const float v = xr[i];
            s_p[i] = v * v;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nb = dim >> 5;
        float ss = orn_lds_seq_sum32(reinterpret_cast<const v4f *>(s_p), nb);
        for (int i = 32 * nb; i < dim; ++i) ss += s_p[i];
        inv_s = 1.0f / sqrtf(ss / (float)dim + 1e-6f);
    }
    __syncthreads();
    const float inv = inv_s;
    if (vec) {
        v4f *o4 = reinterpret_cast<v4f *>(orow);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int i = (int)threadIdx.x + 256 * j;
            if (i < n4) o4[i] = wv[j] * (xv[j] * inv);
        }
    } else {
        for (int i = threadIdx.x; i < dim; i += blockDim.x) orow[i] = w[i] * (xr[i] * inv);
    }
}

// The same for several rows per work group, so that the lanes of one wave run
// the rows' chains side by side: a row's chain of dim dependent adds (5.8 us
// at 2048) is what bounds it, and a work group per row keeps it for one lane.
// 2048 rows of 2048: 48 -> 19 us, 1500 rows 37 -> 17 (event spans around the
// launch, some 8 us of each their own).  dim % 32 == 0 and dim <= RN_MAXD, whose
// eight rows take 66 KB of LDS: two work groups per CU, of 4096 columns one.
constexpr int RN_MAXD = 2048, RN_R = 8;

__global__ void __launch_bounds__(256) k_rmsnorm_rows(float *__restrict__ out,
                                                      const float *__restrict__ x,
                                                      const float *__restrict__ w, int rows,
                                                      int dim)
{
    // 4 floats of padding: the rows' 16-byte reads fall on different banks
    __shared__ __align__(16) float s_p[RN_R][RN_MAXD + 4];
    __shared__ float s_inv[RN_R];
    const int r0 = blockIdx.x * RN_R, tid = threadIdx.x, n4 = dim >> 2;
    const int nr = rows - r0 < RN_R ? rows - r0 : RN_R;
    constexpr int NJ = RN_MAXD / 4 / 256;
    v4f xv[RN_R][NJ], wv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int i = tid + 256 * j;
        if (i < n4) {
#pragma unroll
            for (int r = 0; r < RN_R; ++r)  // rows past the end re-read the last one
                xv[r][j] = reinterpret_cast<const v4f *>(
                    x + (size_t)(r0 + (r < nr ? r : nr - 1)) * dim)[i];
            wv[j] = reinterpret_cast<const v4f *>(w)[i];
        }
    }
#pragma unroll
    for (int r = 0; r < RN_R; ++r)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = tid + 256 * j;
            if (i < n4) *reinterpret_cast<v4f *>(&s_p[r][4 * i]) = xv[r][j] * xv[r][j];
        }
    __syncthreads();
    if (tid < RN_R) {
        const float ss = orn_lds_seq_sum32(reinterpret_cast<const v4f *>(s_p[tid]), dim >> 5);
        s_inv[tid] = 1.0f / sqrtf(ss / (float)dim + 1e-6f);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN_R; ++r) {
        if (r >= nr) break;
        const float inv = s_inv[r];
        v4f *o4 = reinterpret_cast<v4f *>(out + (size_t)(r0 + r) * dim);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int i = tid + 256 * j;
            if (i < n4) o4[i] = wv[j] * (xv[r][j] * inv);
        }
    }
}

}  // namespace

extern "C" int ornk_matmul_f32(float *C, const float *A, const float *B, int M, int N, int K,
                               hipStream_t s)
{
    if (M <= 0 || N <= 0) return hipSuccess;
    const int mt = M > 4 ? 8 : M > 2 ? 4 : M, rs = M > 8 ? 2 : 1;
    const int gy = (M + mt * rs - 1) / (mt * rs);
    // Columns per thread: one while its waves fit the chip three to a SIMD
    // (1024 SIMDs), two while theirs fit two to a SIMD (8-row instances take
    // 150 to 211 registers), else four; more columns mean fewer LDS reads per
    // product but fewer waves.  us with one / two / four columns at K = 2048:
    // 16 rows, N = 65,536 188 / 230 / 340, 131,072 365 / 284 / 357, 248,320
    // 583 / 538 / 441; 8 rows, N = 190,000 274 / 300 / 323, 248,320 407 / 341
    // / 347; 1 row, N = 65,536 106 / 122 / 167, 248,320 349 / 325 / 334.
    const size_t waves = (((size_t)N + 63) / 64) * rs * gy;
    int nc = waves <= 3072 ? 1 : waves <= 4096 || mt <= 4 ? 2 : 4;
    while (nc > 1 && (N % nc || ((uintptr_t)B & (4 * nc - 1)))) nc /= 2;
    const dim3 grid(blocks_for(((size_t)N + nc - 1) / nc, 256 / rs), gy);
#define ORN_MM(MT_, NC_, RS_) \
    hipLaunchKernelGGL((k_matmul<MT_, NC_, RS_>), grid, dim3(256), 0, s, C, A, B, M, N, K)
#define ORN_MM_MT(NC_)                       \
    switch (rs == 2 ? 16 : mt) {             \
    case 1: ORN_MM(1, NC_, 1); break;        \
    case 2: ORN_MM(2, NC_, 1); break;        \
    case 4: ORN_MM(4, NC_, 1); break;        \
    case 8: ORN_MM(8, NC_, 1); break;        \
    default: ORN_MM(8, NC_, 2); break;       \
    }
    if (nc == 4) {
        if (rs == 2) ORN_MM(8, 4, 2);
        else ORN_MM(8, 4, 1);
    } else if (nc == 2) {
        ORN_MM_MT(2)
    } else {
        ORN_MM_MT(1)
    }
#undef ORN_MM_MT
#undef ORN_MM
    return hipGetLastError();
}

extern "C" int ornk_rmsnorm(float *out, const float *x, const float *w, int rows, int dim,
                            hipStream_t s)
{
    if (rows <= 0 || dim <= 0) return hipSuccess;
    if (dim > 16384) return hipErrorInvalidValue;  // the products live in LDS
    const bool al = (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0;
    // Up to 512 rows a work group per row finds room on a CU beside one other,
    // and its norm is the faster: dim 2048, 100 rows 13.4 us against 15.7, 256
    // 13.6 / 16.4, 400 16.3 / 16.8, 600 23.0 / 16.9; dim 256 6.4 / 6.9, 6.5 / 7.3,
    // 7.1 / 7.3, 9.0 / 7.3.
    if (rows > 512 && dim % 32 == 0 && dim <= RN_MAXD && al && out != x) {
        hipLaunchKernelGGL(k_rmsnorm_rows, dim3((rows + RN_R - 1) / RN_R), dim3(256), 0, s, out, x,
                           w, rows, dim);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_rmsnorm, dim3(rows), dim3(256), (size_t)dim * sizeof(float), s, out, x,
                       w, dim);
    return hipGetLastError();
}
