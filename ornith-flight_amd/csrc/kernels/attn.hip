// SPDX-License-Identifier: MIT
//
// The attention-side ops of the gpu.h backend: RoPE, single-head scaled
// dot-product attention, the gated DeltaNet step and the KV-cache append,
// with the semantics of the reference's Metal kernels (ops.metal:113-139,
// attention.metal:17-125) as dispatched by gpu_metal.m:495-583.  fp32
// operands and sums, compiled with -ffp-contract=off; the attention of long
// sequences takes each fp32 operand as three bf16 parts.
#include "common.h"
#include "launch.h"

namespace {

// ops.metal:113-139 on Q (heads [0, n_q)) and K (heads [0, n_k)) in one
// launch: the pair (x[i], x[i+1]), i = 2p < rot, of every head is rotated by
// pos * theta^(-i/rot).  The frequency is computed in double and rounded
// once, so it is the correctly rounded value of the formula (the Metal and
// CPU builds take it from a float pow, within an ulp of that).
__global__ void k_rope(float *Q, float *K, int head_dim, int n_q, int n_k, int rot, int pos,
                       float theta)
{
    const int half = rot / 2;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (half <= 0 || g >= (n_q + n_k) * half) return;
    int head = g / half;
    const int i = 2 * (g % half);
    float *x = Q;
    if (head >= n_q) {
        head -= n_q;
        x = K;
    }
    const float inv_freq = (float)(1.0 / pow((double)theta, (double)i / (double)rot));
    const float ang = (float)pos * inv_freq;
    const float c = cosf(ang), s = sinf(ang);
    float *h = x + (size_t)head * head_dim;
    const float a = h[i], b = h[i + 1];
    h[i] = a * c - b * s;
    h[i + 1] = a * s + b * c;
}

// attention.metal:17-68: out[r][c] = sum_t e^(s_rt) V[t][c] / sum_t e^(s_rt),
// s_rt = (Q[r] . K[t]) * scale, every key for every query (no mask), where
// the shader divides only when the sum exceeds 1e-10 and otherwise returns
// the unnormalised sum; so does this kernel.  The exponent is taken relative
// to the running row maximum m (online softmax): the unshifted sums are
// e^m times the shifted ones.  Where the shader's unshifted e^s overflows
// (scores above ~88, which make its output Inf or NaN) this kernel still
// returns the softmax.
//
// Work group: 256 threads, ATT_R = 16 query rows; keys in tiles of ATT_T =
// 16 staged in LDS (K with a padded row stride, so the 16 keys a row group
// reads at one time sit in different banks); 50 KB of LDS at hd = 256.
// Thread (r = tid/16, j = tid%16) scores key j of the tile for row r and
// owns output columns j, j+16, ... of row r.
constexpr int ATT_R = 16, ATT_T = 16, ATT_MAXD = 256;

__global__ __launch_bounds__(256) void k_attention(float *out, const float *Q, const float *K,
                                                   const float *V, int seq, int hd, float scale)
{
    extern __shared__ float lds[];
    const int ks = hd + 1;                 // padded K row stride
    float *Qs = lds;                       // [ATT_R][ks]
    float *Ks = Qs + ATT_R * ks;           // [ATT_T][ks]
    float *Vs = Ks + ATT_T * ks;           // [ATT_T][hd]
    float *Ps = Vs + ATT_T * hd;           // [ATT_R][ATT_T]
    const int tid = threadIdx.x, r = tid >> 4, j = tid & 15;
    const int row0 = blockIdx.x * ATT_R;
    for (int e = tid; e < ATT_R * hd; e += 256) {
        const int rr = e / hd, d = e - rr * hd;
        Qs[rr * ks + d] = row0 + rr < seq ? Q[(size_t)(row0 + rr) * hd + d] : 0.0f;
    }
    float acc[ATT_MAXD / 16];
#pragma unroll
    for (int c = 0; c < ATT_MAXD / 16; ++c) acc[c] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    for (int t0 = 0; t0 < seq; t0 += ATT_T) {
        __syncthreads();  // the previous tile's Ks/Vs/Ps are consumed
        for (int e = tid; e < ATT_T * hd; e += 256) {
            const int tt = e / hd, d = e - tt * hd;
            const bool in = t0 + tt < seq;
            Ks[tt * ks + d] = in ? K[(size_t)(t0 + tt) * hd + d] : 0.0f;
            Vs[tt * hd + d] = in ? V[(size_t)(t0 + tt) * hd + d] : 0.0f;
        }
        __syncthreads();
        float s0 = 0.0f;
        const float *q = Qs + r * ks, *k0 = Ks + j * ks;
        for (int d = 0; d < hd; ++d) s0 += q[d] * k0[d];
        s0 = t0 + j < seq ? s0 * scale : -INFINITY;
        float tm = s0;
#pragma unroll
        for (int o = 8; o >= 1; o >>= 1) tm = fmaxf(tm, __shfl_xor(tm, o, 16));
        const float mn = fmaxf(m, tm);  // finite: key t0 is always in range
        const float corr = expf(m - mn);
        const float p0 = expf(s0 - mn);
        float ps = p0;
#pragma unroll
        for (int o = 8; o >= 1; o >>= 1) ps += __shfl_xor(ps, o, 16);
        l = l * corr + ps;
        m = mn;
        Ps[r * ATT_T + j] = p0;
        __syncthreads();
        const float *pr = Ps + r * ATT_T;
#pragma unroll
        for (int c = 0; c < ATT_MAXD / 16; ++c) {
            const int col = j + 16 * c;
            if (col < hd) {
                float a = acc[c] * corr;
                for (int t = 0; t < ATT_T; ++t) a += pr[t] * Vs[t * hd + col];
                acc[c] = a;
            }
        }
    }
    if (row0 + r >= seq) return;
    // attention.metal:60-62: normalise only when the unshifted sum e^m * l
    // exceeds 1e-10; else the unnormalised sum e^m * acc
    const float em = expf(m);
    const float f = em * l > 1e-10f ? 1.0f / l : em;
#pragma unroll
    for (int c = 0; c < ATT_MAXD / 16; ++c) {
        const int col = j + 16 * c;
        if (col < hd) out[(size_t)(row0 + r) * hd + col] = acc[c] * f;
    }
}

// Whether any of the operands is not to be split into parts, of ntq
// tiles (k_attn_prep; the same answer in every thread).
__device__ __forceinline__ bool attn_bad(const int *bad, int ntq)
{
    int b = 0;
    for (int i = threadIdx.x; i < 3 * ntq; i += blockDim.x) b |= bad[i];
    return __syncthreads_or(b) != 0;
}

// ---------------------------------------------------------------------------
// The same attention on the matrix cores (v_mfma_f32_16x16x4f32: fp32 operands,
// fp32 accumulation), for head dims that are a multiple of 4 (HD = 64, 128 or
// 256: the smallest instance that holds hd; dims past hd are zero in Q, K and
// V and never stored).
//
// Work group: 4 waves over 64 query rows (wave w: rows 16w..16w+15 of the
// group's tile) and one split of the keys (grid.y splits, whole tiles of 16
// keys each).  Per tile of 16 keys, staged in LDS once for the four waves
// (double buffered, the next tile's loads in flight during this one's math):
//   S = Q K^T     HD/4 MFMAs; the wave's Q rows sit in registers as A
//                 operands, K rows are read from LDS as B operands;
//   p = e^(S*scale - m) with the running row maximum m and sum l (online
//                 softmax; m = -inf until a key is seen);
//   O = O*corr + P V   4 * HD/16 MFMAs; P goes from the C to the A layout
//                 through a 1 KB LDS slice per wave, V is staged transposed.
// The reduction index of every MFMA is permuted identically in both
// operands (k = 16*(s/4) + 4*g + s%4 for lane group g at step s, keys 4g + q
// at PV step q), so a lane's four consecutive steps read one 16-byte LDS
// word.  With one split the group writes out; else it writes O, m, l of its
// split and k_attn_merge combines the splits:
//   M = max m_i, L = sum l_i e^(m_i - M), O = sum O_i e^(m_i - M),
//   out = O / L where the unshifted sum e^M L exceeds 1e-10, else O e^M
// (attention.metal:60-62).
// ---------------------------------------------------------------------------
constexpr int AM_TK = 16;  // keys per tile

template <int HD>
struct AttnLds {
    float k[2][AM_TK][HD + 4];      // key rows (padded: conflict-free B reads)
    float vt[2][HD][AM_TK + 4];     // value tile transposed: vt[col][key]
    float p[4][16][AM_TK + 4];      // per wave: P in row-major, for the A layout
};

template <int HD>
__global__ void __launch_bounds__(256) k_attn_mma(float *out, float *Op, float *mlp,
                                                  const float *Q, const float *K, const float *V,
                                                  int seq, int hd, float scale, int tiles_per_split,
                                                  const int *bad, int ntq)
{
    __shared__ __align__(16) AttnLds<HD> L;  // 79 KB at HD = 256
    if (bad && !attn_bad(bad, ntq)) return;  // k_attn_split has taken it
    constexpr int NS = HD / 4, NC = HD / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, c = lane & 15;
    const int q0 = blockIdx.x * 64 + 16 * wave;
    const int n_tiles = (seq + AM_TK - 1) / AM_TK;
    const int t_lo = blockIdx.y * tiles_per_split;
    const int t_hi = min(n_tiles, t_lo + tiles_per_split);

    // Q rows (A operands): lane row q0 + c, steps s = 4j + i hold k = 16j + 4g + i
    float qa[NS];
    {
        const int r = q0 + c;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int k = 16 * j + 4 * g;
            v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (r < seq && k < hd) v = *reinterpret_cast<const v4f *>(Q + (size_t)r * hd + k);
#pragma unroll
            for (int i = 0; i < 4; ++i) qa[4 * j + i] = v[i];
        }
    }
    // staging: thread tid loads float4 number tid + 256i of each tile
    constexpr int F4 = AM_TK * HD / 4, F4T = F4 / 256;
    static_assert(F4 % 256 == 0, "whole float4s per thread");
    v4f rk[F4T], rv[F4T];
    auto load_tile = [&](int t) {
#pragma unroll
        for (int i = 0; i < F4T; ++i) {
            const int f = tid + 256 * i, key = f / (HD / 4), col = 4 * (f % (HD / 4));
            const int kk = t * AM_TK + key;
            const bool on = kk < seq && col < hd;
            rk[i] = on ? *reinterpret_cast<const v4f *>(K + (size_t)kk * hd + col)
                       : (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            rv[i] = on ? *reinterpret_cast<const v4f *>(V + (size_t)kk * hd + col)
                       : (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    auto store_tile = [&](int buf) {
#pragma unroll
        for (int i = 0; i < F4T; ++i) {
            const int f = tid + 256 * i, key = f / (HD / 4), col = 4 * (f % (HD / 4));
            *reinterpret_cast<v4f *>(&L.k[buf][key][col]) = rk[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) L.vt[buf][col + e][key] = rv[i][e];
        }
    };

    v4f o[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) o[j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    float m[4], l[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        m[r] = -INFINITY;
        l[r] = 0.0f;
    }

    if (t_lo < t_hi) {
        load_tile(t_lo);
        store_tile(0);
        if (t_lo + 1 < t_hi) load_tile(t_lo + 1);
    }
    __syncthreads();
    for (int t = t_lo; t < t_hi; ++t) {
        const int buf = (t - t_lo) & 1;
        // S = Q K^T for this wave's 16 rows and the tile's 16 keys
        v4f sacc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const v4f kb = *reinterpret_cast<const v4f *>(&L.k[buf][c][16 * j + 4 * g]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sacc = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * j + i], kb[i], sacc, 0, 0, 0);
        }
        // C layout: this lane holds key c, rows 4g + r
        const bool key_on = t * AM_TK + c < seq;
        float p[4], corr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float sc = key_on ? sacc[r] * scale : -INFINITY;
            float tm = sc;
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) tm = fmaxf(tm, __shfl_xor(tm, off, 16));
            const float mn = fmaxf(m[r], tm);
            const bool none = mn == -INFINITY;  // no key of this row seen yet
            corr[r] = none ? 1.0f : expf(m[r] - mn);
            p[r] = none ? 0.0f : expf(sc - mn);
            float ps = p[r];
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) ps += __shfl_xor(ps, off, 16);
            l[r] = l[r] * corr[r] + ps;
            m[r] = mn;
        }
        // P to the A layout through this wave's LDS slice
#pragma unroll
        for (int r = 0; r < 4; ++r) L.p[wave][4 * g + r][c] = p[r];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const v4f pa = *reinterpret_cast<const v4f *>(&L.p[wave][c][4 * g]);
        // O rows 4g + r scale by their corr; then O += P V
#pragma unroll
        for (int j = 0; j < NC; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) o[j][r] *= corr[r];
            const v4f vb = *reinterpret_cast<const v4f *>(&L.vt[buf][16 * j + c][4 * g]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[q], vb[q], o[j], 0, 0, 0);
        }
        // the next tile: written into the other buffer (last read two tiles
        // ago, before the previous barrier), then loads for the one after
        if (t + 1 < t_hi) {
            store_tile(buf ^ 1);
            if (t + 2 < t_hi) load_tile(t + 2);
        }
        __syncthreads();
    }

    // rows 4g + r of the wave's tile, columns 16j + c
    const int nsplit = gridDim.y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = q0 + 4 * g + r;
        if (row >= seq) continue;
        if (nsplit == 1) {
            const float em = expf(m[r]);
            const float f = em * l[r] > 1e-10f ? 1.0f / l[r] : em;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int col = 16 * j + c;
                if (col < hd) out[(size_t)row * hd + col] = o[j][r] * f;
            }
        } else {
            float *po = Op + ((size_t)blockIdx.y * seq + row) * hd;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int col = 16 * j + c;
                if (col < hd) po[col] = o[j][r];
            }
            if (c == 0) {
                mlp[((size_t)blockIdx.y * seq + row) * 2] = m[r];
                mlp[((size_t)blockIdx.y * seq + row) * 2 + 1] = l[r];
            }
        }
    }
}

// Combines the key splits: one thread per W outputs (hd % 4 == 0).
template <int W>
__global__ void k_attn_merge(float *out, const float *Op, const float *mlp, int seq, int hd,
                             int nsplit)
{
    typedef float vec __attribute__((ext_vector_type(W)));
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int hw = hd / W;
    if (i >= (size_t)seq * hw) return;
    const size_t row = i / hw, col = W * (i - row * hw);
    float M = -INFINITY;
    for (int sp = 0; sp < nsplit; ++sp) M = fmaxf(M, mlp[((size_t)sp * seq + row) * 2]);
    float Ls = 0.0f;
    vec O = 0.0f;
    for (int sp = 0; sp < nsplit; ++sp) {
        const float mi = mlp[((size_t)sp * seq + row) * 2];
        const float w = mi == -INFINITY ? 0.0f : expf(mi - M);
        Ls += mlp[((size_t)sp * seq + row) * 2 + 1] * w;
        O += *reinterpret_cast<const vec *>(Op + ((size_t)sp * seq + row) * hd + col) * w;
    }
    const float em = expf(M);
    *reinterpret_cast<vec *>(out + row * hd + col) = em * Ls > 1e-10f ? O / Ls : O * em;
}

// ---------------------------------------------------------------------------
// The same attention with every operand split into three bf16 parts
// (v_mfma_f32_32x32x16_bf16), for the sequences whose products, and not their
// launches, take the time.
//
// x = x1 + x2 + x3, each part the rest rounded to nearest: 3 x 8 significant
// bits hold all 24 of x, and bf16 has fp32's exponents, so the parts need no
// scale and a value loses nothing beside a larger one of its row or column.  A
// product is x1*y1 + x1*y2 + x2*y1 + x2*y2 + x1*y3 + x3*y1; what is dropped is
// below 2^-23 of it, of the order of an fp32 product's own rounding, and the
// sums are fp32: 6/16 of the matrix time of fp32 products.  Q, K and V are
// split once per call (k_attn_prep), the softmax weights, times 2^24 so that
// the smallest have all their parts too, in the kernel.
// Operands that hold a NaN, an infinity, a value past 2^59 (whose partial
// products could overflow where the fp32 sum does not) or a non-zero one below
// 2^-100 (whose last part would be subnormal) take k_attn_mma instead, decided
// on the device (bad[]).
//
// Work group: 4 waves of 32 query rows each and one split of the keys, tiles
// of 32 keys.  Scores are formed transposed, S^T = K Q^T, so that a lane holds
// 16 keys of one query: the row maximum and sum are in-lane but for one
// exchange between the lane halves, and the weights are already in the B
// layout of O^T = V^T P^T once V^T's keys are stored in that order (key
// position 8h + e of a step of 16 is key 4h + e for e < 4, 8 + 4h + e - 4
// beyond).  K and V of a tile (48 KB each at HD = 256) go from memory straight
// into one LDS slot each: V's while the scores are formed, the next K's during
// the products with V.
//
// What bounds it: Q's parts and O take 320 registers at HD = 256, so a SIMD
// holds one wave, whose matrix, exponential and LDS phases follow each other:
// the matrix cores are 39 % busy, beside 760 other vector instructions per
// wave and tile (4096 x 256: 116 us of 132 for the call; k_attn_mma takes 254).
// Operand reads two steps ahead instead of one, and two accumulators in turn,
// measured the same.  Error against 64 bits there 4.1e-7 (k_attn_mma 7.0e-7).
// Two fp16 halves per operand, scaled by row and column, take half the
// products and 107 us, but lose what lies 2^-38 below its row's or column's
// largest value, where it may be all that counts.
// ---------------------------------------------------------------------------
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int AS_TK = 32, AS_ROWS = 128;  // keys per tile, query rows per work group
constexpr float AS_MAX = 0x1p59f, AS_MIN = 0x1p-100f;  // magnitudes that are split

struct AttnPrep {
    __bf16 *q;        // [rows][part][HD]
    uint4 *kv;        // per tile [K part] 32 x HD, [V part] HD x 32
    int *bad;         // [tiles][Q, K, V]: not all of the tile's values are to be split
};

__device__ __forceinline__ bool attn_splits_exactly(float x)
{
    const float a = fabsf(x);
    return a == 0.0f || (a >= AS_MIN && a <= AS_MAX);
}

__device__ __forceinline__ void split3(float x, __bf16 &a, __bf16 &b, __bf16 &c)
{
    a = (__bf16)x;
    const float r = x - (float)a;
    b = (__bf16)r;
    c = (__bf16)(r - (float)b);
}

// The 16-byte chunk j of a row of K lies at position j ^ attn_kswz(row), so that
// 16 rows' reads of one chunk cover every LDS bank.
template <int HD>
__device__ __forceinline__ int attn_kswz(int r)
{
    return HD == 64 ? (r >> 1) & 7 : r & 15;
}

template <int HD>
__global__ void __launch_bounds__(256) k_attn_prep(AttnPrep P, const float *Q, const float *K,
                                                   const float *V, int seq, int hd, int nt)
{
    constexpr int W = HD / 64;  // columns per lane of a row
    // blockIdx.y: Q, K or V of tile blockIdx.x
    const int t = blockIdx.x, which = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __bf16 *kt = reinterpret_cast<__bf16 *>(P.kv) + (size_t)t * 6 * AS_TK * HD;
    bool ok = true;
    if (which && t >= nt) {
        // past the last tile of keys: nothing to write but the flag
    } else if (which < 2) {
        const float *src = which ? K : Q;
        constexpr int NR = AS_TK / 4;  // this wave's rows
        float x[NR][W];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int r = t * AS_TK + wave * NR + i;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const int c = W * lane + j;
                x[i][j] = r < seq && c < hd ? src[(size_t)r * hd + c] : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int lr = wave * NR + i, r = t * AS_TK + lr;
            __bf16 part[3][W];
#pragma unroll
            for (int j = 0; j < W; ++j) {
                ok = ok && attn_splits_exactly(x[i][j]);
                split3(x[i][j], part[0][j], part[1][j], part[2][j]);
            }
            __bf16 *d = which ? kt + (size_t)lr * HD : P.q + (size_t)r * 3 * HD;
            const int o = which ? 8 * ((W * lane / 8) ^ attn_kswz<HD>(lr)) + W * lane % 8 : W * lane;
#pragma unroll
            for (int n = 0; n < 3; ++n)
                __builtin_memcpy(__builtin_assume_aligned(d + n * (which ? AS_TK * HD : HD) + o, 2 * W),
                                 part[n], 2 * W);
        }
    } else {
        constexpr int NV = 4 * HD / 256;  // runs of 8 keys of one column per thread
        float x[NV][8];
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int i = tid + 256 * n, c = i % HD, ch = i / HD;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int r = t * AS_TK + 16 * (ch >> 1) + 4 * (ch & 1) + (e & 3) + 8 * (e >> 2);
                x[n][e] = r < seq && c < hd ? V[(size_t)r * hd + c] : 0.0f;
            }
        }
        __bf16 *vt = kt + 3 * AS_TK * HD;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int i = tid + 256 * n, c = i % HD, ch = i / HD;
            v8b part[3];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                __bf16 p0, p1, p2;
                ok = ok && attn_splits_exactly(x[n][e]);
                split3(x[n][e], p0, p1, p2);
                part[0][e] = p0;
                part[1][e] = p1;
                part[2][e] = p2;
            }
            // a column's four 16-byte chunks are rotated among themselves by
            // its number, so that 16 lanes' reads cover every LDS bank
            const int o = c * AS_TK + 8 * (ch ^ ((c >> 2) & 3));
#pragma unroll
            for (int m = 0; m < 3; ++m) *reinterpret_cast<v8b *>(vt + m * AS_TK * HD + o) = part[m];
        }
    }
    const int any = __syncthreads_or(!ok);
    if (tid == 0) P.bad[3 * t + which] = any;
}

// 16 bytes per lane from g + off (g the same in every lane) into LDS at base +
// 16 * lane; complete after the wave's next wait for its loads.  (As asm: for
// the builtin the compiler waits for the load before any LDS read.)
__device__ __forceinline__ uint32_t lds_addr(const void *p)
{
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p;
}
__device__ __forceinline__ void lds_load16(const void *g, uint32_t off, uint32_t base)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(base)), "v"(off), "s"(g)
                 : "memory", "m0");
}

// Keeps a value in the accumulator half of the register file, which the matrix
// instructions read and write directly: O and most of Q take it all, and left
// to itself the compiler moves O across the halves in every tile.
template <class T>
__device__ __forceinline__ void agpr(T &v)
{
    asm volatile("" : "+a"(v));
}

__device__ __forceinline__ v16f mfma_bf16(v8b a, v8b b, v16f c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <int HD>
struct AttnSplitLds {  // one tile's image
    __bf16 k[3][AS_TK * HD];
    __bf16 v[3][HD * AS_TK];
};

template <int HD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
    k_attn_split(float *out, float *Op, float *mlp, AttnPrep P, int seq, int hd, float scale,
                 int nt, int ntq, int tiles_per_split)
{
    __shared__ __align__(16) AttnSplitLds<HD> L;
    constexpr int NK = HD / 16, NJ = HD / 32, NL = 3 * HD / 64;  // NL: 16-byte words per thread of K, of V
    if (attn_bad(P.bad, ntq)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane & 31, h = lane >> 5;
    const int row = blockIdx.y * AS_ROWS + 32 * wave + q;
    const int t_lo = blockIdx.x * tiles_per_split, t_hi = min(nt, t_lo + tiles_per_split);

    v8b qv[3][NK];
    {
        const __bf16 *qr = P.q + (size_t)row * 3 * HD + 8 * h;
#pragma unroll
        for (int n = 0; n < 3; ++n)
#pragma unroll
            for (int s = 0; s < NK; ++s)
                qv[n][s] = *reinterpret_cast<const v8b *>(qr + n * HD + 16 * s);
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            agpr(qv[0][s]);
            agpr(qv[1][s]);
        }
    }

    // K or V of a tile straight into LDS: 1 KB per wave and load
    auto load = [&](const uint4 *p, const void *dst) {
        const uint32_t d = lds_addr(dst) + 1024 * wave;
#pragma unroll
        for (int i = 0; i < NL; ++i) lds_load16(p + 256 * i, 16 * tid, d + 4096 * i);
    };
    auto load_k = [&](int t) { load(P.kv + (size_t)t * (24 * HD), &L.k[0][0]); };
    auto load_v = [&](int t) { load(P.kv + (size_t)t * (24 * HD) + 12 * HD, &L.v[0][0]); };
    // This wave's loads have arrived; past the barrier every wave's have, and
    // every wave is done with what it read before it.
    auto arrived = [&] {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    // S^T of one tile: this lane's query, keys 8 (r / 4) + 4h + r % 4 (a
    // step's operands are read while the step before it multiplies)
    auto scores = [&] {
        v16f s0 = {}, s1 = {};  // the products of the first parts; the others
        v8b kb[2][3];
        auto read = [&](v8b(&r)[3], int s) {
            const int off = q * HD + 8 * ((2 * s + h) ^ attn_kswz<HD>(q));
#pragma unroll
            for (int n = 0; n < 3; ++n) r[n] = *reinterpret_cast<const v8b *>(&L.k[n][off]);
        };
        read(kb[0], 0);
#pragma unroll
        for (int s = 0; s < NK; ++s) {
            if (s + 1 < NK) read(kb[(s + 1) & 1], s + 1);
            __builtin_amdgcn_sched_barrier(0);
            const v8b(&k)[3] = kb[s & 1];
            s1 = mfma_bf16(k[2], qv[0][s], s1);
            s0 = mfma_bf16(k[0], qv[0][s], s0);
            s1 = mfma_bf16(k[0], qv[2][s], s1);
            s1 = mfma_bf16(k[1], qv[1][s], s1);
            s1 = mfma_bf16(k[1], qv[0][s], s1);
            s1 = mfma_bf16(k[0], qv[1][s], s1);
            __builtin_amdgcn_sched_barrier(0);
        }
        return s0 + s1;
    };

    auto read_v = [&](v8b(&r)[2][3], int j) {
        const int c = 32 * j + q;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int off = c * AS_TK + 8 * ((2 * s + h) ^ ((c >> 2) & 3));
#pragma unroll
            for (int n = 0; n < 3; ++n) r[s][n] = *reinterpret_cast<const v8b *>(&L.v[n][off]);
        }
    };

    v16f o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        o[j] = (v16f){};
        agpr(o[j]);
    }
    float m = -INFINITY, l = 0.0f;

    load_k(t_lo);
    for (int t = t_lo; t < t_hi; ++t) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) agpr(o[j]);
        arrived();  // K of tile t; V of tile t - 1 is consumed
        load_v(t);
        __builtin_amdgcn_sched_barrier(0);
        const v16f sc = scores();
        __builtin_amdgcn_sched_barrier(0);
        float p[16];
        float tm = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float v = sc[i] * scale;
            p[i] = AS_TK * t + 8 * (i >> 2) + 4 * h + (i & 3) < seq ? v : -INFINITY;
            tm = fmaxf(tm, p[i]);
        }
        tm = fmaxf(tm, __shfl_xor(tm, 32, 64));
        // The reference m moves only when the maximum has grown past it by a
        // factor of 4 (weights up to 4 stay): O is then left alone in most tiles.
        const float mn = tm > m + 1.38f ? tm : m;
        const bool none = mn == -INFINITY;  // no key of this row seen yet
        if (__any(mn != m)) {
            const float corr = none ? 1.0f : expf(m - mn);
            l *= corr;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                agpr(o[j]);  // 16 of O at a time in the other half
                __builtin_amdgcn_sched_barrier(0);
                v16f x = o[j] * corr;
                agpr(x);
                o[j] = x;
            }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) agpr(o[j]);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = none ? 0.0f : expf(p[r] - mn);
            l += p[r];
        }
        m = mn;
        v8b pv[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                __bf16 p0, p1, p2;
                split3(p[8 * s + e] * 0x1p24f, p0, p1, p2);
                pv[s][0][e] = p0;
                pv[s][1][e] = p1;
                pv[s][2][e] = p2;
            }
        arrived();  // V of tile t; its K is consumed
        if (t + 1 < t_hi) load_k(t + 1);
        v8b vb[2][2][3];
        read_v(vb[0], 0);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j + 1 < NJ) read_v(vb[(j + 1) & 1], j + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const v8b(&v)[3] = vb[j & 1][s];
                o[j] = mfma_bf16(v[2], pv[s][0], o[j]);
                o[j] = mfma_bf16(v[0], pv[s][2], o[j]);
                o[j] = mfma_bf16(v[1], pv[s][1], o[j]);
                o[j] = mfma_bf16(v[1], pv[s][0], o[j]);
                o[j] = mfma_bf16(v[0], pv[s][1], o[j]);
                o[j] = mfma_bf16(v[0], pv[s][0], o[j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    l += __shfl_xor(l, 32, 64);
    if (row >= seq) return;
    const int nsplit = gridDim.x;
    float f = 0x1p-24f;
    float *po;
    if (nsplit == 1) {
        const float em = expf(m);
        f *= em * l > 1e-10f ? 1.0f / l : em;
        po = out + (size_t)row * hd;
    } else {
        po = Op + ((size_t)blockIdx.x * seq + row) * hd;
        if (h == 0) {
            mlp[((size_t)blockIdx.x * seq + row) * 2] = m;
            mlp[((size_t)blockIdx.x * seq + row) * 2 + 1] = l;
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = 32 * j + 8 * i + 4 * h;
            if (c >= hd) continue;  // hd % 4 == 0
            v4f r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = o[j][4 * i + e] * f;
            *reinterpret_cast<v4f *>(po + c) = r;
        }
}

// attention.metal:80-108: thread i updates column i of the dim x dim state,
// state[j][i] = gate*state[j][i] + (1-gate)*K[i]*V[j], then
// out[i] = sum_j Q[j]*state[j][i] (j ascending), in the kernel's own order
// of operations.  Loads and stores are coalesced over i.
__global__ void k_deltanet_step(float *state, const float *Q, const float *K, const float *V,
                                float *out, int dim, float gate)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= dim) return;
    const float ki = K[i], omg = 1.0f - gate;
    for (int j = 0; j < dim; ++j) {
        float *p = state + (size_t)j * dim + i;
        *p = gate * *p + omg * ki * V[j];
    }
    float sum = 0.0f;
    for (int j = 0; j < dim; ++j) sum += Q[j] * state[(size_t)j * dim + i];
    out[i] = sum;
}

// attention.metal:113-125.
__global__ void k_kv_append(float *Kc, float *Vc, const float *Kn, const float *Vn, int pos,
                            int hd)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= hd) return;
    Kc[(size_t)pos * hd + t] = Kn[t];
    Vc[(size_t)pos * hd + t] = Vn[t];
}

}  // namespace

extern "C" int ornk_rope(float *Q, float *K, int head_dim, int n_q, int n_k, int pos, float theta,
                         hipStream_t s)
{
    const int rot = head_dim < 64 ? head_dim : 64;
    const int n = (n_q + n_k) * (rot / 2);
    if (head_dim <= 0 || n_q < 0 || n_k < 0 || n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_rope, dim3((n + 255) / 256), dim3(256), 0, s, Q, K, head_dim, n_q, n_k,
                       rot, pos, theta);
    return hipGetLastError();
}

extern "C" size_t ornk_attention_lds(int hd)
{
    return ((size_t)ATT_R * (hd + 1) + (size_t)ATT_T * (hd + 1) + (size_t)ATT_T * hd +
            (size_t)ATT_R * ATT_T) * sizeof(float);
}

extern "C" int ornk_attention(float *out, const float *Q, const float *K, const float *V, int seq,
                              int hd, float scale, hipStream_t s)
{
    if (seq <= 0 || hd <= 0) return hipSuccess;
    if (hd > ATT_MAXD) return hipErrorInvalidValue;
    const size_t lds = ornk_attention_lds(hd);  // <= 50,304 B
    hipLaunchKernelGGL(k_attention, dim3((seq + ATT_R - 1) / ATT_R), dim3(256), lds, s, out, Q, K,
                       V, seq, hd, scale);
    return hipGetLastError();
}

// The matrix-core attention: hd % 4 == 0 and hd <= 256.  ws: workspace of
// ornk_attention_mma_ws(seq, hd) bytes (the key splits' partial results).
static int attn_splits(int seq)
{
    const int nq = (seq + 63) / 64, nt = (seq + AM_TK - 1) / AM_TK;
    int ns = 512 / nq;
    ns = ns < 1 ? 1 : ns;
    return ns > nt ? nt : ns;
}

static int attn_hd(int hd) { return hd <= 64 ? 64 : hd <= 128 ? 128 : 256; }

// Parts (k_attn_split) from where their two more launches are paid back at
// every head dim; fp32 / parts, us per call: hd = 256 1152 keys 62 / 59, 1408
// 68 / 63, 1700 78 / 66, 4096 258 / 138; hd = 128 1152 50 / 49, 1408 55 / 54,
// 1536 57 / 52, 4096 154 / 93; hd = 64 1600 43 / 43, 1792 45 / 43, 2176 52 /
// 47, 4096 99 / 69.
static int attn_split(int seq, int hd)
{
    const int HD = attn_hd(hd);
    return seq >= (HD == 64 ? 1792 : 1536);
}

static int attn_key_splits(int seq, int *per)
{
    const int nq = (seq + AS_ROWS - 1) / AS_ROWS, nt = (seq + AS_TK - 1) / AS_TK;
    int ns = 256 / nq;
    ns = ns < 1 ? 1 : ns > nt ? nt : ns;
    *per = (nt + ns - 1) / ns;
    return (nt + *per - 1) / *per;  // every split holds at least one tile
}

struct AttnWs {
    size_t q, kv, bad, op, ml, bytes;
};

static AttnWs attn_ws(int seq, int hd)
{
    const int HD = attn_hd(hd), rq = (seq + AS_ROWS - 1) / AS_ROWS * AS_ROWS;
    const int rk = (seq + AS_TK - 1) / AS_TK * AS_TK;
    int per;
    const int ns = attn_key_splits(seq, &per);
    AttnWs w;
    size_t off = 0;
    auto take = [&](size_t n) {
        const size_t o = off;
        off += (n + 255) & ~(size_t)255;
        return o;
    };
    w.q = take((size_t)rq * HD * 6);
    w.kv = take((size_t)rk * HD * 12);
    w.bad = take((size_t)(rq / AS_TK) * 12);
    w.op = take(ns > 1 ? (size_t)ns * seq * hd * 4 : 0);
    w.ml = take(ns > 1 ? (size_t)ns * seq * 8 : 0);
    w.bytes = off;
    return w;
}

extern "C" size_t ornk_attention_mma_ws(int seq, int hd)
{
    if (attn_split(seq, hd)) return attn_ws(seq, hd).bytes;
    const int ns = attn_splits(seq);
    return ns > 1 ? (size_t)ns * seq * (hd + 2) * sizeof(float) : 0;
}

// Four outputs per thread from where that leaves every CU a wave; fewer wait
// longer for the splits than the wider loads save (us per call with one / four:
// 500 keys of 128 40.3 / 41.6, 1000 of 64 42.0 / 43.1, 1300 of 64 41.5 / 40.4,
// 700 of 128 54.5 / 52.7).
static void attn_merge(float *out, const float *Op, const float *mlp, int seq, int hd, int ns,
                       hipStream_t s)
{
    const size_t n = (size_t)seq * hd;
    if (n < 4 * 64 * 256)
        hipLaunchKernelGGL(k_attn_merge<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out, Op,
                           mlp, seq, hd, ns);
    else
        hipLaunchKernelGGL(k_attn_merge<4>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, out,
                           Op, mlp, seq, hd, ns);
}

template <int HD>
static void attn_split_launch(float *out, const float *Q, const float *K, const float *V, int seq,
                              int hd, float scale, uint8_t *ws, hipStream_t s)
{
    const AttnWs w = attn_ws(seq, hd);
    const int nq = (seq + AS_ROWS - 1) / AS_ROWS, nt = (seq + AS_TK - 1) / AS_TK;
    const int ntq = nq * (AS_ROWS / AS_TK);
    int per;
    const int ns = attn_key_splits(seq, &per);
    AttnPrep P;
    P.q = reinterpret_cast<__bf16 *>(ws + w.q);
    P.kv = reinterpret_cast<uint4 *>(ws + w.kv);
    P.bad = reinterpret_cast<int *>(ws + w.bad);
    float *Op = reinterpret_cast<float *>(ws + w.op), *mlp = reinterpret_cast<float *>(ws + w.ml);
    hipLaunchKernelGGL(k_attn_prep<HD>, dim3(ntq, 3), dim3(256), 0, s, P, Q, K, V, seq, hd, nt);
    hipLaunchKernelGGL(k_attn_split<HD>, dim3(ns, nq), dim3(256), 0, s, out, Op, mlp, P, seq, hd,
                       scale, nt, ntq, per);
    // the same splits (twice as many tiles of half the keys), the same partials
    hipLaunchKernelGGL(k_attn_mma<HD>, dim3((seq + 63) / 64, ns), dim3(256), 0, s, out, Op, mlp, Q, K,
                       V, seq, hd, scale, per * (AS_TK / AM_TK), P.bad, ntq);
    if (ns > 1) attn_merge(out, Op, mlp, seq, hd, ns, s);
}

extern "C" int ornk_attention_mma(float *out, const float *Q, const float *K, const float *V,
                                  int seq, int hd, float scale, void *ws, hipStream_t s)
{
    if (seq <= 0 || hd <= 0) return hipSuccess;
    if (hd % 4 || hd > 256) return hipErrorInvalidValue;
    if (attn_split(seq, hd)) {
        if (!ws) return hipErrorInvalidValue;
        uint8_t *w = static_cast<uint8_t *>(ws);
        if (hd <= 64) attn_split_launch<64>(out, Q, K, V, seq, hd, scale, w, s);
        else if (hd <= 128) attn_split_launch<128>(out, Q, K, V, seq, hd, scale, w, s);
        else attn_split_launch<256>(out, Q, K, V, seq, hd, scale, w, s);
        return hipGetLastError();
    }
    const int nt = (seq + AM_TK - 1) / AM_TK;
    int ns = attn_splits(seq);
    const int per = (nt + ns - 1) / ns;
    ns = (nt + per - 1) / per;  // every split holds at least one tile
    if (ns > 1 && !ws) return hipErrorInvalidValue;
    float *Op = static_cast<float *>(ws);
    float *mlp = Op ? Op + (size_t)ns * seq * hd : nullptr;
    const dim3 grid((seq + 63) / 64, ns);
#define ORN_ATT(HD_)                                                                          \
    hipLaunchKernelGGL(k_attn_mma<HD_>, grid, dim3(256), 0, s, out, Op, mlp,                  \
                       Q, K, V, seq, hd, scale, per, (const int *)nullptr, 0)
    if (hd <= 64) ORN_ATT(64);
    else if (hd <= 128) ORN_ATT(128);
    else ORN_ATT(256);
#undef ORN_ATT
    if (ns > 1) attn_merge(out, Op, mlp, seq, hd, ns, s);
    return hipGetLastError();
}

extern "C" int ornk_deltanet_step(float *state, const float *Q, const float *K, const float *V,
                                  float *out, int dim, float gate, hipStream_t s)
{
    if (dim <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_deltanet_step, dim3((dim + 255) / 256), dim3(256), 0, s, state, Q, K, V,
                       out, dim, gate);
    return hipGetLastError();
}

extern "C" int ornk_kv_append(float *Kc, float *Vc, const float *Kn, const float *Vn, int pos,
                              int hd, hipStream_t s)
{
    if (hd <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_kv_append, dim3((hd + 255) / 256), dim3(256), 0, s, Kc, Vc, Kn, Vn, pos,
                       hd);
    return hipGetLastError();
}
