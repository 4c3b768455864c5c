// SPDX-License-Identifier: MIT
//
// Expert products on the matrix cores straight from resident vec@mat K-quant
// blocks (a store without the MFMA layouts): work items of at most 16 or 32
// token rows of one expert, v_mfma_f32_16x16x32_f16 (operand preparation and
// its exactness argument: mfma_ops.h).
//
// A vec@mat block holds 256 outputs of one reduction row, so an operand's
// eight reduction values come from eight blocks.  A lane loads the same four
// bytes of its eight rows (k = 8g .. 8g+7 of the step): four low and four high
// nibbles, that is one operand of each of eight column tiles, whose columns
// are whatever those bytes hold (tile j, lane c -> an output; the outputs'
// order among the tiles is free).  v_perm pairs two rows' bytes into the
// halves that the fp16 pair needs.  Block scales (and mins) are decoded once
// per step by the whole work group into LDS, rows' d and dmin once per slice.
//
// Work group: 2 waves over one 256-column block of one matrix, wave w its half
// of the block's bytes, one slice of the reduction in steps of 32.  Per step
// the group prepares the next step's activation tile (hi/lo of x*s*d and, for
// Q4_K, of x*s*dmin) and scales into the other LDS buffer, one barrier.  The
// row scales s are powers of two from the rows' max |x| and the slice's
// largest |d|.
//
// Range: hi + lo hold a value to 2^-23 of itself down to 2^-17 of the row's and
// slice's largest product, and to a fixed 2^-39 of that below.  What lies so far
// down may be all that counts, where the weights of the rest are 0.  So a work
// group that has such values and sums too small to hide them (SUM_MIN) goes
// over its slice again for what hi + lo left out, times 2^24, and adds that to
// what it stored; each pass reaches 2^24 further down.
//
// What bounds it: the vector instructions that form operands (gate/up 278 per
// wave and step for 18 MFMAs per row tile, down 372 for 24).  The fp32 matvec
// kernels (expert_valu.hip) decode every weight once per token instead: 300
// tokens 1216 us for the layer, here 273.
#include "common.h"
#include "launch.h"
#include "mfma_ops.h"

#include <type_traits>

namespace {

using namespace orn_mfma;

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

#define ORN_INLINE __attribute__((always_inline))
#define ORN_BLK_KT 64  // most steps of a slice

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                             0x00020000);
}

__device__ __forceinline__ uint4 bload16(rsrc_t r, uint32_t voff, uint32_t soff)
{
    const v4u v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint32_t bload4(rsrc_t r, uint32_t voff, uint32_t soff)
{
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}

// Byte bb of two rows' words in the low bytes of the halves: a in the low one.
template <int BB>
__device__ __forceinline__ uint32_t pair_bytes(uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_perm(b, a, 0x0c000c00u | BB | ((4 + BB) << 16));
}

// LDS rows of 32 scales, 16 bytes of padding between them.
#define ORN_BLK_SST 40

template <int RT, int NARR, int NSUB>
struct BlkLds {
    _Float16 A[2][NARR][16 * RT * ORN_AST];
    _Float16 S[2][NSUB][ORN_BLK_SST];
    float d[ORN_BLK_KT * 32];
    float scale[16 * RT], inv[16 * RT];
    float red[2];
    uint32_t least[16 * RT];  // per row
};

// The largest v of the work group's 128 threads, in every one of them.
__device__ __forceinline__ float group_max(float v, float *red)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(red[0], red[1]);
}

// Whether some thread of the work group says so.
__device__ __forceinline__ bool group_any(bool v, float *red)
{
    const float w = __any(v) ? 1.0f : 0.0f;
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
    __syncthreads();
    const bool any = red[0] + red[1] > 0.0f;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(any);
}

// The smallest magnitude but 0 that a thread has split, as bits.
struct Least {
    uint32_t v = ~0u;

    static __device__ __forceinline__ uint32_t key(float x) { return 2 * __float_as_uint(x) - 1; }

    template <int VPT>
    __device__ __forceinline__ void see(const float (&a)[VPT])
    {
#pragma unroll
        for (int i = 0; i < VPT; ++i) v = min(v, key(a[i]));
    }
};

// Whether pass n over the rest has something to add to a row whose least is v:
// the first has of values below 2^-3, the others of those another 2^24 down
// (the fifth starts at 2^-99, where scaled operands begin to lack bits).
__device__ __forceinline__ bool rest_of(uint32_t v, int n)
{
    return n <= 5 && v < Least::key(0x1p-3f) - ((uint32_t)(24 * (n - 1)) << 24);
}

constexpr float REST_UP = 0x1p24f;

// 2^(-24 n)
__device__ __forceinline__ float rest_scale(int n) { return __uint_as_float((uint32_t)(127 - 24 * n) << 23); }

// Sums below which that may count: at 2^8 it is some 2^-21 of the sum (2^-26
// per value, times weights of 2^8, 512 of them).  The largest of a thread's
// eight sums of a row is compared: sums of ordinary operands are about 2^23 and
// one of them may well be small, and a work group that goes over its slice
// again can hold up the launch (gate/up at 300 tokens 147 us; 178 with every
// sum compared by itself).  A row's sums alone decide what is added to them,
// whatever the item's other rows are.
constexpr float SUM_MIN = 0x1p8f;

__device__ __forceinline__ float max8(const v4f (&s)[2])
{
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) m = fmaxf(m, fmaxf(fabsf(s[0][j]), fabsf(s[1][j])));
    return m;
}

// Pass n over a row whose least is v, for the eight sums of one thread (pass
// 0: s; later ones: what those before stored, old, to which s is added where
// it may count).  lim = SUM_MIN in the sums' scale.  Whether another pass may
// count.
template <bool REST>
__device__ __forceinline__ bool add_rest(v4f (&s)[2], const v4f (&old)[2], int n, uint32_t v, float lim)
{
    if constexpr (REST) {
        const bool on = rest_of(v, n) && max8(old) < lim * rest_scale(n - 1);
        const float f = rest_scale(n);
#pragma unroll
        for (int h = 0; h < 2; ++h) s[h] = on ? old[h] + s[h] * f : old[h];
        lim *= f;
    }
    return rest_of(v, n + 1) && max8(s) < lim;
}

// (a0, a1) -> hi and lo as in split2, but both rounded to nearest: 2^-23 of a
// and no bias, where truncation leaves up to 2^-21 of one sign (one token's
// error against 64 bits 2.7e-7 by the fp32 kernels, 6.8e-7 truncated).
__device__ __forceinline__ void split2_rn(float a0, float a1, uint32_t &hi, uint32_t &lo)
{
    typedef float v2f __attribute__((ext_vector_type(2)));
    const uint32_t h = as_u32(__builtin_convertvector((v2f){a0, a1}, v2h));
    float r0, r1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(h), "v"(a0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(h), "v"(a1));
    hi = h;
    lo = as_u32(__builtin_convertvector((v2f){r0, r1}, v2h));
}

// What hi + lo leave out of a, times 2^24; 0 where that is below 2^-23 of a.
__device__ __forceinline__ float split_rest(float a)
{
    if (!(fabsf(a) < 0.125f)) return 0.0f;
    const float r = a - (float)(_Float16)a;
    return (r - (float)(_Float16)r) * REST_UP;
}

// VPT values of one row times d (REST: what the passes before left out of that),
// hi/lo into the row's LDS words.
template <int VPT, bool REST>
__device__ __forceinline__ void store_split(const float *x, const float *d, int pass, Least &least,
                                            _Float16 *hi, _Float16 *lo)
{
    float a[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) a[i] = x[i] * d[i];
    if constexpr (!REST) least.see<VPT>(a);
    else
        for (int n = 0; n < pass; ++n)
#pragma unroll
            for (int i = 0; i < VPT; ++i) a[i] = split_rest(a[i]);
    uint32_t h[VPT / 2], l[VPT / 2];
#pragma unroll
    for (int i = 0; i < VPT / 2; ++i) split2_rn(a[2 * i], a[2 * i + 1], h[i], l[i]);
    if constexpr (VPT == 8) {
        *reinterpret_cast<uint4 *>(hi) = make_uint4(h[0], h[1], h[2], h[3]);
        *reinterpret_cast<uint4 *>(lo) = make_uint4(l[0], l[1], l[2], l[3]);
    } else {
        *reinterpret_cast<uint2 *>(hi) = make_uint2(h[0], h[1]);
        *reinterpret_cast<uint2 *>(lo) = make_uint2(l[0], l[1]);
    }
}

// ---------------------------------------------------------------------------
// Gate/up (Q4_K).  Logical tile = ((item * ks + kslice) * 2 + m) * (H/256) + b;
// output gu[kslice][row][m*H + n].
// ---------------------------------------------------------------------------
template <int RT>
struct GuLds : BlkLds<RT, 4, 16> {  // S: 8 scales, 8 mins
    float dm[ORN_BLK_KT * 32];
};

// Pass 0 over the slice, or (REST) a later one over what those before left out;
// whether another is due.
template <int RT, bool REST>
__device__ __forceinline__ bool
gu_pass(GuLds<RT> &L, int pass, int n_live, const uint8_t *__restrict__ gate,
        const uint8_t *__restrict__ up, const float *__restrict__ xn,
        const float *__restrict__ x_amax, const int4 *__restrict__ items,
        const int *__restrict__ row_token, float *gu, int D, int H, int ks, int rows_max)
{
    constexpr int VPT = 4 * RT;
    const int NB = H >> 8, per_item = 2 * NB * ks;
    const int tile = xcd_remap(blockIdx.x, n_live);
    const int b = tile % NB, m = (tile / NB) & 1, kslice = (tile / (2 * NB)) % ks;
    const int4 itm = items[tile / per_item];
    const int e = itm.w, nrows = itm.z;
    int tid = threadIdx.x;
    if (REST) asm volatile("" : "+v"(tid));  // keeps nothing of pass 0's addresses
    const int lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KT = D / 32 / ks, k0 = 32 * KT * kslice;
    const uint8_t *base =
        (m ? up : gate) + ((size_t)(e * NB + b) * D + k0) * ORN_Q4K_BYTES;
    const rsrc_t rq = make_rsrc(base, (uint32_t)KT * 32 * ORN_Q4K_BYTES);
    const int di = 16 * wave + c, ch = di >> 3;  // this lane's word of qs, its 64-output chunk
    const uint32_t w_off = (uint32_t)(8 * g) * ORN_Q4K_BYTES + ORN_Q4K_OFF_QS + 4 * di;
    const int hr = tid >> 2, hj = 2 * (tid & 3);  // the row and sub-blocks this thread decodes
    const uint32_t h_off = (uint32_t)hr * ORN_Q4K_BYTES;
    constexpr uint32_t STEP = 32 * ORN_Q4K_BYTES;

    struct Ring {
        uint32_t w[8];
        uint4 hd;
    } st0, st1;
    auto load = [&](Ring &r, int kt) ORN_INLINE {
        kt = kt < KT ? kt : KT - 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) r.w[i] = bload4(rq, w_off + i * ORN_Q4K_BYTES, kt * STEP);
        r.hd = bload16(rq, h_off, kt * STEP);
    };
    load(st0, 0);
    load(st1, 1);

    const int ar = tid / (32 / VPT), ak = VPT * (tid % (32 / VPT));
    const bool live = ar < nrows;
    const int tok = row_token[itm.y + (live ? ar : 0)];
    const float *xr = xn + (size_t)tok * D + k0 + ak;
    struct XRow {
        float v[VPT];
    } x0, x1;
    auto load_x = [&](XRow &x, int kt) ORN_INLINE {
        kt = kt < KT ? kt : KT - 1;
#pragma unroll
        for (int i = 0; i < VPT; i += 4) {
            const v4f v = *reinterpret_cast<const v4f *>(xr + 32 * kt + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) x.v[i + j] = v[j];
        }
    };
    load_x(x0, 0);
    load_x(x1, 1);

    // d and dmin of the slice's rows, and the largest of them
    float mx = 0.0f;
    for (int i = tid; i < 32 * KT; i += 128) {
        const uint32_t v = bload4(rq, (uint32_t)i * ORN_Q4K_BYTES, 0);
        const float d = orn_half_to_float(v & 0xFFFFu), dm = orn_half_to_float(v >> 16);
        L.d[i] = d;
        L.dm[i] = dm;
        mx = fmaxf(mx, fmaxf(fabsf(d), fabsf(dm)));
    }
    if (!REST && tid < 16 * RT) L.least[tid] = ~0u;
    mx = group_max(mx, L.red);
    const float as = live ? row_scale(x_amax[tok], mx) : 0.0f;
    if (ak == 0) L.inv[ar] = as != 0.0f ? 1.0f / as : 0.0f;

    Least least;
    auto prep = [&](const uint4 &hd, const XRow &x, int kt, int buf) ORN_INLINE {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t sc, mn;
            orn_scale_min_k4(hj + i, hd.y, hd.z, hd.w, sc, mn);
            L.S[buf][hj + i][hr] = (_Float16)(float)sc;
            L.S[buf][8 + hj + i][hr] = (_Float16)(float)mn;
        }
        kt = kt < KT ? kt : KT - 1;
        float xs[VPT], d[VPT], dm[VPT];
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            // a row past the item's end is a live one's values times 0 (its
            // results are not stored, but a NaN there must not be made)
            xs[i] = live ? x.v[i] * as : 0.0f;
            d[i] = L.d[32 * kt + ak + i];
            dm[i] = L.dm[32 * kt + ak + i];
        }
        const int o = ar * ORN_AST + ak;
        store_split<VPT, REST>(xs, d, pass, least, &L.A[buf][0][o], &L.A[buf][1][o]);
        store_split<VPT, REST>(xs, dm, pass, least, &L.A[buf][2][o], &L.A[buf][3][o]);
    };

    v4f acc[RT][8], accm[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[rt][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
        accm[rt] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    }
    const int rt_live = RT > 1 && nrows > 16 ? RT : 1;

    auto sub = [&](Ring &st, const uint4 &nhd, XRow &nx, int kt, int buf) ORN_INLINE {
        const uint4 slo = *reinterpret_cast<const uint4 *>(&L.S[buf][2 * ch][8 * g]);
        const uint4 shi = *reinterpret_cast<const uint4 *>(&L.S[buf][2 * ch + 1][8 * g]);
        uint4 mz = *reinterpret_cast<const uint4 *>(&L.S[buf][8 + 4 * wave + (c & 3)][8 * g]);
        if (c >= 4) mz = make_uint4(0u, 0u, 0u, 0u);  // 4 sub-blocks a wave: 4 columns
        const v8h bm = __builtin_bit_cast(v8h, mz);
        const uint32_t sl[4] = {slo.x, slo.y, slo.z, slo.w}, sh[4] = {shi.x, shi.y, shi.z, shi.w};
        uint32_t o[8][4];
        auto operand = [&](auto bbc) ORN_INLINE {
            constexpr int BB = decltype(bbc)::value;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const v2h k1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
                const uint32_t u = pair_bytes<BB>(st.w[2 * p], st.w[2 * p + 1]);
                const v2h vl = as_v2h(sl[p]), vh = as_v2h(sh[p]);
                o[BB][p] = as_u32(__builtin_elementwise_fma(as_v2h(magic_pair(u)), vl, vl * k1024));
                o[4 + BB][p] =
                    as_u32(__builtin_elementwise_fma(as_v2h(magic_pair(u >> 4)), vh, vh * k1024));
            }
        };
        operand(std::integral_constant<int, 0>{});
        operand(std::integral_constant<int, 1>{});
        operand(std::integral_constant<int, 2>{});
        operand(std::integral_constant<int, 3>{});
        __builtin_amdgcn_sched_barrier(0);
        load(st, kt + 2);
        __builtin_amdgcn_sched_barrier(0);
        const int ro = c * ORN_AST + 8 * g;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (rt >= rt_live) break;
            const int off = 16 * rt * ORN_AST + ro;
            const v8h ahi = *reinterpret_cast<const v8h *>(&L.A[buf][0][off]);
            const v8h alo = *reinterpret_cast<const v8h *>(&L.A[buf][1][off]);
            const v8h mhi = *reinterpret_cast<const v8h *>(&L.A[buf][2][off]);
            const v8h mlo = *reinterpret_cast<const v8h *>(&L.A[buf][3][off]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                acc[rt][j] = mfma(ahi, to_v8h(o[j][0], o[j][1], o[j][2], o[j][3]), acc[rt][j]);
            accm[rt] = mfma(mhi, bm, accm[rt]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                acc[rt][j] = mfma(alo, to_v8h(o[j][0], o[j][1], o[j][2], o[j][3]), acc[rt][j]);
            accm[rt] = mfma(mlo, bm, accm[rt]);
        }
        prep(nhd, nx, kt + 1, buf ^ 1);
        load_x(nx, kt + 3);
        __syncthreads();
    };
    prep(st0.hd, x0, 0, 0);
    load_x(x0, 2);
    __syncthreads();
    for (int kt = 0; kt < KT; kt += 2) {  // KT is even (launcher)
        sub(st0, st1.hd, x1, kt, 0);
        sub(st1, st0.hd, x0, kt + 1, 1);
    }

    const int col = m * H + 256 * b + 64 * ch + 4 * (di & 7);
    bool again = false;
    if constexpr (!REST) {
        atomicMin(&L.least[ar], least.v);
        __syncthreads();
    }
    float *row0 = gu + ((size_t)kslice * rows_max + itm.y) * (2 * H) + col;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * rt + 4 * g + r;
            const float si = L.inv[row];
            const float ml = __shfl(accm[rt][r], 16 * g + 2 * (c >> 3), 64);
            const float mh = __shfl(accm[rt][r], 16 * g + 2 * (c >> 3) + 1, 64);
            if (row < nrows) {
                v4f sum[2];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    sum[0][j] = (acc[rt][j][r] - ml) * si;
                    sum[1][j] = (acc[rt][4 + j][r] - mh) * si;
                }
                float *o = row0 + (size_t)row * (2 * H);
                v4f old[2];
                if constexpr (REST) {
                    old[0] = *reinterpret_cast<const v4f *>(o);
                    old[1] = *reinterpret_cast<const v4f *>(o + 32);
                }
                again = add_rest<REST>(sum, old, pass, L.least[row], SUM_MIN * si) || again;
                *reinterpret_cast<v4f *>(o) = sum[0];
                *reinterpret_cast<v4f *>(o + 32) = sum[1];
            }
        }
    return group_any(again, L.red);
}

// (Two waves per SIMD: three leave 168 registers, with which the one-tile
// instances spill.)
template <int RT>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
    k_gu_blk(const uint8_t *__restrict__ gate, const uint8_t *__restrict__ up,
             const float *__restrict__ xn, const float *__restrict__ x_amax,
             const int *__restrict__ ctl, const int4 *__restrict__ items,
             const int *__restrict__ row_token, float *gu, int D, int H, int ks, int rows_max)
{
    __shared__ __align__(16) GuLds<RT> L;
    const int n_live = ctl[1] * 2 * (H >> 8) * ks;
    if ((int)blockIdx.x >= n_live) return;
    bool again = gu_pass<RT, false>(L, 0, n_live, gate, up, xn, x_amax, items, row_token, gu,
                                    D, H, ks, rows_max);
    for (int pass = 1; again; ++pass)
        again = gu_pass<RT, true>(L, pass, n_live, gate, up, xn, x_amax, items, row_token, gu,
                                  D, H, ks, rows_max);
}

// ---------------------------------------------------------------------------
// Down (Q6_K).  Logical tile = (item * ks + kslice) * (D/256) + b; output
// dn[kslice][row][n].  Lane c takes half n = c/8 of the block and l = 4(c%8)
// .. +3 of its quarters; wave w the low nibbles of quarter w (ql[64n + 32w +
// l]) and the high ones of quarter w + 2, with their bits of qh[32n + l]
// (gguf.c:64-86).  Sub-scales reach +-128, so every product has the
// remainder operand (q6_b2's form).
// ---------------------------------------------------------------------------
template <int RT>
using DnLds = BlkLds<RT, 2, 16>;

template <int RT, bool REST>
__device__ __forceinline__ bool
dn_pass(DnLds<RT> &L, int pass, int n_live, const uint8_t *__restrict__ body,
        const uint16_t *__restrict__ dv, const float *__restrict__ mid,
        const float *__restrict__ mid_amax, const int4 *__restrict__ items, float *dn,
        int D, int H, int ks, int rows_max)
{
    constexpr int VPT = 4 * RT;
    const int NB = D >> 8, per_item = NB * ks;
    const int tile = xcd_remap(blockIdx.x, n_live);
    const int b = tile % NB, kslice = (tile / NB) % ks;
    const int4 itm = items[tile / per_item];
    const int e = itm.w, nrows = itm.z;
    int tid = threadIdx.x;
    if (REST) asm volatile("" : "+v"(tid));  // keeps nothing of pass 0's addresses
    const int lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KT = H / 32 / ks, k0 = 32 * KT * kslice;
    const size_t blk0 = (size_t)(e * NB + b) * H + k0;
    const rsrc_t rq = make_rsrc(body + blk0 * 208, (uint32_t)KT * 32 * 208);
    const int n = c >> 3, l4 = 4 * (c & 7);
    const uint32_t l_off = (uint32_t)(8 * g) * 208 + 64 * n + 32 * wave + l4;
    const uint32_t q_off = (uint32_t)(8 * g) * 208 + 128 + 32 * n + l4;
    const int hr = tid >> 2, hj = 4 * (tid & 3);  // the row and sub-scales this thread decodes
    const uint32_t s_off = (uint32_t)hr * 208 + 192 + hj;
    const int sub_lo = 8 * n + 2 * wave + (l4 >> 4);
    constexpr uint32_t STEP = 32 * 208;

    struct Ring {
        uint32_t l[8], q[8], sc;
    } st0, st1;
    auto load = [&](Ring &r, int kt) ORN_INLINE {
        kt = kt < KT ? kt : KT - 1;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            r.l[i] = bload4(rq, l_off + i * 208, kt * STEP);
            r.q[i] = bload4(rq, q_off + i * 208, kt * STEP);
        }
        r.sc = bload4(rq, s_off, kt * STEP);
    };
    load(st0, 0);
    load(st1, 1);

    const int ar = tid / (32 / VPT), ak = VPT * (tid % (32 / VPT));
    const bool live = ar < nrows;
    const int arow = itm.y + (live ? ar : 0);
    const float *xr = mid + (size_t)arow * H + k0 + ak;
    struct XRow {
        float v[VPT];
    } x0, x1;
    auto load_x = [&](XRow &x, int kt) ORN_INLINE {
        kt = kt < KT ? kt : KT - 1;
#pragma unroll
        for (int i = 0; i < VPT; i += 4) {
            const v4f v = *reinterpret_cast<const v4f *>(xr + 32 * kt + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) x.v[i + j] = v[j];
        }
    };
    load_x(x0, 0);
    load_x(x1, 1);

    float mx = 0.0f;
    for (int i = tid; i < 32 * KT; i += 128) {
        const float d = orn_half_to_float(dv[blk0 + i]);
        L.d[i] = d;
        mx = fmaxf(mx, fabsf(d));
    }
    if (!REST && tid < 16 * RT) L.least[tid] = ~0u;
    mx = group_max(mx, L.red);
    // The row's largest in this slice: a saturated gate leaves slices whose
    // values are all far below the row's largest, and so are their sums.
    float xm = 0.0f;
    if (ks == 1) {
        xm = mid_amax[arow];
    } else {
#pragma unroll 4
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < VPT; i += 4) {
                const v4f v = *reinterpret_cast<const v4f *>(xr + 32 * kt + i);
                xm = fmaxf(fmaxf(xm, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
            }
#pragma unroll
        for (int o = 1; o < 32 / VPT; o *= 2) xm = fmaxf(xm, __shfl_xor(xm, o, 64));
    }
    const float as = live ? row_scale(xm, mx) : 0.0f;
    if (ak == 0) L.inv[ar] = as != 0.0f ? 1.0f / as : 0.0f;

    Least least;
    auto prep = [&](uint32_t sc, const XRow &x, int kt, int buf) ORN_INLINE {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            L.S[buf][hj + i][hr] = (_Float16)(float)(int)(int8_t)(sc >> (8 * i));
        kt = kt < KT ? kt : KT - 1;
        float xs[VPT], d[VPT];
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            xs[i] = live ? x.v[i] * as : 0.0f;
            d[i] = L.d[32 * kt + ak + i];
        }
        const int o = ar * ORN_AST + ak;
        store_split<VPT, REST>(xs, d, pass, least, &L.A[buf][0][o], &L.A[buf][1][o]);
    };

    v4f acc[RT][8];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[rt][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const int rt_live = RT > 1 && nrows > 16 ? RT : 1;

    auto sub = [&](Ring &st, uint32_t nsc, XRow &nx, int kt, int buf) ORN_INLINE {
        const int ro = c * ORN_AST + 8 * g;
        v8h ahi[RT], alo[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            ahi[rt] = *reinterpret_cast<const v8h *>(&L.A[buf][0][16 * rt * ORN_AST + ro]);
            alo[rt] = *reinterpret_cast<const v8h *>(&L.A[buf][1][16 * rt * ORN_AST + ro]);
        }
        auto half = [&](auto hic) ORN_INLINE {  // quarter `wave` (low nibbles), then wave + 2
            constexpr int HI = decltype(hic)::value;
            const uint4 s4 = *reinterpret_cast<const uint4 *>(&L.S[buf][sub_lo + 4 * HI][8 * g]);
            const uint32_t sv[4] = {s4.x, s4.y, s4.z, s4.w};
            const int sh = 2 * wave + 4 * HI;
            uint32_t o1[4][4], o2[4][4];
            auto operand = [&](auto bbc) ORN_INLINE {
                constexpr int BB = decltype(bbc)::value;
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t u = pair_bytes<BB>(st.l[2 * p], st.l[2 * p + 1]);
                    const uint32_t v = pair_bytes<BB>(st.q[2 * p], st.q[2 * p + 1]);
                    const uint32_t w =
                        magic_pair(HI ? u >> 4 : u) | (((v >> sh) & 0x00030003u) << 4);
                    const v2h qv = as_v2h(w) + (v2h){(_Float16)-1056.0f, (_Float16)-1056.0f};
                    const v2h s2 = as_v2h(sv[p]), bh = qv * s2;
                    o1[BB][p] = as_u32(bh);
                    o2[BB][p] = as_u32(__builtin_elementwise_fma(qv, s2, -bh));
                }
            };
            operand(std::integral_constant<int, 0>{});
            operand(std::integral_constant<int, 1>{});
            operand(std::integral_constant<int, 2>{});
            operand(std::integral_constant<int, 3>{});
            if (HI) {
                __builtin_amdgcn_sched_barrier(0);
                load(st, kt + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (rt >= rt_live) break;
#pragma unroll
                for (int term = 0; term < 3; ++term)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t *o = term == 2 ? o2[j] : o1[j];
                        acc[rt][4 * HI + j] = mfma(term == 1 ? alo[rt] : ahi[rt],
                                                   to_v8h(o[0], o[1], o[2], o[3]),
                                                   acc[rt][4 * HI + j]);
                    }
            }
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
        prep(nsc, nx, kt + 1, buf ^ 1);
        load_x(nx, kt + 3);
        __syncthreads();
    };
    prep(st0.sc, x0, 0, 0);
    load_x(x0, 2);
    __syncthreads();
    for (int kt = 0; kt < KT; kt += 2) {
        sub(st0, st1.sc, x1, kt, 0);
        sub(st1, st0.sc, x0, kt + 1, 1);
    }

    bool again = false;
    if constexpr (!REST) {
        atomicMin(&L.least[ar], least.v);
        __syncthreads();
    }
    float *row0 = dn + ((size_t)kslice * rows_max + itm.y) * D + 256 * b + 128 * n + 32 * wave + l4;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * rt + 4 * g + r;
            const float si = L.inv[row];
            if (row < nrows) {
                v4f sum[2];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    sum[0][j] = acc[rt][j][r] * si;
                    sum[1][j] = acc[rt][4 + j][r] * si;
                }
                float *o = row0 + (size_t)row * D;
                v4f old[2];
                if constexpr (REST) {
                    old[0] = *reinterpret_cast<const v4f *>(o);
                    old[1] = *reinterpret_cast<const v4f *>(o + 64);
                }
                again = add_rest<REST>(sum, old, pass, L.least[row], SUM_MIN * si) || again;
                *reinterpret_cast<v4f *>(o) = sum[0];
                *reinterpret_cast<v4f *>(o + 64) = sum[1];
            }
        }
    return group_any(again, L.red);
}

template <int RT>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
    k_dn_blk(const uint8_t *__restrict__ body, const uint16_t *__restrict__ dv,
             const float *__restrict__ mid, const float *__restrict__ mid_amax,
             const int *__restrict__ ctl, const int4 *__restrict__ items, float *dn, int D, int H,
             int ks, int rows_max)
{
    __shared__ __align__(16) DnLds<RT> L;
    const int n_live = ctl[1] * (D >> 8) * ks;
    if ((int)blockIdx.x >= n_live) return;
    bool again = dn_pass<RT, false>(L, 0, n_live, body, dv, mid, mid_amax, items, dn, D, H, ks,
                                    rows_max);
    for (int pass = 1; again; ++pass)
        again = dn_pass<RT, true>(L, pass, n_live, body, dv, mid, mid_amax, items, dn, D, H, ks,
                                  rows_max);
}

}  // namespace

// Steps of a slice: an even count, at most ORN_BLK_KT.
static bool blk_kt_ok(int kt) { return kt >= 2 && kt % 2 == 0 && kt <= ORN_BLK_KT; }

extern "C" int ornk_blk_supported(int kt_gu, int kt_dn) { return blk_kt_ok(kt_gu) && blk_kt_ok(kt_dn); }

extern "C" int ornk_moe_gateup_blk(const ornk_moe_args *a, hipStream_t s)
{
    const int ks = a->ks_gu;
    if (a->D % 256 || a->H % 256 || ks < 1 || (a->D / 32) % ks || !blk_kt_ok(a->D / 32 / ks) ||
        a->tchunk > 32 || !a->x_amax || !a->router_amax)
        return hipErrorInvalidValue;
    const float *xin = a->apply_norm ? a->xn : a->x;
    const dim3 grid(a->items_max * 2 * (a->H / 256) * ks);
#define ORN_GUB(R)                                                                               \
    ORN_LAUNCH_EV(a, k_gu_blk<R>, grid, dim3(128), 0, s, a->gate, a->up, xin, a->x_amax, a->ctl, \
                  reinterpret_cast<const int4 *>(a->items), a->row_token, a->gu_part, a->D, a->H, \
                  ks, a->rows_max)
    if (a->tchunk > 16) ORN_GUB(2);
    else ORN_GUB(1);
#undef ORN_GUB
    return hipGetLastError();
}

extern "C" int ornk_moe_down_blk(const ornk_moe_args *a, hipStream_t s)
{
    const int ks = a->ks_dn;
    if (a->H % 256 || a->D % 256 || ks < 1 || (a->H / 32) % ks || !blk_kt_ok(a->H / 32 / ks) ||
        a->tchunk > 32)
        return hipErrorInvalidValue;
    const dim3 grid(a->items_max * (a->D / 256) * ks);
#define ORN_DNB(R)                                                                              \
    ORN_LAUNCH_EV(a, k_dn_blk<R>, grid, dim3(128), 0, s, a->down_body, a->down_d, a->mid,       \
                  a->mid_amax, a->ctl, reinterpret_cast<const int4 *>(a->items), a->dn_part, a->D, \
                  a->H, ks, a->rows_max)
    if (a->tchunk > 16) ORN_DNB(2);
    else ORN_DNB(1);
#undef ORN_DNB
    return hipGetLastError();
}
