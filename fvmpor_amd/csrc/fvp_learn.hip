// Mesh message-passing network on gfx950: BF16 weights and activations, FP32
// accumulation on the matrix cores (v_mfma_f32_32x32x8bf16_1k), training
// (forward, backward, Adam) and inference.
//
//   H0 = bf16(relu(X0 We + be));  per layer: A = bf16(mean_N(H)),
//   Z = H W1 + A W2 + b,  H = bf16(H + relu(Z));   y = H Wd + bd
//
// on the node-adjacency graph of a mesh (64 features per node).  The matrix
// products are N x K by K x 64 (K = 16 or 64): one wavefront computes 32 rows x
// 64 columns as two 32 x 32 MFMA tiles, the weights staged transposed in LDS.
// Weight gradients (K x 64, a reduction over the N rows) use the same
// instruction with the rows as the reduction dimension.  No counterpart in the
// reference: it supplies the Newton initial iterate of the integrator.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fvp_internal.h"
#include "fvp_sums.h"

using fvp::DevBuf;
using fvp::set_error;

typedef unsigned short bf16_t;
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

namespace {

constexpr int kF = 16;      // input features (padded)
constexpr int kH = 64;      // hidden width
constexpr int kMaxLayers = 8;

__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) {  // round to nearest even (finite inputs)
    unsigned u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}

// ---- fragments --------------------------------------------------------------------
// The matrix products run as v_mfma_f32_32x32x8bf16_1k with the weights (transposed)
// as the first operand and 32 nodes as the columns of the second: lane l holds, for
// node l % 32, the features 8 s + 4 (l / 32) + (0..3) of K step s, and the result's
// features 32 t + 8 q + 4 (l / 32) + (0..3) in registers 4 q + (0..3) of tile t.  So a
// layer's input fragment s = 4 t + q and its result hold the same features of the
// same node in the same lane, and the residual update needs no data movement.
// Memory wants 16 bytes per lane: the two lanes of a node swap 8-byte halves
// (v_permlane32_swap_b32) on the way in and out.
constexpr int kRow = 68;  // halves per LDS row of 64: 8-byte reads of 32 rows meet no bank twice

__device__ __forceinline__ void swap32(unsigned &a, unsigned &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// 16 bytes per lane (features 16 p + 8 (l / 32) + (0..7)) <-> the fragments of K steps 2 p, 2 p + 1
__device__ __forceinline__ void frag_swap(uint2 &a, uint2 &b) {
    swap32(a.x, b.x);
    swap32(a.y, b.y);
}
__device__ __forceinline__ uint4 frag_to_row(uint2 a, uint2 b) {
    frag_swap(a, b);
    return make_uint4(a.x, a.y, b.x, b.y);
}
__device__ __forceinline__ short4_t as_frag(uint2 v) {
    union { uint2 u; short4_t s; } c;
    c.u = v;
    return c.s;
}
__device__ __forceinline__ float16_t mfma8(uint2 a, uint2 b, float16_t acc) {
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(as_frag(a), as_frag(b), acc, 0, 0, 0);
}
// two floats rounded to nearest even BF16, the first in the low half
__device__ __forceinline__ unsigned pack_bf(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    union { b2 h; unsigned u; } c;
    c.h = __builtin_convertvector((f2){a, b}, b2);
    return c.u;
}
__device__ __forceinline__ float lo_bf(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_bf(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

// whole rows of a wavefront's tile (row 8 p + g, this lane's 16 bytes) to its LDS rows and back
__device__ __forceinline__ void rows_put(bf16_t *t, const uint4 (&v)[4], int g, int lane8) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint2 *q = reinterpret_cast<uint2 *>(t + (8 * p + g) * kRow + 8 * lane8);
        q[0] = make_uint2(v[p].x, v[p].y);
        q[1] = make_uint2(v[p].z, v[p].w);
    }
}
__device__ __forceinline__ uint4 row_get(const bf16_t *t, int p, int g, int lane8) {
    const uint2 *q = reinterpret_cast<const uint2 *>(t + (8 * p + g) * kRow + 8 * lane8);
    return make_uint4(q[0].x, q[0].y, q[1].x, q[1].y);
}

// keeps one wavefront's LDS accesses in program order (the LDS runs them in order)
__device__ __forceinline__ void wave_order() { asm volatile("" ::: "memory"); }

// Neighbour sums: 8 lanes per node (lane8 the lane among them), 8 features each, so
// a gather is one cache line.  The arithmetic bounds it (two instructions per
// feature and neighbour), so the rest is kept small: a lane's list entries are row
// offsets, shared among the node's lanes by a swizzle, and entries past the list
// point at the array's zero row (row N) instead of being masked.
// BIG: row offsets past 32 bits (more than 33 554 430 nodes).
template <bool BIG>
struct Nbrs {
    using Off = typename std::conditional<BIG, int, unsigned>::type;  // BIG: row index, else byte offset of the row
    int k0, k1;
    Off j0, j1;   // this lane's entries of the first two groups of eight neighbours
    float w0, w1;
};
template <bool BIG>
__device__ __forceinline__ void nbrs_ptr(Nbrs<BIG> &b, int m, const int *__restrict__ ia) {
    b.k0 = ia[m];
    b.k1 = ia[m + 1];
}
template <bool BIG>
__device__ __forceinline__ typename Nbrs<BIG>::Off nbr_off(int j) {
    return BIG ? j : (typename Nbrs<BIG>::Off)j << 7;
}
// entry k of the list, and with ideg (1 / degree) its weight
template <bool BIG>
__device__ __forceinline__ void nbrs_entry(typename Nbrs<BIG>::Off &j, float &w, const Nbrs<BIG> &b, int k, int N,
                                           const int *__restrict__ ja, const float *__restrict__ ideg) {
    const int e = b.k0 + k < b.k1 ? ja[b.k0 + k] : N;
    j = nbr_off<BIG>(e);
    w = ideg && e < N ? ideg[e] : 0.f;
}

template <int U, typename T>
__device__ __forceinline__ T swizzle8(T v) {  // lane U of each group of eight
    union { T t; int i; } c;
    c.t = v;
    c.i = __builtin_amdgcn_ds_swizzle(c.i, 0x18 | (U << 5));
    return c.t;
}
template <int U, bool BIG>
__device__ __forceinline__ uint4 nbr_row(typename Nbrs<BIG>::Off j, unsigned lane_off, const bf16_t *__restrict__ H) {
    const auto ju = swizzle8<U>(j);
    const char *base = reinterpret_cast<const char *>(H);
    if (BIG) return *reinterpret_cast<const uint4 *>(base + (size_t)ju * (2 * kH) + lane_off);
    return *reinterpret_cast<const uint4 *>(base + ((unsigned)ju + lane_off));
}
template <bool BIG>
__device__ __forceinline__ void nbrs_gather(uint4 (&v)[8], typename Nbrs<BIG>::Off j, unsigned lane_off,
                                            const bf16_t *__restrict__ H) {
    v[0] = nbr_row<0, BIG>(j, lane_off, H);
    v[1] = nbr_row<1, BIG>(j, lane_off, H);
    v[2] = nbr_row<2, BIG>(j, lane_off, H);
    v[3] = nbr_row<3, BIG>(j, lane_off, H);
    v[4] = nbr_row<4, BIG>(j, lane_off, H);
    v[5] = nbr_row<5, BIG>(j, lane_off, H);
    v[6] = nbr_row<6, BIG>(j, lane_off, H);
    v[7] = nbr_row<7, BIG>(j, lane_off, H);
}
template <bool SCALED>
__device__ __forceinline__ void nbr_add(float (&s)[8], uint4 v, float w) {
    const unsigned d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        s[2 * q] += SCALED ? w * lo_bf(d[q]) : lo_bf(d[q]);
        s[2 * q + 1] += SCALED ? w * hi_bf(d[q]) : hi_bf(d[q]);
    }
}
template <bool SCALED>
__device__ __forceinline__ void nbrs_add(float (&s)[8], const uint4 (&v)[8], float w) {
    nbr_add<SCALED>(s, v[0], swizzle8<0>(w));
    nbr_add<SCALED>(s, v[1], swizzle8<1>(w));
    nbr_add<SCALED>(s, v[2], swizzle8<2>(w));
    nbr_add<SCALED>(s, v[3], swizzle8<3>(w));
    nbr_add<SCALED>(s, v[4], swizzle8<4>(w));
    nbr_add<SCALED>(s, v[5], swizzle8<5>(w));
    nbr_add<SCALED>(s, v[6], swizzle8<6>(w));
    nbr_add<SCALED>(s, v[7], swizzle8<7>(w));
}
// s = sum over the list, in its order, in FP32; SCALED: each row times its weight
template <bool SCALED, bool BIG>
__device__ __forceinline__ void sum_neighbours(const Nbrs<BIG> &b, int N, int lane8, const int *__restrict__ ja,
                                               const float *__restrict__ ideg, const bf16_t *__restrict__ H,
                                               float (&s)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] = 0.f;
    const int n = b.k1 - b.k0;
    const unsigned lo = 16 * lane8;
    uint4 v0[8], v1[8];
    // uniform: list entries that no node of the wavefront has are skipped
    const bool more = __any(n > 8), m10 = __any(n > 10), m12 = __any(n > 12), m14 = __any(n > 14);
    nbrs_gather<BIG>(v0, b.j0, lo, H);
    if (more) {
        v1[0] = nbr_row<0, BIG>(b.j1, lo, H);
        v1[1] = nbr_row<1, BIG>(b.j1, lo, H);
    }
    if (m10) {
        v1[2] = nbr_row<2, BIG>(b.j1, lo, H);
        v1[3] = nbr_row<3, BIG>(b.j1, lo, H);
    }
    if (m12) {
        v1[4] = nbr_row<4, BIG>(b.j1, lo, H);
        v1[5] = nbr_row<5, BIG>(b.j1, lo, H);
    }
    if (m14) {
        v1[6] = nbr_row<6, BIG>(b.j1, lo, H);
        v1[7] = nbr_row<7, BIG>(b.j1, lo, H);
    }
    nbrs_add<SCALED>(s, v0, b.w0);
    if (more) {
        nbr_add<SCALED>(s, v1[0], swizzle8<0>(b.w1));
        nbr_add<SCALED>(s, v1[1], swizzle8<1>(b.w1));
    }
    if (m10) {
        nbr_add<SCALED>(s, v1[2], swizzle8<2>(b.w1));
        nbr_add<SCALED>(s, v1[3], swizzle8<3>(b.w1));
    }
    if (m12) {
        nbr_add<SCALED>(s, v1[4], swizzle8<4>(b.w1));
        nbr_add<SCALED>(s, v1[5], swizzle8<5>(b.w1));
    }
    if (m14) {
        nbr_add<SCALED>(s, v1[6], swizzle8<6>(b.w1));
        nbr_add<SCALED>(s, v1[7], swizzle8<7>(b.w1));
    }
    for (int k = 16; __any(k < n); k += 8) {
        typename Nbrs<BIG>::Off j;
        float w;
        nbrs_entry<BIG>(j, w, b, k + lane8, N, ja, SCALED ? ideg : nullptr);
        nbrs_gather<BIG>(v0, j, lo, H);
        nbrs_add<SCALED>(s, v0, w);
    }
}

// Workgroup b's tiles of 128 nodes: XCD b % 8 takes a contiguous eighth of the
// tiles (its L2 then holds the neighbours its tiles share), its workgroups side by
// side in it.
struct TileRange {
    int first, last, step;
};
__device__ __forceinline__ TileRange tile_range(int tiles) {
    if (gridDim.x < 64) return {(int)blockIdx.x, tiles, (int)gridDim.x};
    const int x = blockIdx.x & 7, lo = (int)((long)tiles * x / 8), hi = (int)((long)tiles * (x + 1) / 8);
    return {lo + (int)(blockIdx.x >> 3), hi, (int)((gridDim.x + 7 - x) >> 3)};
}

// W^T (64 x 64, row n = output feature) into padded LDS rows
__device__ __forceinline__ void stage_weights(const bf16_t *__restrict__ wt, bf16_t *lds) {
    for (int i = threadIdx.x; i < kH * kH / 8; i += blockDim.x) {
        const uint4 v = reinterpret_cast<const uint4 *>(wt)[i];
        uint2 *p = reinterpret_cast<uint2 *>(lds + (i >> 3) * kRow + (i & 7) * 8);
        p[0] = make_uint2(v.x, v.y);
        p[1] = make_uint2(v.z, v.w);
    }
}

// ---- forward ----------------------------------------------------------------------
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));  // a caller's array: any float alignment

// H0 = bf16(relu(bf16(x) We + be)) from the FP32 features; TRAIN keeps bf16(x).
template <bool TRAIN>
__global__ void __launch_bounds__(256) mp_encode(int N, const float *__restrict__ x, const bf16_t *__restrict__ We,
                                                 const float *__restrict__ be, bf16_t *__restrict__ X0,
                                                 bf16_t *__restrict__ H) {
    const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5;
    uint2 w[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            unsigned b[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = We[(8 * s + 4 * h + j) * kH + 32 * t + i];
            w[s][t] = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
        }
    for (int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 32; r0 < N; r0 += gridDim.x * 128) {
        const int row = min(r0 + i, N - 1);
        float16_t acc[2] = {{0}, {0}};
        uint2 f[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float4u v = *reinterpret_cast<const float4u *>(x + (size_t)row * kF + 8 * s + 4 * h);
            f[s] = make_uint2(pack_bf(v.x, v.y), pack_bf(v.z, v.w));
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = mfma8(w[s][t], f[s], acc[t]);
        }
        if (TRAIN) {
            const uint4 v = frag_to_row(f[0], f[1]);
            if (r0 + i < N) *reinterpret_cast<uint4 *>(X0 + (size_t)row * kF + 8 * h) = v;
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            uint2 o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int s = 2 * p + e, t = s >> 2, q = s & 3;
                const float4 b = *reinterpret_cast<const float4 *>(be + 8 * s + 4 * h);
                o[e] = make_uint2(pack_bf(fmaxf(acc[t][4 * q] + b.x, 0.f), fmaxf(acc[t][4 * q + 1] + b.y, 0.f)),
                                  pack_bf(fmaxf(acc[t][4 * q + 2] + b.z, 0.f), fmaxf(acc[t][4 * q + 3] + b.w, 0.f)));
            }
            const uint4 v = frag_to_row(o[0], o[1]);
            if (r0 + i < N) *reinterpret_cast<uint4 *>(H + (size_t)row * kH + 16 * p + 8 * h) = v;
        }
    }
}

// One layer: A = bf16(neighbour mean of H), Z = H W1 + A W2 + b, H' = bf16(H + relu(Z)).
// A wavefront takes 32 nodes: it sums their neighbours eight lanes to a node (whole
// rows, so each gather is a cache line), passes the means through its own LDS rows
// into fragments, and keeps everything else in registers.  TRAIN also stores A and
// bf16(Z) for the backward pass; LAST decodes y = H' . Wd + bd, and without TRAIN
// H' is not stored then.  The neighbour sums bound it: their
// instructions (1480 per 32 nodes, 85 us of issue at 1 024 000 nodes) and the L1's
// 64 bytes per clock (14 rows of 128 bytes per node, 75 us).  1 024 000 nodes: 140 us a
// layer, 115 us the last (no H'); a kernel for the means and one for the products
// took 425 us.
template <bool TRAIN, bool LAST, bool BIG>
__global__ void __launch_bounds__(256, 4) mp_layer(int N, const int *__restrict__ ia, const int *__restrict__ ja,
                                                   const float *__restrict__ ideg, const bf16_t *__restrict__ H, const bf16_t *__restrict__ wt1,
                                                   const bf16_t *__restrict__ wt2, const float *__restrict__ bias,
                                                   bf16_t *__restrict__ A, bf16_t *__restrict__ Z,
                                                   bf16_t *__restrict__ Hout, const bf16_t *__restrict__ wd,
                                                   const float *__restrict__ bd, float *__restrict__ y) {
    __shared__ __align__(16) bf16_t w[2][kH * kRow];
    __shared__ __align__(16) bf16_t mean[4][32 * kRow];
    __shared__ __align__(16) float sb[2 * kH];  // bias, decoder weights
    stage_weights(wt1, w[0]);
    stage_weights(wt2, w[1]);
    if (threadIdx.x < kH) {
        sb[threadIdx.x] = bias[threadIdx.x];
        sb[kH + threadIdx.x] = LAST ? bf2f(wd[threadIdx.x]) : 0.f;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5, g = lane >> 3, lane8 = lane & 7;
    bf16_t *const am = mean[threadIdx.x >> 6];
    const TileRange tr = tile_range((N + 127) / 128);
    // the lists of the tile's four passes of 8 nodes, fetched a tile ahead
    Nbrs<BIG> nb[4];
    const int r1 = tr.first * 128 + (threadIdx.x >> 6) * 32;
#pragma unroll
    for (int p = 0; p < 4; ++p) nbrs_ptr(nb[p], min(r1 + 8 * p + g, N - 1), ia);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        nbrs_entry<BIG>(nb[p].j0, nb[p].w0, nb[p], lane8, N, ja, nullptr);
        nbrs_entry<BIG>(nb[p].j1, nb[p].w1, nb[p], 8 + lane8, N, ja, nullptr);
    }
    for (int tile = tr.first; tile < tr.last; tile += tr.step) {
        const int r0 = tile * 128 + (threadIdx.x >> 6) * 32;
        if (r0 >= N) break;  // this wavefront's later tiles are past the end too
        const int row = min(r0 + i, N - 1);
        uint4 own[4];
#pragma unroll
        for (int p = 0; p < 4; ++p)
            own[p] = *reinterpret_cast<const uint4 *>(H + (size_t)min(r0 + 8 * p + g, N - 1) * kH + 8 * lane8);
        uint2 f[8];
        rows_put(am, own, g, lane8);
        wave_order();
#pragma unroll
        for (int s = 0; s < 8; ++s) f[s] = *reinterpret_cast<const uint2 *>(am + i * kRow + 8 * s + 4 * h);
        wave_order();
        const int rn = r0 + tr.step * 128;  // the next tile's lists: pointers now, indices after the sums
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int m = r0 + 8 * p + g;
            float s[8];
            sum_neighbours<false, BIG>(nb[p], N, lane8, ja, nullptr, H, s);
            const float inv = ideg[min(m, N - 1)];
            nbrs_ptr(nb[p], min(rn + 8 * p + g, N - 1), ia);
            const uint4 v = make_uint4(pack_bf(s[0] * inv, s[1] * inv), pack_bf(s[2] * inv, s[3] * inv),
                                       pack_bf(s[4] * inv, s[5] * inv), pack_bf(s[6] * inv, s[7] * inv));
            uint2 *o = reinterpret_cast<uint2 *>(am + (8 * p + g) * kRow + 8 * lane8);
            o[0] = make_uint2(v.x, v.y);
            o[1] = make_uint2(v.z, v.w);
            if (TRAIN && m < N) *reinterpret_cast<uint4 *>(A + (size_t)m * kH + 8 * lane8) = v;
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            nbrs_entry<BIG>(nb[p].j0, nb[p].w0, nb[p], lane8, N, ja, nullptr);
            nbrs_entry<BIG>(nb[p].j1, nb[p].w1, nb[p], 8 + lane8, N, ja, nullptr);
        }
        wave_order();
        float16_t acc[2] = {{0}, {0}};
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = mfma8(*reinterpret_cast<const uint2 *>(w[0] + (32 * t + i) * kRow + 8 * s + 4 * h), f[s], acc[t]);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint2 a = *reinterpret_cast<const uint2 *>(am + i * kRow + 8 * s + 4 * h);
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = mfma8(*reinterpret_cast<const uint2 *>(w[1] + (32 * t + i) * kRow + 8 * s + 4 * h), a, acc[t]);
        }
        wave_order();  // the next tile's means overwrite am
        float dot = 0.f;
        uint2 oz[TRAIN ? 8 : 1];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int t = s >> 2, q = s & 3;
            const float4 b = *reinterpret_cast<const float4 *>(sb + 8 * s + 4 * h);
            const float z0 = acc[t][4 * q] + b.x, z1 = acc[t][4 * q + 1] + b.y;
            const float z2 = acc[t][4 * q + 2] + b.z, z3 = acc[t][4 * q + 3] + b.w;
            if (TRAIN) oz[s] = make_uint2(pack_bf(z0, z1), pack_bf(z2, z3));
            const uint2 oh = make_uint2(pack_bf(lo_bf(f[s].x) + fmaxf(z0, 0.f), hi_bf(f[s].x) + fmaxf(z1, 0.f)),
                                        pack_bf(lo_bf(f[s].y) + fmaxf(z2, 0.f), hi_bf(f[s].y) + fmaxf(z3, 0.f)));
            if (TRAIN || !LAST) *reinterpret_cast<uint2 *>(am + i * kRow + 8 * s + 4 * h) = oh;
            if (LAST) {
                const float4 d = *reinterpret_cast<const float4 *>(sb + kH + 8 * s + 4 * h);
                dot += lo_bf(oh.x) * d.x;
                dot += hi_bf(oh.x) * d.y;
                dot += lo_bf(oh.y) * d.z;
                dot += hi_bf(oh.y) * d.w;
            }
        }
        wave_order();
        // out as whole rows
        if (TRAIN || !LAST)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint4 v = row_get(am, p, g, lane8);
                const int m = r0 + 8 * p + g;
                if (m < N) *reinterpret_cast<uint4 *>(Hout + (size_t)m * kH + 8 * lane8) = v;
            }
        wave_order();
        if (TRAIN) {
#pragma unroll
            for (int s = 0; s < 8; ++s) *reinterpret_cast<uint2 *>(am + i * kRow + 8 * s + 4 * h) = oz[s];
            wave_order();
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint4 v = row_get(am, p, g, lane8);
                const int m = r0 + 8 * p + g;
                if (m < N) *reinterpret_cast<uint4 *>(Z + (size_t)m * kH + 8 * lane8) = v;
            }
            wave_order();
        }
        if (LAST) {
            dot += __shfl_xor(dot, 32);
            if (h == 0 && r0 + i < N) y[row] = dot + bd[0];
        }
    }
}

// ---- backward ---------------------------------------------------------------------
// The loss and the decoder at one node: d = y - t, dy = 2 d / N (dH = dy Wd).
// One layer, from the last to the first: dH (FP32) becomes complete (DEC: the
// decoder's, dy Wd; otherwise the stored one plus the adjoint of the next layer's
// neighbour mean, sum_j dA_j / deg_j), dZ = bf16(dH where Z > 0) takes Z's place,
// dA = bf16(dZ W2^T) goes out for the layer before, and dH + dZ W1^T is stored.
// Tiles, fragments and gathers as mp_layer's; dZ passes to fragments, and the
// product dZ W1^T back to whole rows, through the wavefront's LDS rows.
// DEC also leaves block partials of the loss, dWd = H^T dy and dbd = sum dy.
// Bound as mp_layer.  194 672 nodes: 59 us, the last layer (DEC) 33 us; the mask,
// products and adjoint mean as kernels of their own took 133 us a layer.
constexpr int kRowF = 68;  // floats per LDS row of 64

template <bool DEC, bool BIG>
__global__ void __launch_bounds__(256, 3) mp_back(int N, const int *__restrict__ ia, const int *__restrict__ ja,
                                               const float *__restrict__ ideg, const bf16_t *__restrict__ w1,
                                               const bf16_t *__restrict__ w2, const bf16_t *__restrict__ dAn,
                                               bf16_t *__restrict__ Z, bf16_t *__restrict__ dA,
                                               float *__restrict__ dH, const bf16_t *__restrict__ H,
                                               const bf16_t *__restrict__ wd, const float *__restrict__ y,
                                               const float *__restrict__ t, float *__restrict__ part,
                                               double *__restrict__ lpart) {
    __shared__ __align__(16) bf16_t w[2][kH * kRow];
    __shared__ __align__(16) float rows[4][32 * kRowF];  // dZ as BF16 rows first, then dZ W1^T
    stage_weights(w1, w[0]);
    stage_weights(w2, w[1]);
    __syncthreads();
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63, i = lane & 31, h = lane >> 5, g = lane >> 3, lane8 = lane & 7;
    bf16_t *const dz = reinterpret_cast<bf16_t *>(rows[wave]);
    float *const rf = rows[wave];
    float wdf[8], gwd[8], gbd = 0.f;
    double loss = 0.;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        wdf[q] = DEC ? bf2f(wd[8 * lane8 + q]) : 0.f;
        gwd[q] = 0.f;
    }
    const TileRange tr = tile_range((N + 127) / 128);
    Nbrs<BIG> nb[4];
    if (!DEC) {
        const int r1 = tr.first * 128 + wave * 32;
#pragma unroll
        for (int p = 0; p < 4; ++p) nbrs_ptr(nb[p], min(r1 + 8 * p + g, N - 1), ia);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            nbrs_entry<BIG>(nb[p].j0, nb[p].w0, nb[p], lane8, N, ja, ideg);
            nbrs_entry<BIG>(nb[p].j1, nb[p].w1, nb[p], 8 + lane8, N, ja, ideg);
        }
    }
    for (int tile = tr.first; tile < tr.last; tile += tr.step) {
        const int r0 = tile * 128 + wave * 32;
        if (r0 >= N) break;
        const int rn = r0 + tr.step * 128;
        float d[4][8];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int m = r0 + 8 * p + g, mc = min(m, N - 1);
            const size_t o = (size_t)mc * kH + 8 * lane8;
            const uint4 z = *reinterpret_cast<const uint4 *>(Z + o);
            if (DEC) {
                const uint4 hv = *reinterpret_cast<const uint4 *>(H + o);
                const float e = y[mc] - t[mc], dy = m < N ? 2.f * e / (float)N : 0.f;
                const unsigned hu[4] = {hv.x, hv.y, hv.z, hv.w};
#pragma unroll
                for (int q = 0; q < 8; ++q) d[p][q] = dy * wdf[q];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    gwd[2 * q] += lo_bf(hu[q]) * dy;
                    gwd[2 * q + 1] += hi_bf(hu[q]) * dy;
                }
                if (lane8 == 0 && m < N) {
                    gbd += dy;
                    loss += (double)e * e;
                }
            } else {
                const float4 a = *reinterpret_cast<const float4 *>(dH + o), b = *reinterpret_cast<const float4 *>(dH + o + 4);
                float s[8];
                sum_neighbours<true, BIG>(nb[p], N, lane8, ja, ideg, dAn, s);
                nbrs_ptr(nb[p], min(rn + 8 * p + g, N - 1), ia);
                d[p][0] = a.x + s[0]; d[p][1] = a.y + s[1]; d[p][2] = a.z + s[2]; d[p][3] = a.w + s[3];
                d[p][4] = b.x + s[4]; d[p][5] = b.y + s[5]; d[p][6] = b.z + s[6]; d[p][7] = b.w + s[7];
            }
            const unsigned zu[4] = {z.x, z.y, z.z, z.w};
            unsigned v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                v[q] = pack_bf(lo_bf(zu[q]) > 0.f ? d[p][2 * q] : 0.f, hi_bf(zu[q]) > 0.f ? d[p][2 * q + 1] : 0.f);
            uint2 *q = reinterpret_cast<uint2 *>(dz + (8 * p + g) * kRow + 8 * lane8);
            q[0] = make_uint2(v[0], v[1]);
            q[1] = make_uint2(v[2], v[3]);
            if (m < N) *reinterpret_cast<uint4 *>(Z + o) = make_uint4(v[0], v[1], v[2], v[3]);
        }
        if (!DEC) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                nbrs_entry<BIG>(nb[p].j0, nb[p].w0, nb[p], lane8, N, ja, ideg);
                nbrs_entry<BIG>(nb[p].j1, nb[p].w1, nb[p], 8 + lane8, N, ja, ideg);
            }
        }
        wave_order();
        uint2 f[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) f[s] = *reinterpret_cast<const uint2 *>(dz + i * kRow + 8 * s + 4 * h);
        wave_order();
        float16_t acc[2] = {{0}, {0}};
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                acc[q] = mfma8(*reinterpret_cast<const uint2 *>(w[0] + (32 * q + i) * kRow + 8 * s + 4 * h), f[s], acc[q]);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int q = 4 * (s & 3);
            *reinterpret_cast<float4 *>(rf + i * kRowF + 8 * s + 4 * h) =
                make_float4(acc[s >> 2][q], acc[s >> 2][q + 1], acc[s >> 2][q + 2], acc[s >> 2][q + 3]);
        }
        wave_order();
        acc[0] = float16_t{0};
        acc[1] = float16_t{0};
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                acc[q] = mfma8(*reinterpret_cast<const uint2 *>(w[1] + (32 * q + i) * kRow + 8 * s + 4 * h), f[s], acc[q]);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int m = r0 + 8 * p + g;
            const float4 a = *reinterpret_cast<const float4 *>(rf + (8 * p + g) * kRowF + 8 * lane8);
            const float4 b = *reinterpret_cast<const float4 *>(rf + (8 * p + g) * kRowF + 8 * lane8 + 4);
            if (m < N) {
                float4 *o = reinterpret_cast<float4 *>(dH + (size_t)m * kH + 8 * lane8);
                o[0] = make_float4(d[p][0] + a.x, d[p][1] + a.y, d[p][2] + a.z, d[p][3] + a.w);
                o[1] = make_float4(d[p][4] + b.x, d[p][5] + b.y, d[p][6] + b.z, d[p][7] + b.w);
            }
        }
        wave_order();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int q = 4 * (s & 3);
            *reinterpret_cast<uint2 *>(dz + i * kRow + 8 * s + 4 * h) =
                make_uint2(pack_bf(acc[s >> 2][q], acc[s >> 2][q + 1]), pack_bf(acc[s >> 2][q + 2], acc[s >> 2][q + 3]));
        }
        wave_order();
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint4 v = row_get(dz, p, g, lane8);
            const int m = r0 + 8 * p + g;
            if (m < N) *reinterpret_cast<uint4 *>(dA + (size_t)m * kH + 8 * lane8) = v;
        }
        wave_order();
    }
    if (DEC) {
        // the lanes of a wavefront that hold the same features, then the four wavefronts
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) {
#pragma unroll
            for (int q = 0; q < 8; ++q) gwd[q] += __shfl_xor(gwd[q], off);
            gbd += __shfl_xor(gbd, off);
            loss += __shfl_xor(loss, off);
        }
        __syncthreads();
        float *const red = rows[0];
        double *const lred = reinterpret_cast<double *>(rows[1]);
        if (g == 0)
#pragma unroll
            for (int q = 0; q < 8; ++q) red[wave * (kH + 1) + 8 * lane8 + q] = gwd[q];
        if (lane == 0) {
            red[wave * (kH + 1) + kH] = gbd;
            lred[wave] = loss;
        }
        __syncthreads();
        if (threadIdx.x <= kH) {
            float s = 0.f;
            for (int k = 0; k < 4; ++k) s += red[k * (kH + 1) + threadIdx.x];
            part[(size_t)blockIdx.x * (kH + 1) + threadIdx.x] = s;
        }
        if (threadIdx.x == 0) lpart[blockIdx.x] = lred[0] + lred[1] + lred[2] + lred[3];
    }
}

// The encoder's dZ0 = bf16(dH0 where H0 > 0), dH0 completed by layer 0's adjoint
// mean.  A wavefront takes 8 nodes: 32 us at 194 672 nodes, 40 us with 32 nodes at a
// time and the next ones' lists in flight (fewer wavefronts to hide the gathers).
template <bool BIG>
__global__ void __launch_bounds__(256) mp_back_encoder(int N, const int *__restrict__ ia, const int *__restrict__ ja,
                                                       const float *__restrict__ ideg, const bf16_t *__restrict__ dAn,
                                                       const float *__restrict__ dH, const bf16_t *__restrict__ H0,
                                                       bf16_t *__restrict__ dZ) {
    const int lane8 = threadIdx.x & 7;
    const long m = blockIdx.x * 32L + (threadIdx.x >> 3);
    const int mc = (int)min(m, (long)N - 1);
    const size_t o = (size_t)mc * kH + 8 * lane8;
    const uint4 hv = *reinterpret_cast<const uint4 *>(H0 + o);
    const float4 a = *reinterpret_cast<const float4 *>(dH + o), b = *reinterpret_cast<const float4 *>(dH + o + 4);
    Nbrs<BIG> nb;
    nbrs_ptr(nb, mc, ia);
    nbrs_entry<BIG>(nb.j0, nb.w0, nb, lane8, N, ja, ideg);
    nbrs_entry<BIG>(nb.j1, nb.w1, nb, 8 + lane8, N, ja, ideg);
    float s[8];
    sum_neighbours<true, BIG>(nb, N, lane8, ja, ideg, dAn, s);
    const float d[8] = {a.x + s[0], a.y + s[1], a.z + s[2], a.w + s[3], b.x + s[4], b.y + s[5], b.z + s[6], b.w + s[7]};
    const unsigned hu[4] = {hv.x, hv.y, hv.z, hv.w};
    unsigned v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        v[q] = pack_bf(lo_bf(hu[q]) > 0.f ? d[2 * q] : 0.f, hi_bf(hu[q]) > 0.f ? d[2 * q + 1] : 0.f);
    if (m < N) *reinterpret_cast<uint4 *>(dZ + o) = make_uint4(v[0], v[1], v[2], v[3]);
}

// ---- weight gradients -------------------------------------------------------------
// Per layer (blockIdx.y) G1 = H^T dZ, G2 = A^T dZ (64 x 64) and the column sums of
// dZ: block partials over this block's rows.  The rows are the matrix cores'
// reduction dimension.  A workgroup stages 64 rows of dZ, H and A in LDS (16 bytes
// per lane; two buffers, and the loads of the next 128 rows in flight meanwhile, so
// its barrier waits for LDS accesses only); wavefronts 0 and 1 form G1, 2 and 3 G2,
// each over half of the rows, reading both operands transposed (ds_read_b64_tr_b16:
// each lane four rows of one column).  Memory bounds it (each row read once).
// 194 672 nodes, three layers: 48 us (225 MB of rows: 4.7 TB/s), from
// 7 launches of 24 us and 4 of 32 us for the sums; one wavefront per SIMD holding both
// gradients took 151 us, one gradient per wavefront with rows of its own 93 us.
// ENC: the encoder's, X0 (N x 16) in H's place and no A, a quarter of the rows per
// wavefront.
constexpr int kGradOut = 2 * kH * kH + kH;  // values per layer: G1, G2, column sums
constexpr int kEncOut = kF * kH + kH;

__device__ __forceinline__ uint2 read_tr(const bf16_t *tile, int row, int col, int lane) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    // 16 lanes read 4 rows of 16 columns and get, each, 4 rows of their own column
    const int c = lane & 15;
    const bf16_t *p = tile + (row + 4 * (lane >> 5) + (c >> 2)) * kRow + col + 16 * ((lane >> 4) & 1) + 4 * (c & 3);
    union { s4 s; uint2 u; } r;
    r.s = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p);
    return r.u;
}

// workgroup barrier for LDS data: global loads issued ahead stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <bool ENC>
__global__ void __launch_bounds__(256) mp_wgrad(int N, long stride, const bf16_t *__restrict__ X, long zstride,
                                                const bf16_t *__restrict__ A, const bf16_t *__restrict__ D,
                                                float *__restrict__ part) {
    constexpr int NM = ENC ? 1 : 2;                    // 32-feature tiles of the first operand
    constexpr int kRows = 64, kS = ENC ? 2 : 4;        // rows per step; K steps of 8 per wavefront
    constexpr int kOut = ENC ? kEncOut : kGradOut;
    __shared__ __align__(16) bf16_t tiles[2][(ENC ? 2 : 3) * kRows * kRow];
    float *const red = reinterpret_cast<float *>(tiles);  // after the rows
    static_assert(sizeof(tiles) >= sizeof(float) * kOut, "the block's sums take the tiles' place");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, h = lane >> 5;
    X += (size_t)blockIdx.y * stride;
    D += (size_t)blockIdx.y * zstride;
    if (!ENC) A += (size_t)blockIdx.y * zstride;
    const int which = ENC ? 0 : wave >> 1, rw = ENC ? 16 * wave : 32 * (wave & 1);
    float16_t acc[NM][2];
#pragma unroll
    for (int a = 0; a < NM; ++a) acc[a][0] = acc[a][1] = float16_t{0};
    float cs[2] = {0.f, 0.f};
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    const int rr = tid >> 3, c = 8 * (tid & 7);        // rows rr, rr + 32, features c ..
    const int re = (tid & 127) >> 1, ce = 8 * (tid & 1);  // ENC's first operand
    struct Rows {
        uint4 d[2], x[2], a[2];
    };
    auto load = [&](Rows &q, int r0) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int r = r0 + rr + 32 * p;
            const size_t o = (size_t)r * kH + c;
            q.d[p] = q.x[p] = q.a[p] = zero;
            if (r < N) {
                q.d[p] = *reinterpret_cast<const uint4 *>(D + o);
                if (!ENC) {
                    q.x[p] = *reinterpret_cast<const uint4 *>(X + o);
                    q.a[p] = *reinterpret_cast<const uint4 *>(A + o);
                }
            }
        }
        if (ENC && r0 + re < N) q.x[0] = *reinterpret_cast<const uint4 *>(X + (size_t)(r0 + re) * kF + ce);
    };
    auto put = [&](bf16_t *t, int row, int col, uint4 v) {
        uint2 *q = reinterpret_cast<uint2 *>(t + row * kRow + col);
        q[0] = make_uint2(v.x, v.y);
        q[1] = make_uint2(v.z, v.w);
    };
    auto step = [&](const Rows &q, bf16_t *t) {
        bf16_t *const td = t, *const tx = t + kRows * kRow, *const ta = tx + kRows * kRow;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            put(td, rr + 32 * p, c, q.d[p]);
            if (!ENC) {
                put(tx, rr + 32 * p, c, q.x[p]);
                put(ta, rr + 32 * p, c, q.a[p]);
            }
        }
        if (ENC) put(tx, re, (tid < 128 ? 0 : kF) + ce, tid < 128 ? q.x[0] : zero);  // zeros for features 16 .. 31
        lds_barrier();
        const bf16_t *const tm = which ? ta : tx;
#pragma unroll
        for (int s = 0; s < kS; ++s) {
            const int r = rw + 8 * s;
            const uint2 d0 = read_tr(td, r, 0, lane), d1 = read_tr(td, r, 32, lane);
            if (ENC || which) {
                cs[0] += (lo_bf(d0.x) + hi_bf(d0.x)) + (lo_bf(d0.y) + hi_bf(d0.y));
                cs[1] += (lo_bf(d1.x) + hi_bf(d1.x)) + (lo_bf(d1.y) + hi_bf(d1.y));
            }
#pragma unroll
            for (int a = 0; a < NM; ++a) {
                const uint2 m = read_tr(tm, r, 32 * a, lane);
                acc[a][0] = mfma8(m, d0, acc[a][0]);
                acc[a][1] = mfma8(m, d1, acc[a][1]);
            }
        }
    };
    // a wavefront is at most one step ahead of another (the barrier), so two buffers do
    const int adv = gridDim.x * kRows;
    Rows q0, q1;
    int r0 = blockIdx.x * kRows;
    load(q0, r0);
    load(q1, r0 + adv);
    for (; r0 < N; r0 += 2 * adv) {
        step(q0, tiles[0]);
        load(q0, r0 + 2 * adv);
        if (r0 + adv < N) {  // uniform
            step(q1, tiles[1]);
            load(q1, r0 + 3 * adv);
        }
    }
    // the wavefronts' sums, one after another in LDS, then this block's partial
    __syncthreads();
    const int turns = ENC ? 4 : 2;
    for (int k = 0; k < turns; ++k) {
        if ((ENC ? wave : wave & 1) == k) {
#pragma unroll
            for (int a = 0; a < NM; ++a)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int m = 32 * a + (v >> 2) * 8 + 4 * h + (v & 3), n = 32 * u + i;
                        if (ENC && m >= kF) continue;
                        float *o = red + which * kH * kH + m * kH + n;
                        *o = k ? *o + acc[a][u][v] : acc[a][u][v];
                    }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const float q = cs[u] + __shfl_xor(cs[u], 32);
                float *o = red + (kOut - kH) + 32 * u + i;
                if (h == 0 && (ENC || which)) *o = k ? *o + q : q;
            }
        }
        __syncthreads();
    }
    float *const out = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kOut;
    for (int k = tid; k < kOut; k += 256) out[k] = red[k];
}

// The block partials summed into the gradients (in block order) and the loss.
// part: the encoder's (nb x kEncOut), the layers' (L x nb x kGradOut), the
// decoder's (nd x 65).  64 parameters per block, sixteen slices of the partials each:
// its time is the partials' latency, so few loads in a row per lane.
struct GradSrc {
    long o_Wd, np;  // decoder offset and count of the parameters
    int L, nb, nd, N;
};
__global__ void __launch_bounds__(1024) mp_gradsum(GradSrc gs, const float *__restrict__ part,
                                                   const double *__restrict__ lpart, float *__restrict__ G,
                                                   double *slot, double tag) {
    constexpr int kSlices = 16;
    __shared__ float red[kSlices][64];
    const int k = threadIdx.x & 63, c = threadIdx.x >> 6;
    const long q = blockIdx.x * 64L + k;
    const float *src = nullptr;
    int n = gs.nb, stride = kEncOut;
    if (q < kEncOut) src = part + q;  // We, be
    else if (q < gs.o_Wd) {
        const long e = q - kEncOut, l = e / kGradOut;
        src = part + (size_t)gs.nb * kEncOut + (size_t)l * gs.nb * kGradOut + (e - l * kGradOut);
        stride = kGradOut;
    } else if (q < gs.np) {
        src = part + (size_t)gs.nb * kEncOut + (size_t)gs.L * gs.nb * kGradOut + (q - gs.o_Wd);
        n = gs.nd;
        stride = kH + 1;
    }
    float s = 0.f;
    if (src) {
        const int per = (n + kSlices - 1) / kSlices, b1 = min(n, (c + 1) * per);
        for (int b = c * per; b < b1; b += 12) {
            float v[12];
#pragma unroll
            for (int u = 0; u < 12; ++u) v[u] = b + u < b1 ? src[(size_t)(b + u) * stride] : 0.f;
#pragma unroll
            for (int u = 0; u < 12; ++u) s += v[u];
        }
    }
    red[c][k] = s;
    __syncthreads();
    if (c == 0 && q < gs.np) {
        float v = red[0][k];
#pragma unroll
        for (int u = 1; u < kSlices; ++u) v += red[u][k];
        G[q] = v;
    }
    if (blockIdx.x == 0 && c == 1) {
        double v = 0.;
        for (int b = k; b < gs.nd; b += 64) v += lpart[b];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (k == 0 && slot) {
            slot[0] = v / gs.N;
            fvp::slot_post(slot, tag);
        }
    }
}

// The gradients to pinned host memory, then tag behind them (one workgroup: the tag
// follows every thread's stores).  A training pass that reads its loss and gradients
// was two copies and waits of the runtime's, about 20 us each with the queue idle;
// with both polled 194 672 nodes take 441 -> 415 us.
__global__ void __launch_bounds__(1024) mp_post_grads(long np, const float *__restrict__ g,
                                                      float *__restrict__ host, double *slot,
                                                      double tag) {
#pragma unroll 8
    for (long i = threadIdx.x; i < np; i += 1024) host[i] = g[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) fvp::slot_post(slot, tag);
}

// Set-up: 1 / degree (1 for a node without neighbours), the zero rows behind the layers
// of H and dA, Adam's moments and the gradients
__global__ void mp_init(int N, int layers, const int *__restrict__ ia, float *__restrict__ ideg, bf16_t *__restrict__ H,
                        bf16_t *__restrict__ dA, long np, float *__restrict__ m, float *__restrict__ v,
                        float *__restrict__ g) {
    const size_t layer = ((size_t)N + 1) * kH, end = (size_t)N * kH;
    const long step = (long)gridDim.x * blockDim.x, i0 = blockIdx.x * (long)blockDim.x + threadIdx.x;
    for (long i = i0; i < N; i += step) ideg[i] = 1.f / (float)max(1, ia[i + 1] - ia[i]);
    for (long i = i0; i < (layers + 3) * kH; i += step) {
        const int l = (int)(i / kH);
        (l <= layers ? H + l * layer : dA + (l - layers - 1) * layer)[end + i % kH] = 0;
    }
    for (long i = i0; i < np; i += step) m[i] = v[i] = g[i] = 0.f;
}

__global__ void f32_to_bf16(long n, const float *__restrict__ x, bf16_t *__restrict__ y) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// Adam on the FP32 master parameters, then their BF16 copy
__global__ void mp_adam(long n, float lr, float b1, float b2, float eps, float c1, float c2, float *__restrict__ p,
                        float *__restrict__ m, float *__restrict__ v, const float *__restrict__ g,
                        bf16_t *__restrict__ pb) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    pb[i] = f2bf(pi);
}

// W1, W2 of each layer (blockIdx.y = 2 l + which; w0: the first layer's W1 among the
// parameters) as they are and transposed
__global__ void mp_weights(const bf16_t *__restrict__ w0, bf16_t *__restrict__ wb, bf16_t *__restrict__ wt1,
                           bf16_t *__restrict__ wt2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, l = blockIdx.y >> 1, which = blockIdx.y & 1;
    if (i >= kH * kH) return;
    const bf16_t v = w0[(size_t)l * kGradOut + which * kH * kH + i];
    wb[(size_t)blockIdx.y * kH * kH + i] = v;
    (which ? wt2 : wt1)[(size_t)l * kH * kH + (i % kH) * kH + i / kH] = v;
}

inline int nb(long n, int bs) { return (int)((n + bs - 1) / bs); }

}  // namespace

struct fvp_mpnn {
    int device = 0, N = 0, L = 3;
    hipStream_t stream = nullptr, own_stream = nullptr;
    DevBuf<int> ia, ja;
    // parameters (FP32 master, BF16 copy, Adam moments, gradients), one flat layout:
    // We (16 x 64), be (64), per layer W1 (64 x 64), W2 (64 x 64), b (64), Wd (64), bd (1)
    long np = 0;
    long o_We = 0, o_be = 0, o_W1[kMaxLayers], o_W2[kMaxLayers], o_b[kMaxLayers], o_Wd = 0, o_bd = 0;
    DevBuf<float> p, m, v, g;
    DevBuf<unsigned short> pb, wt1, wt2, wb;  // BF16 copy, per layer: transposed W1, W2; W1 and W2 (aligned)
    long step = 0;
    // activations: H (L + 1) x (N + 1) x 64, each layer's last row zero (padding of the
    // neighbour sums); A, Z: L x N x 64 (the backward pass puts dZ in Z's place); dA:
    // two of (N + 1) x 64, last rows zero
    DevBuf<unsigned short> X0, H, A, Z, dZ, dA;
    DevBuf<float> y, dH, part, ideg;  // ideg: 1 / degree (1 for a node without neighbours)
    DevBuf<double> lpart;
    // results for the host, allocated on first use: the loss's and the gradients' slots,
    // and the gradients themselves (pinned)
    fvp::HostSlots host;
    float *hgrad = nullptr;
    size_t layer() const { return ((size_t)N + 1) * kH; }
    bool big() const { return (size_t)N + 1 > (size_t)1 << 25; }  // row offsets past 32 bits
    // Workgroups of the row kernels: as many as the device holds at once (four per CU
    // forward, three backward), each taking several tiles of 128 nodes (weights staged
    // once).  Backward every workgroup gets the same count as nearly as it goes (1521
    // tiles: 761 workgroups, 59 us a layer against 65 with 768 in two uneven rounds);
    // forward that measured slower (39 us against 36 with 1024).
    int forward_grid() const { return std::min((N + 127) / 128, 1024); }
    int back_grid() const {
        const int tiles = (N + 127) / 128, each = (tiles + 767) / 768;
        return (tiles + each - 1) / each;
    }
    // blocks of a layer's weight gradients: two per CU over all layers, 512 rows or more
    // each (a block's partial is as many bytes as 86 of its rows)
    int grad_blocks() const { return std::max(1, std::min(512 / L, (N + 511) / 512)); }
};

static int host_results(fvp_mpnn *m) { return m->host.p ? 0 : m->host.alloc(2); }

static void layout(fvp_mpnn *m) {
    long o = 0;
    m->o_We = o; o += kF * kH;
    m->o_be = o; o += kH;
    for (int l = 0; l < m->L; ++l) {
        m->o_W1[l] = o; o += kH * kH;
        m->o_W2[l] = o; o += kH * kH;
        m->o_b[l] = o; o += kH;
    }
    m->o_Wd = o; o += kH;
    m->o_bd = o; o += 1;
    m->np = o;
}

// the BF16 copies that the products read, from the BF16 parameters
static int refresh_weights(fvp_mpnn *m) {
    mp_weights<<<dim3(nb(kH * kH, 256), 2 * m->L), 256, 0, m->stream>>>(m->pb.p + m->o_W1[0], m->wb.p, m->wt1.p,
                                                                        m->wt2.p);
    FVP_HIP(hipGetLastError());
    return 0;
}

static int refresh_bf16(fvp_mpnn *m) {
    f32_to_bf16<<<nb(m->np, 256), 256, 0, m->stream>>>(m->np, m->p.p, m->pb.p);
    return refresh_weights(m);
}

// forward from the FP32 features x to y (N); TRAIN keeps every layer's activations
template <bool TRAIN, bool BIG>
static int forward_impl(fvp_mpnn *m, const float *x, float *y) {
    hipStream_t s = m->stream;
    const int N = m->N, g = m->forward_grid();
    const size_t NH = (size_t)N * kH, W = kH * kH;
    const bf16_t *pb = m->pb.p;
    mp_encode<TRAIN><<<g, 256, 0, s>>>(N, x, pb + m->o_We, m->p.p + m->o_be, m->X0.p, m->H.p);
    for (int l = 0; l < m->L; ++l) {
        auto layer = l + 1 < m->L ? mp_layer<TRAIN, false, BIG> : mp_layer<TRAIN, true, BIG>;
        layer<<<g, 256, 0, s>>>(N, m->ia.p, m->ja.p, m->ideg.p, m->H.p + l * m->layer(), m->wt1.p + l * W,
                                m->wt2.p + l * W, m->p.p + m->o_b[l], m->A.p + l * NH, m->Z.p + l * NH,
                                m->H.p + (l + 1) * m->layer(), pb + m->o_Wd, m->p.p + m->o_bd, y);
    }
    FVP_HIP(hipGetLastError());
    return 0;
}

// backward of the mean squared error of m->y against t; gradients to m->g, the loss to
// the host's slot, if given
template <bool BIG>
static int backward_impl(fvp_mpnn *m, const float *t, double *slot, double tag) {
    hipStream_t s = m->stream;
    const int N = m->N, L = m->L, g = m->back_grid(), gb = m->grad_blocks();
    const size_t NH = (size_t)N * kH, W = kH * kH;
    float *const pe = m->part.p, *const pl = pe + (size_t)gb * kEncOut, *const pd = pl + (size_t)L * gb * kGradOut;
    bf16_t *dA[2] = {m->dA.p, m->dA.p + m->layer()};
    for (int l = L - 1; l >= 0; --l) {
        auto back = l == L - 1 ? mp_back<true, BIG> : mp_back<false, BIG>;
        back<<<g, 256, 0, s>>>(N, m->ia.p, m->ja.p, m->ideg.p, m->wb.p + 2 * l * W, m->wb.p + (2 * l + 1) * W,
                               dA[(l + 1) & 1], m->Z.p + l * NH, dA[l & 1], m->dH.p, m->H.p + L * m->layer(),
                               m->pb.p + m->o_Wd, m->y.p, t, pd, m->lpart.p);
    }
    mp_back_encoder<BIG><<<nb(N, 32), 256, 0, s>>>(N, m->ia.p, m->ja.p, m->ideg.p, dA[0], m->dH.p, m->H.p, m->dZ.p);
    mp_wgrad<false><<<dim3(gb, L), 256, 0, s>>>(N, (long)m->layer(), m->H.p, (long)NH, m->A.p, m->Z.p, pl);
    mp_wgrad<true><<<gb, 256, 0, s>>>(N, 0, m->X0.p, 0, nullptr, m->dZ.p, pe);
    GradSrc gs{};
    gs.o_Wd = m->o_Wd;
    gs.np = m->np;
    gs.L = L;
    gs.nb = gb;
    gs.nd = g;
    gs.N = N;
    mp_gradsum<<<nb(m->np, 64), 1024, 0, s>>>(gs, m->part.p, m->lpart.p, m->g.p, slot, tag);
    FVP_HIP(hipGetLastError());
    return 0;
}

namespace fvp {
int mpnn_nodes(const fvp_mpnn *m) { return m ? m->N : -1; }
}  // namespace fvp

// ---- C ABI ---------------------------------------------------------------------------
extern "C" int fvp_mpnn_create(int device, int n_nodes, const int *ia, const int *ja, int layers,
                               unsigned long long seed, fvp_mpnn **out) {
    if (!ia || !ja || !out || n_nodes <= 0) { set_error("null argument"); return -1; }
    if (layers < 1 || layers > kMaxLayers) { set_error("layers must be 1..8"); return -1; }
    FVP_HIP(hipSetDevice(device));
    fvp_mpnn *m = new fvp_mpnn();
    m->device = device;
    m->N = n_nodes;
    m->L = layers;
    layout(m);
    if (hipStreamCreateWithFlags(&m->own_stream, hipStreamNonBlocking) != hipSuccess) {
        delete m;
        set_error("stream creation failed");
        return -1;
    }
    m->stream = m->own_stream;
    const size_t NH = (size_t)n_nodes * kH;
    // He / Glorot-like initial weights from a fixed-seed generator, zero biases
    std::vector<float> p0(m->np, 0.f);
    unsigned long long st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto gauss = [&]() {
        auto u = [&]() {
            st = st * 6364136223846793005ULL + 1442695040888963407ULL;
            return ((st >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        };
        const double a = u(), b = u();
        return std::sqrt(-2.0 * std::log(a)) * std::cos(6.283185307179586 * b);
    };
    for (long k = 0; k < kF * kH; ++k) p0[m->o_We + k] = (float)(gauss() * std::sqrt(2.0 / kF));
    for (int l = 0; l < layers; ++l)
        for (long k = 0; k < kH * kH; ++k) {
            p0[m->o_W1[l] + k] = (float)(gauss() * std::sqrt(1.0 / kH));
            p0[m->o_W2[l] + k] = (float)(gauss() * std::sqrt(1.0 / kH));
        }
    for (long k = 0; k < kH; ++k) p0[m->o_Wd + k] = (float)(gauss() * std::sqrt(1.0 / kH));
    const size_t nparts = (size_t)m->grad_blocks() * (kEncOut + (size_t)layers * kGradOut) +
                          (size_t)m->back_grid() * (kH + 1);
    if (m->ia.upload(ia, n_nodes + 1) || m->ja.upload(ja, ia[n_nodes]) || m->p.upload(p0.data(), m->np) ||
        m->m.alloc(m->np) || m->v.alloc(m->np) || m->g.alloc(m->np) || m->pb.alloc(m->np) ||
        m->wt1.alloc((size_t)layers * kH * kH) || m->wt2.alloc((size_t)layers * kH * kH) ||
        m->wb.alloc(2 * (size_t)layers * kH * kH) || m->ideg.alloc(n_nodes) ||
        m->X0.alloc((size_t)n_nodes * kF) || m->H.alloc((layers + 1) * m->layer()) || m->A.alloc(layers * NH) ||
        m->Z.alloc(layers * NH) || m->dZ.alloc(NH) || m->dA.alloc(2 * m->layer()) || m->y.alloc(n_nodes) ||
        m->dH.alloc(NH) || m->part.alloc(nparts) || m->lpart.alloc(m->back_grid())) {
        fvp_mpnn_destroy(m);
        return -1;
    }
    mp_init<<<std::min(nb(n_nodes, 256), 2048), 256, 0, m->stream>>>(n_nodes, layers, m->ia.p, m->ideg.p, m->H.p, m->dA.p,
                                                                    m->np, m->m.p, m->v.p, m->g.p);
    if (refresh_bf16(m)) { fvp_mpnn_destroy(m); return -1; }
    FVP_HIP(hipStreamSynchronize(m->stream));
    *out = m;
    return 0;
}

extern "C" int fvp_mpnn_destroy(fvp_mpnn *m) {
    if (!m) return 0;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    m->ia.release(); m->ja.release(); m->p.release(); m->m.release(); m->v.release(); m->g.release();
    m->pb.release(); m->wt1.release(); m->wt2.release(); m->X0.release(); m->H.release(); m->A.release();
    m->Z.release(); m->dZ.release(); m->dA.release(); m->y.release(); m->dH.release(); m->wb.release(); m->ideg.release();
    m->part.release(); m->lpart.release();
    m->host.release();
    if (m->hgrad) (void)hipHostFree(m->hgrad);
    if (m->own_stream) (void)hipStreamDestroy(m->own_stream);
    delete m;
    return 0;
}

extern "C" long fvp_mpnn_num_params(const fvp_mpnn *m) { return m ? m->np : -1; }

extern "C" int fvp_mpnn_set_stream(fvp_mpnn *m, void *stream) {
    if (!m) { set_error("null model"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    FVP_HIP(hipStreamSynchronize(m->stream));
    m->stream = stream ? (hipStream_t)stream : m->own_stream;
    return 0;
}

extern "C" int fvp_mpnn_get_params(fvp_mpnn *m, float *host) {
    if (!m || !host) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    FVP_HIP(hipStreamSynchronize(m->stream));
    FVP_HIP(hipMemcpy(host, m->p.p, sizeof(float) * m->np, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int fvp_mpnn_set_params(fvp_mpnn *m, const float *host) {
    if (!m || !host) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    FVP_HIP(hipStreamSynchronize(m->stream));
    FVP_HIP(hipMemcpy(m->p.p, host, sizeof(float) * m->np, hipMemcpyHostToDevice));
    if (refresh_bf16(m)) return -1;
    FVP_HIP(hipStreamSynchronize(m->stream));
    return 0;
}

extern "C" int fvp_mpnn_get_grads(fvp_mpnn *m, float *host) {
    if (!m || !host) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    if (host_results(m)) return -1;
    if (!m->hgrad) {
        if (hipHostMalloc((void **)&m->hgrad, sizeof(float) * m->np, hipHostMallocCoherent) != hipSuccess) {
            m->hgrad = nullptr;
            set_error("pinned host allocation failed");
            return -1;
        }
    }
    double *const slot = m->host.p + fvp::kSlot, tag = ++m->host.tag;
    mp_post_grads<<<1, 1024, 0, m->stream>>>(m->np, m->g.p, m->hgrad, slot, tag);
    FVP_HIP(hipGetLastError());
    if (fvp::slot_wait(m->stream, slot, tag)) return -1;
    std::memcpy(host, m->hgrad, sizeof(float) * m->np);
    return 0;
}

// x: N x 16 FP32 features (device); y: N outputs (device, FP32)
extern "C" int fvp_mpnn_forward(fvp_mpnn *m, const float *x, float *y) {
    if (!m || !x || !y) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    return m->big() ? forward_impl<false, true>(m, x, y) : forward_impl<false, false>(m, x, y);
}

// forward + backward of the mean squared error against t (device, N); the
// gradients stay on the device (fvp_mpnn_get_grads, fvp_mpnn_adam)
extern "C" int fvp_mpnn_loss_grad(fvp_mpnn *m, const float *x, const float *t, double *loss) {
    if (!m || !x || !t) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    if (loss && host_results(m)) return -1;
    double *const slot = loss ? m->host.p : nullptr, tag = loss ? ++m->host.tag : 0.;
    if (m->big() ? forward_impl<true, true>(m, x, m->y.p) || backward_impl<true>(m, t, slot, tag)
                 : forward_impl<true, false>(m, x, m->y.p) || backward_impl<false>(m, t, slot, tag))
        return -1;
    if (loss) {
        if (fvp::slot_wait(m->stream, slot, tag)) return -1;
        *loss = slot[0];
    }
    return 0;
}

extern "C" int fvp_mpnn_adam(fvp_mpnn *m, float lr) {
    if (!m) { set_error("null model"); return -1; }
    FVP_HIP(hipSetDevice(m->device));
    ++m->step;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - (float)std::pow(b1, (double)m->step), c2 = 1.f - (float)std::pow(b2, (double)m->step);
    mp_adam<<<nb(m->np, 256), 256, 0, m->stream>>>(m->np, lr, b1, b2, 1e-8f, c1, c2, m->p.p, m->m.p, m->v.p, m->g.p,
                                                   m->pb.p);
    return refresh_weights(m);
}

extern "C" int fvp_mpnn_synchronize(fvp_mpnn *m) {
    if (!m) { set_error("null model"); return -1; }
    FVP_HIP(hipStreamSynchronize(m->stream));
    return 0;
}
