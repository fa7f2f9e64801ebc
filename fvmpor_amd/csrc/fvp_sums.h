// Sums over vectors without a launch or a copy of their own: partials per
// workgroup that the next kernel adds up, and results the host reads from
// pinned memory while the queue goes on.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

namespace fvp {

constexpr int kGsThreads = 512;
constexpr int kGsNb = 256;  // workgroups: one per CU
constexpr int kGsWaves = kGsThreads / 64;

// workgroups of kGsThreads for n rows, two rows a thread at least
static inline int gs_nb(long n) {
    return (int)std::max(1L, std::min((long)kGsNb, ((n >> 1) + kGsThreads - 1) / kGsThreads));
}

// Sums L columns over the wavefront: at each step a lane keeps one half of the
// columns and gives the other to its partner, L / 2 + L / 4 + ... exchanges
// instead of 6 L.  Returns column col's sum, if col < end (else the lane has none).
template <int BIT, int L>
__device__ __forceinline__ double fold_cols(const double (&v)[L], int &col, int &end) {
    if constexpr (BIT == 0) {
        static_assert(L == 1, "at most 64 columns");
        return v[0];
    } else if constexpr (L == 1) {
        double k[1] = {v[0] + __shfl_xor(v[0], BIT, 64)};
        return fold_cols<BIT / 2, 1>(k, col, end);
    } else {
        constexpr int H = (L + 1) / 2;
        const bool up = threadIdx.x & BIT;
        double k[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const double lo = v[i], hi = i + H < L ? v[i + H] : 0.;
            k[i] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, BIT, 64);
        }
        if (up) col += H;
        else end = end < col + H ? end : col + H;
        return fold_cols<BIT / 2, H>(k, col, end);
    }
}

// Block partials of K columns over kGsThreads threads: part[c * nb + block]
template <int K>
__device__ __forceinline__ void gs_store(const double (&acc)[K], int nk, int nb, double *__restrict__ part) {
    __shared__ double lds[kGsWaves][K];
    int col = 0, end = K;
    const double v = fold_cols<32, K>(acc, col, end);
    if (col < end) lds[threadIdx.x >> 6][col] = v;
    __syncthreads();
    if ((int)threadIdx.x < nk) {
        double t = 0.;
#pragma unroll
        for (int w = 0; w < kGsWaves; ++w) t += lds[w][threadIdx.x];
        part[threadIdx.x * nb + blockIdx.x] = t;
    }
}

// out[c] (LDS) = sum of column c's nb partials, c < K, in an order that depends
// on nb alone: every workgroup gets the same values.  Ends with a barrier.
template <int K>
__device__ __forceinline__ void gs_sums(int nb, const double *__restrict__ part, double *out) {
    constexpr int CW = (K + kGsWaves - 1) / kGsWaves, U = kGsNb / 64;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double v[CW][U], s[CW];
#pragma unroll
    for (int i = 0; i < CW; ++i) {
        const int c = wv + i * kGsWaves;
#pragma unroll
        for (int u = 0; u < U; ++u) v[i][u] = c < K && lane + 64 * u < nb ? part[c * nb + lane + 64 * u] : 0.;
    }
#pragma unroll
    for (int i = 0; i < CW; ++i) {
        s[i] = 0.;
#pragma unroll
        for (int u = 0; u < U; ++u) s[i] += v[i][u];
    }
    int col = 0, end = CW;
    const double t = fold_cols<32, CW>(s, col, end);
    if (col < end && wv + col * kGsWaves < K) out[wv + col * kGsWaves] = t;
    __syncthreads();
}

// ---- results for the host ----------------------------------------------------------
// A slot is kSlot doubles of pinned memory: up to three values and a tag.  The
// writer stores the tag last; the host polls it.  Tags count up, so that a slot
// never holds the awaited one beforehand.
constexpr int kSlot = 4;
struct HostSlots {
    double *p = nullptr;
    double tag = 0.;  // last one given out
    int alloc(int slots);  // contents and tag cleared
    void release();
};

// the tag, after the slot's values
__device__ __forceinline__ void slot_post(double *slot, double tag) {
    __threadfence_system();
    __hip_atomic_store(slot + kSlot - 1, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Waits for tag in a slot (written by a kernel queued on s).
int slot_wait(hipStream_t s, const double *slot, double tag);

// out[0, K) = the sums of K columns' partials, to the host's slot as well, if given
template <int K>
__global__ void __launch_bounds__(kGsThreads) gs_post(int nb, const double *__restrict__ part,
                                                      double *__restrict__ out, double *slot, double tag) {
    static_assert(K < kSlot, "a slot's values");
    __shared__ double s[K];
    gs_sums<K>(nb, part, s);
    if (threadIdx.x) return;
#pragma unroll
    for (int c = 0; c < K; ++c) out[c] = s[c];
    if (!slot) return;
#pragma unroll
    for (int c = 0; c < K; ++c) slot[c] = s[c];
    slot_post(slot, tag);
}

// A word that ends a kernel early when nonzero.  Read first and tested only
// where the kernel waits for other loads anyway (volatile keeps it there).
__device__ __forceinline__ double skip_word(const double *skip) {
    return skip ? *reinterpret_cast<const volatile double *>(skip) : 0.;
}

}  // namespace fvp
