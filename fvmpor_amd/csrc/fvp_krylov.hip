// Sparse linear algebra and the Newton-Krylov inner loop on gfx950.
//
//  * CSR SpMV: the entries of 64 rows by whole lines into the LDS, four lanes to a
//    row (rows hold ~7 (2D) to ~15 (3D) entries).
//  * ILU(0): level-scheduled factorisation and triangular solves.  Levels come
//    from the dependency DAG of L (forward) and U (backward); rows of a level
//    are independent.  Matrices whose solution fits the LDS take one launch for
//    all levels, larger ones a launch per level.
//  * Block-Jacobi ILU(0): a workgroup factors a block, a wavefront solves it.
//  * Jacobi: inverse diagonal.
//  * GMRES: right-preconditioned, restarted (gmres.c:26-201) with classical
//    Gram-Schmidt fused into one multi-dot and one multi-axpy pass per sweep
//    (applied twice when re-orthogonalising), so each Arnoldi step reads the
//    basis twice instead of 2(j+1) times as modified Gram-Schmidt would.  The
//    (m+1) x m Hessenberg system is reduced with Givens rotations on the
//    device; the host reads each step's residual estimate one step late.
//  * Coloured finite-difference Jacobian (preconditioner_dss.cpp:284-372): one
//    residual per colour of a distance-2 colouring.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <array>
#include <cmath>
#include <complex>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <numeric>
#include <set>
#include <utility>
#include <vector>

#include "fvp_blas.h"
#include "fvp_dense.h"
#include "fvp_internal.h"
#include "fvp_sums.h"

using fvp::DevBuf;
using fvp::set_error;

struct fvp_schur;

// Pattern tables of a factorisation (see bj_factor), the rows as level-ordered
// slots: per slot its record, per L entry the position of its pivot u_kk, and
// the byte offsets of the u_kj that update each entry of the row.
struct FactorTab {
    DevBuf<uint4> slot, out;
    DevBuf<unsigned> piv;
    DevBuf<uint2> off;
    int nc = 1;  // registers of the longest row (16 entries each): 1, 2 or 4
    bool mostly_long = false;  // more than one row in eight needs four
    void release() { slot.release(); out.release(); piv.release(); off.release(); }
};

// One triangle of the one-workgroup ILU(0) solve (see ilu0_solve)
struct IluTri {
    DevBuf<int> pptr;                  // pieces: first slot of each, then the slot count
    DevBuf<unsigned> row;              // per slot: row | entries << 16
    DevBuf<unsigned short> col;        // per slot: o_win columns
    DevBuf<double> val;                // the current factor: per slot its o_win entries, then (U) the slots' inverted pivots
    int npieces = 0, nslots = 0;
    void release() { pptr.release(); row.release(); col.release(); val.release(); }
};

// Packed layout of the block solve (see bj_solve), per triangle: the levels of at most
// 64 lanes, win entries per lane, their columns (two per word) and the row; out: where
// the factorisation puts a row (see factor_tables), place: the entries of a row of
// several slots
struct BjPack {
    int win = 0, levmax_l = 0, levmax_u = 0;  // win 0: not made
    fvp::DevBuf<int> lev_l, lptr_l, lev_u, lptr_u;
    fvp::DevBuf<unsigned> col_l, col_u, place;
    fvp::DevBuf<unsigned short> row_l, row_u;
    fvp::DevBuf<uint4> out;
    void release() {
        lev_l.release(); lptr_l.release(); lev_u.release(); lptr_u.release();
        col_l.release(); col_u.release(); place.release(); row_l.release(); row_u.release(); out.release();
    }
};

// Launch of the block factorisation: its threads, the levels in pieces of one slot per
// lane group, the LDS bytes that staging the values takes and whether they are staged
struct FacPieces {
    DevBuf<int> lev, lptr;
    int most = 0, threads = 0;  // pieces of one block
    size_t lds = 0;
    bool staged = false;
    void release() { lev.release(); lptr.release(); }
};

// The blocks as the host lays them out (see build_bj), kept until both precisions have
// their layout of the solve
struct BjTables {
    std::vector<int> roff, bia, bdiag;
    std::vector<unsigned short> bja, rows;
};

struct fvp_csr {
    int device = 0;
    hipStream_t stream = nullptr, own_stream = nullptr;
    int n = 0, nnz = 0, longest = 0;    // longest: entries of the longest row
    std::vector<int> ia_h, ja_h;
    DevBuf<int> ia, ja;
    DevBuf<double> a;
    // preconditioner
    int ptype = -1;
    DevBuf<double> lu, jac;
    DevBuf<int> diag;
    bool levels = false;
    std::vector<int> lptr_h, uptr_h;
    DevBuf<int> lrows, urows;
    DevBuf<int> flag;  // device error flag (zero pivot)
    // block-Jacobi ILU(0): per-block local CSR (columns relative to the block start)
    bool bj = false;
    int bs = FVP_BLOCK_ROWS;                // owned rows per block
    std::vector<int> bstart;                // explicit block boundaries (nb + 1), empty: every bs rows
    int overlap = 0;                        // layers of neighbouring rows added to each block (RAS)
    int nblk = 0, b_maxnz = 0, b_maxrows = 0, lds_max = 0;
    int factor_mode = -1;                   // staging form of the last block factorisation (bj_factor)
    DevBuf<int> b_roff, b_rowid, b_own;     // per block: first local row; global row of each local row; owned range
    DevBuf<double> b_zn2;                   // per block: its share of ||z||^2 of the last scaled solve
    DevBuf<int> b_ia, b_src;                // row pointers into the block arrays, source entry
    DevBuf<double> b_lu;
    DevBuf<float> b_lu32;                   // FP32 factor (FVP_PRECON_BJILU0_F32)
    FactorTab fac;                          // block factorisation (bj_factor), its slots the blocks' level order
    // global ILU(0) in one workgroup: its factor tables, and per triangle the
    // solve's pieces and padded row windows (see ilu0_solve)
    bool one = false;
    FactorTab ofac;
    DevBuf<int> o_fptr;                     // {0, n}, {0, pieces}, then the factorisation's pieces of slots
    IluTri otri[2];
    int o_threads = 64, o_fthreads = 512, o_win = 0;  // threads of the solve and of the factorisation
    size_t o_lds = 0;
    FacPieces fp[2];                        // FP64's and FP32's
    // packed solve layouts, FP64's (also FP32's where no row is longer than its lanes)
    // and FP32's, made at the first build that wants them; values, which bj_factor writes
    // (the rest stays zero), and per U lane the inverted diagonal
    std::unique_ptr<BjTables> tables;
    BjPack pack[2];
    int b_longest = 0;                      // entries of the longest row of a triangle
    const BjPack &pack_of(bool f32) const { return pack[f32 && b_longest > 4]; }
    DevBuf<double> val_l, val_u, dinv;
    DevBuf<float> val32_l, val32_u, dinv32;
    // workspace
    int m_alloc = -1;
    DevBuf<double> Q, w, r, z, part, scal, hdev;
    DevBuf<double> Hd, gd, csd, snd;        // Hessenberg (column-major, m+1 rows), rhs, Givens pairs
    fvp::HostSlots hstat;                   // GMRES, see GmresWork
    fvp::HostSlots hflag;                   // factorisation: the pivot flag
    const double *skip = nullptr;           // while GMRES queues a step: its word that ends the cycle
    DevBuf<double> Qk;                      // deflated GMRES: the kept harmonic Ritz vectors
    fvp_schur *sc = nullptr;                // Schur-complement preconditioner (FVP_PRECON_SCHUR)
};

// One-level Schur-complement preconditioner over subdomains of `bs`
// consecutive rows.  Interior unknowns (all couplings inside their subdomain)
// are numbered first, subdomain by subdomain, then the boundary unknowns.
struct fvp_schur {
    int nI = 0, nG = 0, nsub = 0, maxg = 0;
    fvp_csr *B = nullptr;                   // interior block: block-Jacobi ILU(0), one block per subdomain
    fvp::DevBuf<int> irow, grow;            // original row of each interior / boundary unknown
    fvp::DevBuf<int> bsrc;                  // source entry in A of each B entry
    fvp::DevBuf<int> e_ia, e_ja, e_loc, e_src;  // E (interior x boundary): column = boundary unknown, its
                                            // index inside the subdomain, source entry in A
    fvp::DevBuf<int> f_ia, f_ja, f_src;     // F (boundary x interior): column = interior unknown
    fvp::DevBuf<double> ev, fv;             // current values of E and F
    fvp::DevBuf<int> c_src;                 // C_ii entries: source in A and position in the dense blocks
    fvp::DevBuf<long> c_pos;
    fvp::DevBuf<int> goff, gsub, glocal;    // first boundary unknown per subdomain; subdomain and local index
    fvp::DevBuf<long> soff;                 // per subdomain: offset of its dense block (column major)
    fvp::DevBuf<double> S;                  // S_i, inverted in place by the build
    fvp::DevBuf<double> t1, t2, yG;         // work vectors (nI, nI, nG)
};

namespace fvp {

constexpr int kThreads = 256;

// ---- kernels ------------------------------------------------------------------
// y = alpha A x + beta y.  A workgroup's R rows are one contiguous range of
// entries: its threads load them entry by entry (whole lines, four values of x in flight
// each) into the LDS, a chunk of 1024 at a time, and 256 / R lanes to a row sum them
// from there.  What bounds it is the latency of row pointer -> column -> x, then its
// bytes (4.5 TB/s at 524 288 rows of 14.6).  Against eight lanes to a row straight from
// memory: 191 771 rows of 14.6 11.3 -> 9.3 us, 524 288 of 14.6 26.9 -> 21.0, 4 141 of 6.9
// 4.8 -> 4.0.  R, so that a workgroup's rows fill a chunk or two: 128 for rows of up to 9
// entries on average (64 / 128: 200 000 rows of 2 6.2 / 4.8 us, 10^6 of 3 23.9 / 14.0,
// 800 000 of 5 20.2 / 13.0, 400 000 of 9 12.1 / 12.5, 200 000 random of 11 13.1 / 14.5),
// not where single rows are long (one of 100 000: 1051 / 2054, lanes to a row straight
// from memory 1736); 16 for more than 40 (16 / 64: 4 000 rows of 61 4.8 / 6.6, 60 000 of 61
// 10.0 / 11.2, 60 000 of 45 8.3 / 7.6, 120 000 of 41 14.3 / 13.6, 3 000 of 480 17.6 / 184).
template <int R>
__global__ void __launch_bounds__(256) csr_gemv_kernel(int n, const int *__restrict__ ia, const int *__restrict__ ja,
                                                       const double *__restrict__ a, double alpha,
                                                       const double *__restrict__ x, double beta,
                                                       double *__restrict__ y, const double *skip) {
    constexpr int L = 256 / R, U = 4, CH = 256 * U;
    __shared__ double qa[CH], qx[CH];
    const double over = skip_word(skip);
    const int r0 = blockIdx.x * R, row = r0 + threadIdx.x / L, lane = threadIdx.x % L;
    const int b0 = ia[r0], len = ia[min(n, r0 + R)] - b0;
    const int k1 = (row < n ? ia[row + 1] : b0 + len) - b0;
    int k = (row < n ? ia[row] : b0 + len) - b0 + lane;
    if (over != 0.) return;
    double s = 0.;
    for (int c0 = 0; c0 < len; c0 += CH) {
        int j[U];
        double va[U], vx[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = b0 + min(c0 + 256 * u + (int)threadIdx.x, len - 1);
            j[u] = ja[e];
            va[u] = a[e];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) vx[u] = x[j[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            qa[256 * u + threadIdx.x] = va[u];
            qx[256 * u + threadIdx.x] = vx[u];
        }
        __syncthreads();
        for (const int end = min(k1, c0 + CH); k < end; k += L) s += qa[k - c0] * qx[k - c0];
        __syncthreads();
    }
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) s += __shfl_down(s, off, L);
    if (row < n && lane == 0) y[row] = beta == 0. ? alpha * s : alpha * s + beta * y[row];
}

__global__ void ilu0_factor_level(int cnt, const int *__restrict__ rows, const int *__restrict__ ia,
                                  const int *__restrict__ ja, const int *__restrict__ diag, double *__restrict__ lu,
                                  int *__restrict__ flag) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    int i = rows[t];
    int end = ia[i + 1];
    for (int kk = ia[i]; kk < diag[i]; ++kk) {
        int k = ja[kk];
        int kpos = ia[k], kend = ia[k + 1];
        double lik = lu[kk] * lu[diag[k]];
        lu[kk] = lik;
        for (int jj = kk + 1; jj < end; ++jj) {
            int j = ja[jj];
            while (kpos < kend && ja[kpos] < j) kpos++;
            if (kpos == kend) break;
            if (ja[kpos] == j) lu[jj] -= lik * lu[kpos];
        }
    }
    double d = lu[diag[i]];
    if (d == 0.) { atomicOr(flag, 1); lu[diag[i]] = 0.; }
    else lu[diag[i]] = 1. / d;
}

template <int LANES>
__global__ void __launch_bounds__(256) ilu0_lower_level(int cnt, const int *__restrict__ rows,
                                                        const int *__restrict__ ia, const int *__restrict__ ja,
                                                        const int *__restrict__ diag, const double *__restrict__ lu,
                                                        const double *__restrict__ x, double *__restrict__ y) {
    int tid = blockIdx.x * blockDim.x + threadIdx.x;
    int t = tid / LANES, lane = tid % LANES;
    int i = t < cnt ? rows[t] : 0;
    double s = 0.;
    if (t < cnt)
        for (int k = ia[i] + lane; k < diag[i]; k += LANES) s += lu[k] * y[ja[k]];
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) s += __shfl_down(s, off, LANES);
    if (t < cnt && lane == 0) y[i] = x[i] - s;
}

template <int LANES>
__global__ void __launch_bounds__(256) ilu0_upper_level(int cnt, const int *__restrict__ rows,
                                                        const int *__restrict__ ia, const int *__restrict__ ja,
                                                        const int *__restrict__ diag, const double *__restrict__ lu,
                                                        double *__restrict__ y) {
    int tid = blockIdx.x * blockDim.x + threadIdx.x;
    int t = tid / LANES, lane = tid % LANES;
    int i = t < cnt ? rows[t] : 0;
    double s = 0.;
    if (t < cnt)
        for (int k = diag[i] + 1 + lane; k < ia[i + 1]; k += LANES) s += lu[k] * y[ja[k]];
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) s += __shfl_down(s, off, LANES);
    if (t < cnt && lane == 0) y[i] = (y[i] - s) * lu[diag[i]];
}

__global__ void jacobi_build(int n, const int *__restrict__ ia, const int *__restrict__ ja,
                             const double *__restrict__ a, double *__restrict__ J, int *__restrict__ flag) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int pos = ia[i];
    while (pos < ia[i + 1] && ja[pos] < i) pos++;
    if (pos == ia[i + 1] || ja[pos] != i || a[pos] == 0.) { atomicOr(flag, 1); J[i] = 0.; return; }
    J[i] = 1. / a[pos];
}

// the pivot flag to the host's slot (a copy and a blocking wait cost about
// 15 us after the kernel), cleared for the next factorisation
__global__ void flag_post(int *__restrict__ flag, double *slot, double tag) {
    if (threadIdx.x) return;
    slot[0] = flag[0];
    flag[0] = 0;
    slot_post(slot, tag);
}

__global__ void vmul(long n, const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ c) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) c[i] = a[i] * b[i];
}

__global__ void vdiv(long n, const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ c) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) c[i] = a[i] / b[i];
}

__global__ void vcopy(long n, const double *__restrict__ a, double *__restrict__ b) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}

// y = b - y
__global__ void vrsub(long n, const double *__restrict__ b, double *__restrict__ y) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) y[i] = b[i] - y[i];
}

// y += x
__global__ void vadd(long n, const double *__restrict__ x, double *__restrict__ y) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) y[i] += x[i];
}

// compiler-only ordering of one wavefront's LDS accesses (the LDS executes a
// wavefront's accesses in issue order; no wait for outstanding memory loads)
__device__ __forceinline__ void wave_lds_order() { asm volatile("" ::: "memory"); }

constexpr int kChunk = 16;  // basis columns per Gram-Schmidt dot pass

__device__ __forceinline__ double wave_reduce(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Workgroups of the Gram-Schmidt passes: 512 x 256 threads (2 per CU), each
// thread streaming several row pairs per column.  Measured on the 1M-node
// box's node graph (30 unpreconditioned GMRES steps): 4.62 ms with 2048
// workgroups, 4.53 with 1024, 4.42-4.47 with 512, 4.42 with 256; fewer
// workgroups also mean fewer partials to reduce.
constexpr int kGsBlocks = 512;

// Leading dimension of the basis: columns padded to an even length, so that
// every column starts 16-byte aligned for the pairwise loads.
static inline long gs_ldq(long n) { return (n + 1) & ~1L; }
static inline int gs_blocks(long n) {
    return (int)std::max(1L, std::min((long)kGsBlocks, ((n >> 1) + kThreads - 1) / kThreads));
}

__device__ __forceinline__ void block_partial(double v, double *__restrict__ out) {
    __shared__ double lds[kThreads / 64];
    v = wave_reduce(v);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.;
        for (int k = 0; k < kThreads / 64; ++k) t += lds[k];
        *out = t;
    }
}

// Block partials of K values at once: every wavefront reduces all K with
// shuffles, one barrier, then thread c sums the wavefronts' values of column c
// into part[c * gridDim.x + block].
template <int K>
__device__ __forceinline__ void block_partials(const double (&acc)[K], int nk, double *__restrict__ part) {
    __shared__ double lds[kThreads / 64][K];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < K; ++c) {
        const double v = wave_reduce(acc[c]);
        if (lane == 0) lds[wv][c] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < nk) {
        double t = 0.;
        for (int k = 0; k < kThreads / 64; ++k) t += lds[k][threadIdx.x];
        part[threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

// Block partials of w . Q[:, c] for c < NC and of w . w (stored as column NC
// when ww is set): part[c * gridDim.x + block].  Each thread reads element
// pairs (16-byte loads; the basis columns are padded to an even length, ldq),
// every column load of a pair issued before the first product.  Skipped
// entirely when skip[0] == 0 (second pass not needed).
template <int NC>
__global__ void __launch_bounds__(kThreads) mdot_kernel(long n, const double *__restrict__ w,
                                                        const double *__restrict__ Q, long ldq, int ww,
                                                        double *__restrict__ part, const double *__restrict__ skip) {
    if (skip && skip[0] == 0.) return;
    double acc[NC + 1];
#pragma unroll
    for (int c = 0; c <= NC; ++c) acc[c] = 0.;
    const long np = n >> 1;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < np; p += (long)gridDim.x * blockDim.x) {
        const double2 a = reinterpret_cast<const double2 *>(w)[p];
        double2 q[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) q[c] = reinterpret_cast<const double2 *>(Q + c * ldq)[p];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += a.x * q[c].x + a.y * q[c].y;
        acc[NC] += a.x * a.x + a.y * a.y;
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const double a = w[n - 1];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += a * Q[c * ldq + n - 1];
        acc[NC] += a * a;
    }
    block_partials<NC + 1>(acc, ww ? NC + 1 : NC, part);
}

// w -= Q[:, 0..NC) coef, and block partials of the updated w . w into
// part[block]; element pairs as in mdot_kernel.
template <int NC>
__global__ void __launch_bounds__(kThreads) axpy_norm(long n, double *__restrict__ w, const double *__restrict__ Q,
                                                      long ldq, const double *__restrict__ coef,
                                                      double *__restrict__ part, const double *__restrict__ skip) {
    if (skip && skip[0] == 0.) return;
    double h[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) h[c] = coef[c];
    double acc = 0.;
    const long np = n >> 1;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < np; p += (long)gridDim.x * blockDim.x) {
        double2 q[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) q[c] = reinterpret_cast<const double2 *>(Q + c * ldq)[p];
        double2 a = reinterpret_cast<double2 *>(w)[p];
        double sx = 0., sy = 0.;
#pragma unroll
        for (int c = 0; c < NC; ++c) { sx += h[c] * q[c].x; sy += h[c] * q[c].y; }
        a.x -= sx;
        a.y -= sy;
        reinterpret_cast<double2 *>(w)[p] = a;
        acc += a.x * a.x + a.y * a.y;
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        double sx = 0.;
#pragma unroll
        for (int c = 0; c < NC; ++c) sx += h[c] * Q[c * ldq + n - 1];
        const double a = w[n - 1] - sx;
        w[n - 1] = a;
        acc += a * a;
    }
    block_partial(acc, part + blockIdx.x);
}

using MdotLaunch = void (*)(hipStream_t, int, long, const double *, const double *, long, int, double *,
                           const double *);
using AxpyLaunch = void (*)(hipStream_t, int, long, double *, const double *, long, const double *, double *,
                           const double *);
template <int NC>
static void mdot_launch(hipStream_t s, int nb, long n, const double *w, const double *Q, long ldq, int ww,
                        double *part, const double *skip) {
    mdot_kernel<NC><<<nb, kThreads, 0, s>>>(n, w, Q, ldq, ww, part, skip);
}
template <int NC>
static void axpy_launch(hipStream_t s, int nb, long n, double *w, const double *Q, long ldq, const double *coef,
                        double *part, const double *skip) {
    axpy_norm<NC><<<nb, kThreads, 0, s>>>(n, w, Q, ldq, coef, part, skip);
}
template <int... I>
static constexpr std::array<MdotLaunch, sizeof...(I)> mdot_table(std::integer_sequence<int, I...>) {
    return {&mdot_launch<I + 1>...};
}
template <int... I>
static constexpr std::array<AxpyLaunch, sizeof...(I)> axpy_table(std::integer_sequence<int, I...>) {
    return {&axpy_launch<I + 1>...};
}
// per column count 1..kChunk
static const auto kMdot = mdot_table(std::make_integer_sequence<int, kChunk>{});
static const auto kAxpy = axpy_table(std::make_integer_sequence<int, kChunk>{});

// Selective reorthogonalisation (Kahan-Parlett "twice is enough"): a second
// classical Gram-Schmidt pass when the first one cancelled more than half of
// ||w||^2 (mode 1), always (mode 2) or never (mode 0).
__global__ void reorth_decide(const double *__restrict__ ww, const double *__restrict__ n1, int mode,
                              double *__restrict__ flag) {
    if (threadIdx.x == 0) flag[0] = mode == 2 ? 1. : mode == 0 ? 0. : (n1[0] < 0.5 * ww[0] ? 1. : 0.);
}

// netlib drotg
__host__ __device__ inline void drotg_dev(double *da, double *db, double *c, double *s) {
    double roe = fabs(*da) > fabs(*db) ? *da : *db;
    double scale = fabs(*da) + fabs(*db), r, z;
    if (scale == 0.) { *c = 1.; *s = 0.; r = 0.; z = 0.; }
    else {
        double a = *da / scale, b = *db / scale;
        r = scale * sqrt(a * a + b * b);
        r = (roe >= 0 ? 1. : -1.) * r;
        *c = *da / r; *s = *db / r;
        z = 1.;
        if (fabs(*da) > fabs(*db)) z = *s;
        if (fabs(*db) >= fabs(*da) && *c != 0.) z = 1. / *c;
    }
    *da = r; *db = z;
}

// End of Arnoldi step j in one launch.  Every block forms 1/h_{j+1,j} from the
// same norm (||w||^2 after the first pass, or after the second when flag is
// set) and scales its slice of w into q_{j+1}.  Block 0 also sets the new
// Hessenberg column j = h1 (+ h2 after a second pass) with h_{j+1,j} = ||w||,
// applies the previous rotations and the new Givens rotation, rotates the
// right-hand side g, and writes {|g_{j+1}|, h_{j+1,j}} to stat and, when hslot
// is given (pinned host memory the device can write), there too, then tag.
// With npart, ||w||^2 is not reduced beforehand: every block sums the nb
// partials of the single Gram-Schmidt pass itself, in reduce_cols' order (the
// same value bit for bit, one launch fewer), and the slices are grid-strided.
// Workgroups of arnoldi_finish (grid-strided): few enough that every one
// summing the norm's partials costs little.
constexpr int kFinishBlocks = 512;
__global__ void __launch_bounds__(256) arnoldi_finish(int j, int m, const double *__restrict__ h1,
                                                      const double *__restrict__ h2, const double *__restrict__ n1,
                                                      const double *__restrict__ n2, const double *__restrict__ flag,
                                                      double *__restrict__ H, double *__restrict__ cs,
                                                      double *__restrict__ sn, double *__restrict__ g,
                                                      double *__restrict__ stat, double *hslot, double tag, long n,
                                                      const double *__restrict__ w, double *__restrict__ q,
                                                      const double *__restrict__ npart = nullptr, int nb = 0) {
    __shared__ double lds[4];
    const bool two = !npart && flag && flag[0] != 0.;
    double nn;
    if (npart) {
        // each lane's partials in order, four loads in flight at a time
        double s = 0.;
        const int bd = blockDim.x;
        for (int b0 = threadIdx.x; b0 < nb; b0 += 4 * bd) {
            double q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = b0 + u * bd < nb ? npart[b0 + u * bd] : 0.;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (b0 + u * bd < nb) s += q[u];
        }
        s = wave_reduce(s);
        if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
        __syncthreads();
        double v = 0.;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) v += lds[k];
        nn = v;
    } else {
        nn = two ? n2[0] : n1[0];
    }
    const double hn = sqrt(nn);
    const double ninv = hn > 0. ? 1. / hn : 0.;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        q[i] = w[i] * ninv;
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    double *hc = H + (size_t)j * (m + 1);
    for (int k = 0; k <= j; ++k) hc[k] = two ? h1[k] + h2[k] : h1[k];
    hc[j + 1] = hn;
    for (int k = 0; k < j; ++k) {
        const double t1 = cs[k] * hc[k] + sn[k] * hc[k + 1];
        hc[k + 1] = cs[k] * hc[k + 1] - sn[k] * hc[k];
        hc[k] = t1;
    }
    double a = hc[j], b = hc[j + 1], c, sv;
    drotg_dev(&a, &b, &c, &sv);
    cs[j] = c; sn[j] = sv;
    hc[j] = c * hc[j] + sv * hc[j + 1];
    hc[j + 1] = 0.;
    const double gj = g[j];
    g[j] = c * gj;
    g[j + 1] = -sv * gj;
    stat[0] = fabs(g[j + 1]);
    stat[1] = hn;
    if (hslot) {
        hslot[0] = fabs(g[j + 1]);
        hslot[1] = hn;
        slot_post(hslot, tag);
    }
}

// ---- Arnoldi steps of up to kGsCols basis columns in three launches --------------
// gs_dots: block partials of Q^T w and w . w; gs_update: sums them (every
// workgroup by itself), w -= Q h1, block partials of the second pass's dots and
// of the updated w . w; gs_finish: sums those, the second update where the first
// pass cancelled, q_{j+1}, the Hessenberg column and its rotations.  A reduction
// launch of its own costs about as much as the pass it follows (192 000 rows, 10
// columns: 6 us for the dots, 3 + 2 us for the launch that sums 10 x 512 numbers),
// so the partials go to the next kernel, kGsNb workgroups x (NC + 1) columns,
// 4 loads a lane; more workgroups would read more than the basis itself.
// What bounds the three: the basis, read once each (twice with the second
// update), and at 192 000 rows and below the latency of one round of loads per
// thread, which is why every column's load is issued before the sums.
// Per step of the Krylov solve of 191 771 rows, 21 steps (Jacobi): 65 -> 33 us.
constexpr int kGsCols = 32;  // columns held in registers; longer bases go through mdot_kernel and axpy_norm
static_assert(kGsNb * (kGsCols + 1) <= kGsBlocks * (kChunk + 1), "partials fit the workspace");

// a wavefront-uniform value in scalar registers
__device__ __forceinline__ double uniform(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// Rows per load: pairs while the columns' loads in flight fit 64 registers,
// then single rows
template <int NC>
using GsRow = std::conditional_t<(NC <= 16), double2, double>;
__device__ __forceinline__ double gs_dot(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ double gs_dot(double a, double b) { return a * b; }
__device__ __forceinline__ void gs_fma(double2 &s, double h, double2 q) { s.x += h * q.x; s.y += h * q.y; }
__device__ __forceinline__ void gs_fma(double &s, double h, double q) { s += h * q; }
__device__ __forceinline__ void gs_sub(double2 &a, double2 s) { a.x -= s.x; a.y -= s.y; }
__device__ __forceinline__ void gs_sub(double &a, double s) { a -= s; }
__device__ __forceinline__ double2 gs_scale(double2 a, double f) { return {a.x * f, a.y * f}; }
__device__ __forceinline__ double gs_scale(double a, double f) { return a * f; }
__device__ __forceinline__ double2 gs_mul(double2 a, double2 b) { return {a.x * b.x, a.y * b.y}; }
__device__ __forceinline__ double gs_mul(double a, double b) { return a * b; }

// Runs f on every row group of the grid and, with pairs, g on an odd last row.
// The leading dimension of Q is even; w, the diagonal and the caller's vectors
// end at n, so the odd row is read by itself.
template <int NC>
__device__ __forceinline__ long gs_groups(long n) { return NC <= 16 ? n >> 1 : n; }
template <int NC>
__device__ __forceinline__ bool gs_tail(long n) { return NC <= 16 && (n & 1) && blockIdx.x == 0 && threadIdx.x == 0; }

template <int NC>
__global__ void __launch_bounds__(kGsThreads) gs_dots(long n, const double *__restrict__ w,
                                                      const double *__restrict__ Q, long ldq,
                                                      double *__restrict__ part) {
    using R = GsRow<NC>;
    double acc[NC + 1];
#pragma unroll
    for (int c = 0; c <= NC; ++c) acc[c] = 0.;
    const long np = gs_groups<NC>(n);
    for (long p = blockIdx.x * (long)kGsThreads + threadIdx.x; p < np; p += (long)gridDim.x * kGsThreads) {
        const R a = reinterpret_cast<const R *>(w)[p];
        R q[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) q[c] = reinterpret_cast<const R *>(Q + c * ldq)[p];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += gs_dot(a, q[c]);
        acc[NC] += gs_dot(a, a);
    }
    if (gs_tail<NC>(n)) {
        const double a = w[n - 1];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += a * Q[c * ldq + n - 1];
        acc[NC] += a * a;
    }
    gs_store<NC + 1>(acc, NC + 1, gridDim.x, part);
}

// h1[0, NC] = the sums; twice: the second pass's dots too.  ctl[1] != 0: the
// cycle has converged, nothing is done.
template <int NC>
__global__ void __launch_bounds__(kGsThreads) gs_update(long n, double *__restrict__ w,
                                                        const double *__restrict__ Q, long ldq, int twice,
                                                        const double *__restrict__ part, double *__restrict__ part2,
                                                        double *__restrict__ h1, const double *__restrict__ ctl) {
    using R = GsRow<NC>;
    __shared__ double hs[NC + 1];
    const long np = gs_groups<NC>(n), step = (long)gridDim.x * kGsThreads;
    long p = blockIdx.x * (long)kGsThreads + threadIdx.x;
    const double done = ctl[1];
    R a{}, q[NC];
    auto load = [&]() {
        a = reinterpret_cast<const R *>(w)[p];
#pragma unroll
        for (int c = 0; c < NC; ++c) q[c] = reinterpret_cast<const R *>(Q + c * ldq)[p];
    };
    if (p < np) load();
    gs_sums<NC + 1>(gridDim.x, part, hs);
    if (done != 0.) return;
    if (blockIdx.x == 0 && (int)threadIdx.x <= NC) h1[threadIdx.x] = hs[threadIdx.x];
    double h[NC], acc[NC + 1];
#pragma unroll
    for (int c = 0; c < NC; ++c) h[c] = uniform(hs[c]);
#pragma unroll
    for (int c = 0; c <= NC; ++c) acc[c] = 0.;
    while (p < np) {
        R s{};
#pragma unroll
        for (int c = 0; c < NC; ++c) gs_fma(s, h[c], q[c]);
        gs_sub(a, s);
        reinterpret_cast<R *>(w)[p] = a;
        if (twice) {
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[c] += gs_dot(a, q[c]);
        }
        acc[NC] += gs_dot(a, a);
        p += step;
        if (p < np) load();
    }
    if (gs_tail<NC>(n)) {
        double qt[NC], s = 0.;
#pragma unroll
        for (int c = 0; c < NC; ++c) { qt[c] = Q[c * ldq + n - 1]; s += h[c] * qt[c]; }
        const double at = w[n - 1] - s;
        w[n - 1] = at;
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] += at * qt[c];
        acc[NC] += at * at;
    }
    gs_store<NC + 1>(acc, NC + 1, gridDim.x, part2);
}

// Column j = NC - 1 of the Hessenberg matrix: the previous rotations, the new
// one, the right-hand side g, {|g_{j+1}|, h_{j+1,j}} to stat and, when hslot is
// given (pinned host memory), there too, then tag behind them; ctl[1] = 1 when
// the cycle ends here by the host's own test.  By one wavefront: everything the
// rotations' serial chain needs is loaded into the LDS at once.
__device__ inline void gs_hessenberg(int j, int m, double hk, double hn, double thr, double *__restrict__ H,
                                     double *__restrict__ cs, double *__restrict__ sn, double *__restrict__ g,
                                     double *__restrict__ ctl, double *__restrict__ stat, double *hslot, double tag) {
    __shared__ double hc[kGsCols + 1], cl[kGsCols], sl[kGsCols];
    const int l = threadIdx.x & 63;
    if (l <= j) hc[l] = hk;
    if (l < j) { cl[l] = cs[l]; sl[l] = sn[l]; }
    wave_lds_order();
    if (l == 0) {
        const double gj = g[j];
        double a = hc[0];
        for (int k = 0; k < j; ++k) {
            const double b = hc[k + 1], c = cl[k], s = sl[k];
            hc[k] = c * a + s * b;
            a = c * b - s * a;
        }
        double b = hn, c, s, r = a;
        drotg_dev(&r, &b, &c, &s);
        cs[j] = c;
        sn[j] = s;
        hc[j] = c * a + s * hn;
        g[j] = c * gj;
        const double g1 = -s * gj, est = fabs(g1);
        g[j + 1] = g1;
        stat[0] = est;
        stat[1] = hn;
        if (est < thr || !(hn > 1e-16)) ctl[1] = 1.;
        if (hslot) {
            hslot[0] = est;
            hslot[1] = hn;
            slot_post(hslot, tag);
        }
    }
    wave_lds_order();
    double *col = H + (size_t)j * (m + 1);
    if (l <= j) col[l] = hc[l];
    if (l == 0) col[j + 1] = 0.;
}

// End of step j = NC - 1.  mode: 0 never a second update, 1 where the first pass
// cancelled more than half of ||w||^2, 2 always (Kahan-Parlett "twice is
// enough").  The norm after the second update is ||w||^2 - ||h2||^2 (q's
// orthonormal columns), whose rounding error is that of ||w||^2 as long as
// ||h2||^2 is a small part of it; above 2^-10 of it (w lies in the basis' span to
// rounding) the update is written unscaled, and the last workgroup to finish
// takes its norm and scales it.  All workgroups but the last stream rows, that
// one sets the Hessenberg column.  diag: z = diag q_{j+1} as well.
template <int NC>
__global__ void __launch_bounds__(kGsThreads) gs_finish(int mode, int m, long n, const double *__restrict__ w,
                                                        double *__restrict__ Q, long ldq,
                                                        double *__restrict__ part, const double *__restrict__ part2,
                                                        const double *__restrict__ h1, double thr,
                                                        double *__restrict__ H, double *__restrict__ cs,
                                                        double *__restrict__ sn, double *__restrict__ g,
                                                        double *__restrict__ ctl, double *__restrict__ stat,
                                                        double *hslot, double tag, const double *__restrict__ diag,
                                                        double *__restrict__ z) {
    using R = GsRow<NC>;
    __shared__ double hs[NC + 1];
    const int nb = gridDim.x - 1, wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double done = ctl[1], ww = h1[NC];
    if (mode) {
        gs_sums<NC + 1>(nb, part2, hs);
    } else {
        gs_sums<1>(nb, part2 + (size_t)NC * nb, hs + NC);
    }
    if (done != 0.) return;
    const double n1 = uniform(hs[NC]);
    const bool two = mode == 2 || (mode == 1 && n1 < 0.5 * ww);
    double hh = 0.;
    if (two)
#pragma unroll
        for (int c = 0; c < NC; ++c) hh += hs[c] * hs[c];
    const bool exact = two && !(hh <= n1 * (1. / 1024));
    const double nn = two ? n1 - hh : n1;
    if ((int)blockIdx.x == nb) {
        if (!exact && wv == 0)
            gs_hessenberg(NC - 1, m, lane < NC ? (two ? h1[lane] + hs[lane] : h1[lane]) : 0., sqrt(nn), thr, H, cs, sn,
                          g, ctl, stat, hslot, tag);
        return;
    }
    const double hn = sqrt(nn), f = exact ? 1. : hn > 0. ? 1. / hn : 0.;
    double *__restrict__ qn = Q + (size_t)NC * ldq;
    const long np = gs_groups<NC>(n), step = (long)nb * kGsThreads;
    const long p0 = blockIdx.x * (long)kGsThreads + threadIdx.x;
    double acc = 0.;
    auto put = [&](auto *out, long p, auto a) {
        using A = decltype(a);
        acc += gs_dot(a, a);
        a = gs_scale(a, f);
        out[p] = a;
        if (diag) reinterpret_cast<A *>(z)[p] = gs_mul(a, reinterpret_cast<const A *>(diag)[p]);
    };
    if (two) {
        double h[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) h[c] = uniform(hs[c]);
        for (long p = p0; p < np; p += step) {
            R a = reinterpret_cast<const R *>(w)[p], q[NC], s{};
#pragma unroll
            for (int c = 0; c < NC; ++c) q[c] = reinterpret_cast<const R *>(Q + c * ldq)[p];
#pragma unroll
            for (int c = 0; c < NC; ++c) gs_fma(s, h[c], q[c]);
            gs_sub(a, s);
            put(reinterpret_cast<R *>(qn), p, a);
        }
        if (gs_tail<NC>(n)) {
            double s = 0.;
#pragma unroll
            for (int c = 0; c < NC; ++c) s += h[c] * Q[c * ldq + n - 1];
            put(qn, n - 1, w[n - 1] - s);
        }
    } else {
        for (long p = p0; p < np; p += step) put(reinterpret_cast<R *>(qn), p, reinterpret_cast<const R *>(w)[p]);
        if (gs_tail<NC>(n)) put(qn, n - 1, w[n - 1]);
    }
    if (!exact) return;
    // part's first column is free here: gs_update has summed it
    __shared__ int last;
    {
        double a1[1] = {acc};
        gs_store<1>(a1, 1, nb, part);
    }
    __threadfence();
    __syncthreads();
    unsigned *ticket = reinterpret_cast<unsigned *>(ctl + 2);
    if (threadIdx.x == 0) last = atomicAdd(ticket, 1u) == (unsigned)nb - 1;
    __syncthreads();
    if (!last) return;
    __threadfence();
    if (threadIdx.x == 0) *ticket = 0;
    __shared__ double ex[kGsWaves];
    const double pv = (int)threadIdx.x < nb ? __hip_atomic_load(part + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.;
    const double ps = wave_reduce(pv);
    if (lane == 0) ex[wv] = ps;
    __syncthreads();
    double en = 0.;
#pragma unroll
    for (int k = 0; k < kGsWaves; ++k) en += ex[k];
    const double he = sqrt(en), fe = he > 0. ? 1. / he : 0.;
    for (long i = threadIdx.x; i < n; i += kGsThreads) {
        const double q = __hip_atomic_load(qn + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * fe;
        qn[i] = q;
        if (diag) z[i] = q * diag[i];
    }
    if (wv == 0)
        gs_hessenberg(NC - 1, m, lane < NC ? h1[lane] + hs[lane] : 0., he, thr, H, cs, sn, g, ctl, stat, hslot, tag);
}

struct GsStep {
    void (*dots)(long, const double *, const double *, long, double *);
    void (*update)(long, double *, const double *, long, int, const double *, double *, double *, const double *);
    void (*finish)(int, int, long, const double *, double *, long, double *, const double *, const double *, double,
                   double *, double *, double *, double *, double *, double *, double *, double, const double *,
                   double *);
};
template <int... I>
static constexpr std::array<GsStep, sizeof...(I)> gs_table(std::integer_sequence<int, I...>) {
    return {GsStep{&gs_dots<I + 1>, &gs_update<I + 1>, &gs_finish<I + 1>}...};
}
static const auto kGs = gs_table(std::make_integer_sequence<int, kGsCols>{});

// Start of a cycle: q_0 = r / beta (and z = diag q_0), g = beta e_1, the
// control words cleared.
__global__ void gs_start(long n, const double *__restrict__ r, const double *__restrict__ nsq, double beta,
                         double *__restrict__ q, const double *__restrict__ diag, double *__restrict__ z,
                         double *__restrict__ g, int len, double *__restrict__ ctl) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < len; k += blockDim.x) g[k] = k == 0 ? beta : 0.;
        if (threadIdx.x < 3) ctl[threadIdx.x] = 0.;
    }
    if (i >= n) return;
    const double v = r[i] * (1. / sqrt(nsq[0]));
    q[i] = v;
    if (diag) z[i] = v * diag[i];
}

// r = b - r, block partials of r . r and b . b
__global__ void __launch_bounds__(kGsThreads) gs_residual(long n, const double *__restrict__ b,
                                                          double *__restrict__ r, double *__restrict__ part) {
    double acc[2] = {0., 0.};
    for (long i = blockIdx.x * (long)kGsThreads + threadIdx.x; i < n; i += (long)gridDim.x * kGsThreads) {
        const double bi = b[i], v = bi - r[i];
        r[i] = v;
        acc[0] += v * v;
        acc[1] += bi * bi;
    }
    gs_store<2>(acc, 2, gridDim.x, part);
}

// End of a cycle: y = R^-1 g on the first k rotated columns, then out = Q y, or
// with add x += diag (Q y) (diag null: x += Q y).  Every workgroup solves the
// small triangle by itself, a lane per row, from the LDS (one thread reading
// memory entry by entry took 23 us for 21 columns).
__global__ void __launch_bounds__(256) gs_solution(long n, int k, int m, const double *__restrict__ H,
                                                   const double *__restrict__ g, const double *__restrict__ Q,
                                                   long ldq, const double *__restrict__ diag, int add,
                                                   double *__restrict__ out) {
    __shared__ double R[63 * 64 / 2], y[64];
    for (int c = threadIdx.x >> 6; c < k; c += 4) {
        const int l = threadIdx.x & 63;
        if (l <= c) R[c * (c + 1) / 2 + l] = H[(size_t)c * (m + 1) + l];
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const int l = threadIdx.x;
        double v = l < k ? g[l] : 0.;
        for (int c = k - 1; c >= 0; --c) {
            const double *col = R + c * (c + 1) / 2;
            const double yc = __shfl(v, c, 64) / col[c];
            if (l < c) v -= col[l] * yc;
            if (l == c) y[c] = yc;
        }
    }
    __syncthreads();
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        double s = 0.;
        int c = 0;
        for (; c + 8 <= k; c += 8) {
            double q[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) q[u] = Q[(c + u) * ldq + i];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += y[c + u] * q[u];
        }
        for (; c < k; ++c) s += y[c] * Q[c * ldq + i];
        if (add) out[i] += diag ? s * diag[i] : s;
        else out[i] = s;
    }
}

// out[c] = sum over blocks of part[c * nb + block]; skip: see mdot_kernel
__global__ void __launch_bounds__(kThreads) reduce_cols(int nb, const double *__restrict__ part,
                                                        double *__restrict__ out, const double *__restrict__ skip) {
    if (skip && skip[0] == 0.) return;
    __shared__ double lds[kThreads / 64];
    int c = blockIdx.x;
    // each lane's partials in order, four loads in flight at a time
    double s = 0.;
    const int bd = blockDim.x;
    const double *pc = part + (size_t)c * nb;
    for (int b0 = threadIdx.x; b0 < nb; b0 += 4 * bd) {
        double q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = b0 + u * bd < nb ? pc[b0 + u * bd] : 0.;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (b0 + u * bd < nb) s += q[u];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) v += lds[k];
        out[c] = v;
    }
}

// out = sum_c y[c] Q[:, c]  (y on the device)
__global__ void lincomb(long n, double *__restrict__ out, const double *__restrict__ Q, long ldq, int nc,
                        const double *__restrict__ y) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.;
    for (int c = 0; c < nc; ++c) s += Q[c * ldq + i] * y[c];
    out[i] = s;
}

// y = a x + b y  (host scalars)
__global__ void vaxpby(long n, double a, const double *__restrict__ x, double b, double *__restrict__ y) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[i] = b == 0. ? a * x[i] : a * x[i] + b * y[i];
}

// ---- block-Jacobi ILU(0): one workgroup per block of bs consecutive rows
// (factorisation: bj_factor; the rows of one level run concurrently)

// workgroup barrier for LDS data: waits for LDS accesses only, so global loads
// issued ahead stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Factorisation (IKJ order).  Rows of one level only need rows of earlier
// levels, so when a level begins every u_kj that its rows use is final: a group
// of kBjGroup lanes holds one row in registers (entry j in lane j mod 16), loads
// all the u_kj and pivots of its L entries in one round, and runs the row's
// chain (l_ik = a_ik u_kk^-1, then a_ij -= l_ik u_kj for the columns both rows
// have) in registers with broadcasts inside the group.  What bounds it is the
// level chain (one round of loads, the row's chain, one barrier per level) and,
// inside it, instruction issue (about 250 per wavefront and level), so everything
// that does not depend on values is loaded ahead (slot records two levels, pivot
// positions, offsets and the row's own values one), and L entries that no row of
// a wavefront has are skipped four at a time.  The pattern gives per L entry
// (i, k) the position of u_kk, and per entry j of row i one byte: the distance
// from u_kk to u_kj in row k, or 0.  Eight bytes (eight L entries) are one load
// per lane.  141k-node box, FP32, 1024-row blocks, one overlap layer: 86 us
// with 1024 threads, 110 with 512, the solve's packed copies written as well; pairs read, modified and written in
// memory one L entry after another, and a packing pass, took 500 + 25 us.
// STAGED: the block's values are held in LDS; otherwise in place in memory.
constexpr int kBjGroup = 16;
// Threads: 64 to 512 or, for rows of up to 16 entries, 1024 (4 to 64 rows of a level at
// once; longer rows' registers leave room for 512), the cheapest by this estimate, the
// more of equal ones.  A round of resident blocks costs its pieces of levels, each a
// latency or, where that is longer, what its wavefronts issue (a wavefront without a row
// loads ahead all the same), and the values' way in and out.  The constants fit 386
// builds (blocks of 64 to 4096 rows, with and without overlap, of meshes, grids, bands
// and random patterns, each with every thread count) to 8 % of each one's best.  138 blocks
// of 1024 rows with an overlap layer, FP32: 110 us with 512 threads, 86 with 1024; 977
// chains of 256 rows, FP64: 210 us with 64, 428 with 512; 129 blocks with levels of 4
// rows: 437 us with 64, 216 with 512.
constexpr int kFacThreads[] = {1024, 512, 256, 128, 64};
static double fac_cost(int th, int nc, size_t vb, long blocks, long nz, size_t lds, long lds_max, int pieces) {
    if (th == 1024 && nc > 1) return 1e300;
    const int waves = th / 64, most = nc == 1 ? 16 : nc == 2 && vb == 4 ? 12 : 8;  // wavefronts a CU holds
    const long cus = 256, fit = std::max(1L, std::min((long)most / waves, lds ? lds_max / (long)lds : 64L));
    const long rounds = (blocks + cus * fit - 1) / (cus * fit);
    const double issue = 0.35 * (double)std::min(fit, (blocks + cus - 1) / cus) * waves / 4;
    return (double)rounds * (pieces * std::max(1., issue) + 0.8 * (double)nz / th);
}
constexpr int kAhead = 2;  // offset words of eight L entries loaded a level ahead

// x of lane K of each 16-lane row, in every lane of that row
template <int K>
__device__ __forceinline__ int row_bcast(int x) {
    return __builtin_amdgcn_update_dpp(0, x, 0x150 + K, 0xf, 0xf, true);
}
template <int K>
__device__ __forceinline__ unsigned row_bcast(unsigned x) { return (unsigned)row_bcast<K>((int)x); }
template <int K>
__device__ __forceinline__ float row_bcast(float x) { return __int_as_float(row_bcast<K>(__float_as_int(x))); }
template <int K>
__device__ __forceinline__ double row_bcast(double x) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)row_bcast<K>((int)(unsigned)b), hi = (unsigned)row_bcast<K>((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The layout of the solve's packed copies: win values per lane; place: where
// the entries of a row of several slots go (out.w > 0), from out.w - 1 on; all within
// the block, whose first slots are ptr[lev[b]] of the solve's levels (null: 0)
struct FacOut {
    unsigned win;
    const unsigned *place;
    const int *lev_l, *ptr_l, *lev_u, *ptr_u;
};

// What a row needs besides the other rows' values, loaded a level ahead.
template <typename T, int NC>
struct FacRow {
    int s0, len, d;           // first entry, entries, L entries
    unsigned tab, l0;         // its first offset word, its first L entry
    unsigned at[NC];          // place of each entry in the solve's packed copies
    T a[NC];                  // this lane's entries
    unsigned piv;             // pivot position of L entry `lane`
    unsigned off[2 * kAhead][NC];  // distances, four L entries a word, 0: none
};

// The registers (1, 2 or 4) that the rows of a wavefront need, uniform: rows of up to 16
// entries take one, also where others of the matrix have more.  100 000 tridiagonal rows
// in blocks of 1024 with overlap, FP64 / FP32, us: 737 / 715; with one row of 24 entries
// 804 / 802 (1096 / 1053 with two registers for every row), of 40 900 / 860 (1654 / 1431).
template <int NC>
__device__ __forceinline__ int fac_regs(int len) {
    if (NC == 1 || !__any(len > kBjGroup)) return 1;
    return NC == 2 || !__any(len > 2 * kBjGroup) ? 2 : NC;
}

template <int C0, int C1, typename T, int NC>
__device__ __forceinline__ void fac_load_part(FacRow<T, NC> &w, uint4 out, int gl, const uint2 *__restrict__ off,
                                              const FacOut &fo, const T *val) {
    const int nch = (w.len + kBjGroup - 1) / kBjGroup;
#pragma unroll
    for (int c = C0; c < C1; ++c) {
        const int e = gl + kBjGroup * c;
        w.at[c] = e < w.d ? out.x * fo.win + e : e > w.d ? out.y * fo.win + (e - w.d - 1) : out.y;
        if (out.w && e < w.len && e != w.d) w.at[c] = fo.place[out.w - 1 + e];
    }
#pragma unroll
    for (int c = C0; c < C1; ++c) w.a[c] = gl + kBjGroup * c < w.len ? val[w.s0 + gl + kBjGroup * c] : T(0);
#pragma unroll
    for (int b = 0; b < kAhead; ++b)
#pragma unroll
        for (int c = C0; c < C1; ++c) {
            const uint2 o = 8 * b < w.d && c < nch ? off[(size_t)(w.tab + b * nch + c) * kBjGroup + gl]
                                                   : make_uint2(0u, 0u);
            w.off[2 * b][c] = o.x;
            w.off[2 * b + 1][c] = o.y;
        }
}

// Registers that no row of the wavefront needs (see fac_regs) are left as they are.
template <typename T, int NC>
__device__ __forceinline__ void fac_row_load(FacRow<T, NC> &w, uint4 m, uint4 out, int gl,
                                             const unsigned *__restrict__ piv, const uint2 *__restrict__ off,
                                             const FacOut &fo, const T *val) {
    w.s0 = (int)m.x;
    w.len = (int)(m.y & 0xffu);
    w.d = (int)((m.y >> 8) & 0xffu);
    w.tab = m.z;
    w.l0 = m.w;
    const int regs = fac_regs<NC>(w.len);
    fac_load_part<0, 1>(w, out, gl, off, fo, val);
    w.piv = gl < w.d ? piv[w.l0 + gl] : 0u;
    if constexpr (NC > 1)
        if (regs > 1) fac_load_part<1, 2>(w, out, gl, off, fo, val);
    if constexpr (NC > 2)
        if (regs > 2) fac_load_part<2, NC>(w, out, gl, off, fo, val);
}

// L entries 4 B .. 4 B + 3 of a row: their u_kj (an entry without one loads the pivot, unused)
template <int B, int M, typename T, int NC>
__device__ __forceinline__ void fac_load_u(const FacRow<T, NC> &w, const T *val, T (&u)[4][M]) {
    constexpr int K0 = 4 * B;
    const unsigned p[4] = {row_bcast<K0>(w.piv), row_bcast<K0 + 1>(w.piv), row_bcast<K0 + 2>(w.piv),
                           row_bcast<K0 + 3>(w.piv)};
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int c = 0; c < M; ++c) u[k][c] = val[p[k] + ((w.off[B][c] >> (8 * k)) & 0xffu)];
}

// L entry K: l_ik = a_ik u_kk^-1 (lane K's product, final since only earlier L
// entries update entry K), then the row's entries that row k has too
template <int K, int M, typename T, int NC>
__device__ __forceinline__ void fac_step(FacRow<T, NC> &w, T pv, const T (&u)[4][M]) {
    const T lik = row_bcast<K>(w.a[0] * pv);
#pragma unroll
    for (int c = 0; c < M; ++c) {
        const T t = w.a[c] - lik * u[K & 3][c];
        w.a[c] = (w.off[K / 4][c] & (0xffu << (8 * (K & 3)))) ? t : w.a[c];
    }
}

template <int B, int M, typename T, int NC>
__device__ __forceinline__ void fac_chain(FacRow<T, NC> &w, T pv, const T (&u)[4][M]) {
    fac_step<4 * B>(w, pv, u);
    fac_step<4 * B + 1>(w, pv, u);
    fac_step<4 * B + 2>(w, pv, u);
    fac_step<4 * B + 3>(w, pv, u);
}

// One row of up to M registers, once every row that it uses is final: the u_kj of its
// first sixteen L entries in one round of loads, then their chain; more L entries one at
// a time.
template <int M, typename T, int NC>
__device__ __forceinline__ void fac_row_m(FacRow<T, NC> &w, int gl, const unsigned *__restrict__ piv,
                                          const uint2 *__restrict__ off, const T *val) {
    // uniform: batches, and entries past the sixteenth, that no row of the wavefront has
    const bool b1 = __any(w.d > 4), b2 = __any(w.d > 8), b3 = __any(w.d > 12);
    const T pv = val[w.piv];
    T u0[4][M], u1[4][M], u2[4][M], u3[4][M];
    fac_load_u<0>(w, val, u0);
    if (b1) fac_load_u<1>(w, val, u1);
    if (b2) fac_load_u<2>(w, val, u2);
    if (b3) fac_load_u<3>(w, val, u3);
    fac_chain<0>(w, pv, u0);
    if (b1) fac_chain<1>(w, pv, u1);
    if (b2) fac_chain<2>(w, pv, u2);
    if (b3) fac_chain<3>(w, pv, u3);
    if (gl < w.d) w.a[0] *= pv;
    if (M > 1 && __any(w.d > 8 * kAhead)) {
        const int nch = (w.len + kBjGroup - 1) / kBjGroup;
        for (int k = 8 * kAhead; __any(k < w.d); ++k) {
            const bool in = k < w.d;
            T ak = T(0);
#pragma unroll
            for (int c = 0; c < M; ++c) {
                const T q = __shfl(w.a[c], k & (kBjGroup - 1), kBjGroup);
                if (c == k / kBjGroup) ak = q;
            }
            const unsigned pk = in ? piv[w.l0 + k] : 0u;
            const T lik = in ? ak * val[pk] : T(0);
#pragma unroll
            for (int c = 0; c < M; ++c) {
                const uint2 o2 = in && c < nch ? off[(size_t)(w.tab + (k >> 3) * nch + c) * kBjGroup + gl]
                                               : make_uint2(0u, 0u);
                const unsigned o = ((k & 4 ? o2.y : o2.x) >> (8 * (k & 3))) & 0xffu;
                if (o) w.a[c] -= lik * val[pk + o];
                if (in && gl + kBjGroup * c == k) w.a[c] = lik;
            }
        }
    }
}

// The factored row to val and to the solve's packed copies, its pivot inverted
// (a zero pivot sets the flag).
template <int M, typename T, int NC>
__device__ __forceinline__ void fac_row_store(const FacRow<T, NC> &w, int gl, T *val, T *__restrict__ vl,
                                              T *__restrict__ vu, T *__restrict__ vd,
                                              int *__restrict__ flag) {
#pragma unroll
    for (int c = 0; c < M; ++c) {
        const int e = gl + kBjGroup * c;
        T v = w.a[c];
        if (e == w.d) {
            if (v == T(0)) { atomicOr(flag, 1); v = T(0); }
            else v = T(1) / v;
        }
        if (e < w.len) {
            val[w.s0 + e] = v;
            (e < w.d ? vl : e > w.d ? vu : vd)[w.at[c]] = v;
        }
    }
}

// a wavefront's rows (have: those it has), factored and stored
template <typename T, int NC>
__device__ __forceinline__ void fac_row(FacRow<T, NC> &w, bool have, int gl, const unsigned *__restrict__ piv,
                                        const uint2 *__restrict__ off, T *val, T *__restrict__ vl,
                                        T *__restrict__ vu, T *__restrict__ vd, int *__restrict__ flag) {
    const int regs = fac_regs<NC>(w.len);
    if (regs == 1) {
        fac_row_m<1>(w, gl, piv, off, val);
        if (have) fac_row_store<1>(w, gl, val, vl, vu, vd, flag);
    }
    if constexpr (NC > 1)
        if (regs == 2) {
            fac_row_m<2>(w, gl, piv, off, val);
            if (have) fac_row_store<2>(w, gl, val, vl, vu, vd, flag);
        }
    if constexpr (NC > 2)
        if (regs == NC) {
            fac_row_m<NC>(w, gl, piv, off, val);
            if (have) fac_row_store<NC>(w, gl, val, vl, vu, vd, flag);
        }
}

// One workgroup per block b: values ia[roff[b]] ... ia[roff[b + 1]] of lu, the
// slots of its level pieces (at most TH / kBjGroup each)
// lptr[blev[b]] ... lptr[blev[b + 1]].  src null: lu already holds the values to
// factor.  vl, vu, vd: the solve's packed L, U and inverted diagonal.  STAGED: values
// and piece pointers (npmax + 1 ints) in LDS, so that a barrier waits for LDS accesses
// only and rows are loaded kRing levels ahead.
template <typename T, int NC, bool STAGED, int TH>
__global__ void __launch_bounds__(TH, NC == 1 ? 4 : 2) bj_factor(
    const int *__restrict__ roff, const int *__restrict__ ia, const int *__restrict__ src,
    const double *__restrict__ a, const uint4 *__restrict__ slot, const uint4 *__restrict__ sout,
    const unsigned *__restrict__ piv, const uint2 *__restrict__ off, const int *__restrict__ blev,
    const int *__restrict__ lptr, T *lu, T *__restrict__ vl, T *__restrict__ vu, T *__restrict__ vd,
    FacOut fo, int *__restrict__ flag, int npmax) {
    extern __shared__ double smem[];
    const int b = blockIdx.x;
    const int z0 = ia[roff[b]], nzb = ia[roff[b + 1]] - z0;
    const int l0 = blev[b], nl = blev[b + 1] - l0;
    if (fo.ptr_l) {
        const size_t sl = fo.ptr_l[fo.lev_l[b]], su = fo.ptr_u[fo.lev_u[b]];
        vl += sl * fo.win;
        vu += su * fo.win;
        vd += su;
    }
    int *pp = reinterpret_cast<int *>(smem);
    T *val = STAGED ? reinterpret_cast<T *>(smem + (npmax + 2) / 2) : lu + z0;
    if (src)
        for (int k = threadIdx.x; k < nzb; k += TH) val[k] = (T)a[src[z0 + k]];
    else if (STAGED)
        for (int k = threadIdx.x; k < nzb; k += TH) val[k] = lu[z0 + k];
    if (STAGED)
        for (int k = threadIdx.x; k <= nl; k += TH) pp[k] = lptr[l0 + k];
    else
        __threadfence_block();
    __syncthreads();
    if (nl == 0) return;
    const int gl = threadIdx.x & (kBjGroup - 1), g = threadIdx.x / kBjGroup;
    // piece l's slot of this group: a group without a row takes the piece's last
    // slot (loads stay in range) and stores nothing
    auto slot_of = [&](int l, bool &have) {
        const int lc = min(l, nl - 1);
        const int p0 = STAGED ? pp[lc] : lptr[l0 + lc], p1 = STAGED ? pp[lc + 1] : lptr[l0 + lc + 1];
        have = l < nl && p0 + g < p1;
        return min(p0 + g, p1 - 1);
    };
    // a wavefront none of whose groups has a row in a piece skips the work on it
    if (STAGED) {
        constexpr int kRing = 4;
        FacRow<T, NC> w[kRing];
        bool have[kRing], have1[kRing];
        uint4 m[kRing], o[kRing];
#pragma unroll
        for (int q = 0; q < kRing; ++q) {
            const int sl = slot_of(q, have[q]);
            m[q] = slot[sl];
            o[q] = sout[sl];
        }
#pragma unroll
        for (int q = 0; q < kRing; ++q) fac_row_load(w[q], m[q], o[q], gl, piv, off, fo, val);
#pragma unroll
        for (int q = 0; q < kRing; ++q) {
            const int sl = slot_of(q + kRing, have1[q]);
            m[q] = slot[sl];
            o[q] = sout[sl];
        }
        for (int lb = 0; lb < nl; lb += kRing) {
#pragma unroll
            for (int q = 0; q < kRing; ++q) {
                if (__any(have[q])) fac_row(w[q], have[q], gl, piv, off, val, vl, vu, vd, flag);
                fac_row_load(w[q], m[q], o[q], gl, piv, off, fo, val);
                have[q] = have1[q];
                const int sl = slot_of(lb + q + 2 * kRing, have1[q]);
                m[q] = slot[sl];
                o[q] = sout[sl];
                lds_barrier();
            }
        }
        for (int k = threadIdx.x; k < nzb; k += TH) lu[z0 + k] = val[k];
    } else {
        bool have, have1, have2;
        FacRow<T, NC> w;
        const int sl0 = slot_of(0, have), sl1 = slot_of(1, have1);
        fac_row_load(w, slot[sl0], sout[sl0], gl, piv, off, fo, val);
        uint4 m1 = slot[sl1], o1 = sout[sl1];
        for (int l = 0; l < nl; ++l) {
            FacRow<T, NC> nx;
            fac_row_load(nx, m1, o1, gl, piv, off, fo, val);
            const int sl = slot_of(l + 2, have2);
            const uint4 m2 = slot[sl], o2 = sout[sl];
            if (__any(have)) fac_row(w, have, gl, piv, off, val, vl, vu, vd, flag);
            __threadfence_block();
            __syncthreads();
            w = nx;
            have = have1;
            m1 = m2;
            o1 = o2;
            have1 = have2;
        }
    }
}

// Solve: one wavefront per block.  Only the block's solution and its level
// pointers live in LDS (so that every block of the matrix is resident at once
// and the CU interleaves their dependency chains).  The factor streams from a
// level-ordered packed copy per triangle, which bj_factor writes: slots of one lane or,
// with PAIR, of up to two, W entries to a lane (zero past the row's length, with the row
// itself as the column), up to 64 lanes a level.  A pair's second lane (its row: its own
// spare place) passes its sum to the first.  A row longer than a slot takes further slots
// in earlier levels, for the entries whose rows are final there: each subtracts its share
// from v[r] (with d = 1 in U).  T is the factor's arithmetic type (double, or float for the
// FP32 preconditioner); x and y stay FP64.
// W = 4 and one lane, in FP32 where every row fits it; else 6 in pairs: a row's sum is that
// of entries 0 to 5 and of 6 to 11, whatever lanes they lie in, since FP32 shows a row
// rounded once more (194 672-row box in blocks of 1024, one overlap layer, against FP64:
// 1.09e-7; with slots of 4 1.14e-7).
// What bounds it is one wavefront's instruction issue and LDS latency per level, and
// for many blocks the factor's bytes.  A tetrahedral box's rows have 7 entries a
// triangle (10 next to other blocks) inside a block, 5 on average in blocks of 256 rows,
// 2.5 in blocks of 64; lanes of 8 entries (12 in FP32) read zeros for the rest.
// One overlap layer, us, FP64 / FP32, now, with lanes of 8 and 12, and with rows end to end
// (no padding, a lane pair to a row, twice the levels): 524 288 rows in blocks of 64
// 135 / 116, 179 / 166, 160 / 114; in blocks of 256 48 / 43, 69 / 51, 54 / 50; 194 672 in
// blocks of 1024 40 / 39, 48 / 46, 66 / 65; a band of 61, 9 000 rows, no overlap,
// 262 / 314, 345 / 405, 3565 / 3564.  Only where wide levels are full of long rows are lanes
// of 8 the better in FP64: 27-point stencil, 27 000 rows in blocks of 1024, 58, 52, 114.
template <typename T, int W>
struct BjWin {
    T a[W];
    unsigned c[W / 2];  // local columns, two per word
    unsigned r;
    T d;                // inverted diagonal (U)
    bool mine;
};

// lane s of the block's
template <typename T, int W, bool UPPER>
__device__ __forceinline__ void bj_win_load(BjWin<T, W> &w, unsigned s, bool mine, const T *__restrict__ val,
                                            const unsigned *__restrict__ col, const unsigned short *__restrict__ row,
                                            const T *__restrict__ dinv) {
    using T2 = typename std::conditional<sizeof(T) == 4, float2, double2>::type;
    const T2 *p = reinterpret_cast<const T2 *>(val + W * s);
#pragma unroll
    for (int i = 0; i < W / 2; ++i) {
        const T2 q = p[i];
        w.a[2 * i] = q.x; w.a[2 * i + 1] = q.y;
        w.c[i] = col[W / 2 * s + i];
    }
    w.r = row[s];
    w.d = UPPER ? dinv[s] : T(0);
    w.mine = mine;
}

// the other lane's of a pair
__device__ __forceinline__ float swap_pair(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xb1, 0xf, 0xf, true));
}

// levels loaded ahead: deep enough to cover a memory round trip with the short
// per-level arithmetic, as far as the registers of four wavefronts a SIMD go
template <typename T>
constexpr int bj_ahead() { return sizeof(T) == 4 ? 8 : 7; }

// One triangle of one block: lane t takes the t-th lane of each level (lp: the
// levels' lanes within the block; spare: the first spare place).  The windows are
// loads in flight, kA levels ahead, one per lane and level, each consumed by the same unrolled stage that
// issued it kA stages earlier (no loop-carried register holds a pending load, so
// the compiler's wait counts keep all kA levels in flight).  Every pass runs all
// kA levels (those past the last have no lane with work).  Every lane forms and
// stores s, lanes without a slot to their own spare place vd, so that v[r]'s read
// stays with the window's (rows of one level do not depend on each other, so it
// is final here).
template <typename T, int W, bool PAIR, bool UPPER>
__device__ __forceinline__ void bj_sweep(T *v, T *vd, unsigned spare, int nl, const int *lp, const T *__restrict__ val,
                                         const unsigned *__restrict__ col, const unsigned short *__restrict__ row,
                                         const T *__restrict__ dinv) {
    if (nl <= 0) return;
    constexpr int kA = bj_ahead<T>();
    auto load = [&](BjWin<T, W> &w, int l, int p0, int p1) {
        const int s = p0 + (int)threadIdx.x;
        bj_win_load<T, W, UPPER>(w, min(s, p1 - 1), l < nl && s < p1, val, col, row, dinv);
    };
    BjWin<T, W> wr[kA];
#pragma unroll
    for (int d = 0; d < kA; ++d) {
        const int lc = min(d, nl - 1);
        load(wr[d], d, lp[lc], lp[lc + 1]);
        wave_lds_order();
    }
    // Level lb + d + kA's range is read with the update's values; its window is
    // issued last.
    for (int lb = 0; lb < nl; lb += kA) {
#pragma unroll
        for (int d = 0; d < kA; ++d) {
            const int ln = lb + d + kA, lc = min(ln, nl - 1);
            const int p0 = lp[lc], p1 = lp[lc + 1];
            const BjWin<T, W> &w = wr[d];
            T q0 = T(0), q1 = T(0);
#pragma unroll
            for (int u = 0; u < W; ++u) {
                const T x = v[(u & 1) ? w.c[u / 2] >> 16 : w.c[u / 2] & 0xffffu];
                if (sizeof(T) == 4 || u < W / 2) q0 += w.a[u] * x;
                else q1 += w.a[u] * x;
            }
            const T vr = v[w.r];
            if constexpr (PAIR) q1 = swap_pair(w.r >= spare ? q0 : T(0));
            T s = vr - (q0 + q1);
            if (UPPER) s *= w.d;
            *(w.mine ? v + w.r : vd) = s;
            load(wr[d], ln, p0, p1);
            // one wavefront: the LDS executes its accesses in order, so only
            // the compiler must keep them in program order
            wave_lds_order();
        }
    }
}

// LDS bytes of one block's solve: the solution (T x maxrows) and a spare
// place per lane (T x 64), its L and U level pointers
__host__ __device__ inline size_t bj_solve_lds(size_t tsize, int maxrows, int levl, int levu) {
    return ((tsize * (size_t)(maxrows + 64) + 7) & ~(size_t)7) + 4 * (size_t)(levl + levu + 2);
}

// rowid: global row of each local row (nullptr: block b's rows are the
// contiguous range starting at roff[b]); own: the block's owned local rows,
// the only ones written back (restricted additive Schwarz).  One wavefront per
// block, so that every block of the matrix is resident at once.  (Staging the
// whole block in LDS was measured slower: it limits the resident blocks, and
// one wavefront stages too slowly.)  Per triangle: solve levels blev (per
// block) into lptr (per level, into the level-ordered slots, at most 64 per
// level), the slots' values, columns and rows, U's inverted diagonals.
template <typename T, int W, bool PAIR>
__global__ void __launch_bounds__(64) bj_solve(const int *__restrict__ roff, const int *__restrict__ rowid,
                                               const int *__restrict__ own, const int *__restrict__ blev_l,
                                               const int *__restrict__ lptr_l, const T *__restrict__ val_l,
                                               const unsigned *__restrict__ col_l,
                                               const unsigned short *__restrict__ row_l,
                                               const int *__restrict__ blev_u, const int *__restrict__ lptr_u,
                                               const T *__restrict__ val_u, const unsigned *__restrict__ col_u,
                                               const unsigned short *__restrict__ row_u,
                                               const T *__restrict__ dinv, int maxrows,
                                               const double *__restrict__ x, const double *__restrict__ xdiv,
                                               double *__restrict__ y, double *__restrict__ yn2, const double *skip) {
    extern __shared__ double smem[];
    const double over = skip_word(skip);
    const int b = blockIdx.x;
    const int base = roff[b];
    const int cnt = roff[b + 1] - base;
    char *lds = reinterpret_cast<char *>(smem);
    T *v = reinterpret_cast<T *>(lds);
    // v: the block's rows, then one spare place per lane
    T *vd = v + maxrows + threadIdx.x;
    const int l0 = blev_l[b], nl = blev_l[b + 1] - l0;
    const int u0 = blev_u[b], nu = blev_u[b + 1] - u0;
    const long sl = lptr_l[l0], su = lptr_u[u0];  // the block's first slots
    int *lpl = reinterpret_cast<int *>(lds + ((sizeof(T) * (size_t)(maxrows + 64) + 7) & ~(size_t)7));
    int *lpu = lpl + nl + 1;
    for (int k = threadIdx.x; k <= nl; k += 64) lpl[k] = lptr_l[l0 + k] - (int)sl;
    for (int k = threadIdx.x; k <= nu; k += 64) lpu[k] = lptr_u[u0 + k] - (int)su;
    // stage x (optionally scaled by 1 / xdiv) in batches of kBjStage rows per
    // lane, so that a batch's gathers are in flight together
    constexpr int kBjStage = 16;
    for (int r0 = threadIdx.x; r0 < cnt; r0 += 64 * kBjStage) {
        int g[kBjStage];
        double xv[kBjStage], dv[kBjStage];
#pragma unroll
        for (int k = 0; k < kBjStage; ++k) {
            const int r = min(r0 + 64 * k, cnt - 1);
            g[k] = rowid ? rowid[base + r] : base + r;
        }
#pragma unroll
        for (int k = 0; k < kBjStage; ++k) {
            xv[k] = x[g[k]];
            dv[k] = xdiv ? xdiv[g[k]] : 1.;
        }
#pragma unroll
        for (int k = 0; k < kBjStage; ++k) {
            const int r = r0 + 64 * k;
            if (r < cnt) v[r] = (T)(xdiv ? xv[k] / dv[k] : xv[k]);
        }
    }
    wave_lds_order();
    if (over != 0.) return;
    bj_sweep<T, W, PAIR, false>(v, vd, maxrows, nl, lpl, val_l + W * sl, col_l + W / 2 * sl, row_l + sl, nullptr);
    bj_sweep<T, W, PAIR, true>(v, vd, maxrows, nu, lpu, val_u + W * su, col_u + W / 2 * su, row_u + su, dinv + su);
    const int olo = own[2 * b], ohi = own[2 * b + 1];
    double q = 0.;
    for (int r0 = olo + threadIdx.x; r0 < ohi; r0 += 64 * kBjStage) {
        int g[kBjStage];
#pragma unroll
        for (int k = 0; k < kBjStage; ++k) {
            const int r = min(r0 + 64 * k, ohi - 1);
            g[k] = rowid ? rowid[base + r] : base + r;
        }
#pragma unroll
        for (int k = 0; k < kBjStage; ++k) {
            const int r = r0 + 64 * k;
            if (r < ohi) {
                const double yr = (double)v[r];
                y[g[k]] = yr;
                q += yr * yr;
            }
        }
    }
    if (yn2) {  // this block's share of ||y||^2 (owned rows partition the rows)
        q = wave_reduce(q);
        if (threadIdx.x == 0) yn2[b] = q;
    }
}

// Global ILU(0) solve of a matrix whose solution fits the LDS, in one
// workgroup: y = U^-1 L^-1 (x / xdiv).  Rows lie in level order, one lane per
// row; a level wider than the workgroup is cut into pieces.  Per slot a padded
// window of KW entries, so a piece's loads have fixed addresses and go out kA
// pieces ahead; the chain per piece is one batch of LDS reads, the row's sum and
// one LDS store.  One wavefront needs no barrier (the LDS runs its accesses in
// order); wider workgroups meet at one per piece.  A 4 141-node slice (141 levels
// per triangle) takes 52 us, and its factorisation 205 us; one launch per level
// and triangle (the form that matrices outside these limits keep) took 707 to
// 1075 us, and 1500 us.  The chain bounds it: 0.18 us per level.
// kOneWidth: rows per level, on average over both triangles, up to which one
// workgroup is used: a launch per level costs 2.5 us in the solve and 10 us in
// the factorisation, one workgroup 0.2 us per piece of up to 1024 rows and 1.5
// us per 64 rows of a level.
constexpr long kOneWidth = 256;

template <int KW>
struct IluWin {
    double a[KW];
    unsigned c[KW / 2];
    unsigned rm;
    double d;
    bool have;
};

template <int KW, int TH, bool UPPER>
__device__ __forceinline__ void ilu0_sweep(double *v, double *spare, int np, const int *pp,
                                           const unsigned *__restrict__ row, const unsigned short *__restrict__ col,
                                           const double *__restrict__ val, const double *__restrict__ dinv) {
    constexpr int kA = KW <= 4 ? (TH > 256 ? 4 : 8) : KW == 8 ? (TH > 256 ? 2 : 4) : KW == 16 ? 2 : 1;
    const int t = threadIdx.x;
    auto load = [&](IluWin<KW> &w, int p) {
        const int pc = min(p, np - 1), p0 = pp[pc], p1 = pp[pc + 1];
        const int sl = min(p0 + t, p1 - 1);  // a lane without a row reads the piece's last
        w.have = p < np && p0 + t < p1;
        w.rm = row[sl];
        const double2 *pa = reinterpret_cast<const double2 *>(val + (size_t)sl * KW);
        const unsigned *pc2 = reinterpret_cast<const unsigned *>(col + (size_t)sl * KW);
#pragma unroll
        for (int k = 0; k < KW / 2; ++k) {
            const double2 q = pa[k];
            w.a[2 * k] = q.x;
            w.a[2 * k + 1] = q.y;
            w.c[k] = pc2[k];
        }
        w.d = UPPER ? dinv[sl] : 0.;
    };
    IluWin<KW> w[kA];
#pragma unroll
    for (int q = 0; q < kA; ++q) load(w[q], q);
    for (int pb = 0; pb < np; pb += kA) {
#pragma unroll
        for (int q = 0; q < kA; ++q) {
            const int r = (int)(w[q].rm & 0xffffu), kn = (int)(w[q].rm >> 16);
            double xv[KW];
#pragma unroll
            for (int k = 0; k < KW; ++k) xv[k] = v[(k & 1) ? w[q].c[k / 2] >> 16 : w[q].c[k / 2] & 0xffffu];
            const double vr = v[r];
            double s = 0.;
#pragma unroll
            for (int k = 0; k < KW; ++k) s += k < kn ? w[q].a[k] * xv[k] : 0.;
            s = vr - s;
            if (UPPER) s *= w[q].d;
            *(w[q].have ? v + r : spare) = s;
            load(w[q], pb + q + kA);
            if (TH > 64) lds_barrier();
            else wave_lds_order();
        }
    }
}

template <int KW, int TH>
__global__ void __launch_bounds__(TH) ilu0_solve(int n, int npl, const int *__restrict__ ppl,
                                                 const unsigned *__restrict__ row_l,
                                                 const unsigned short *__restrict__ col_l,
                                                 const double *__restrict__ val_l, int npu,
                                                 const int *__restrict__ ppu, const unsigned *__restrict__ row_u,
                                                 const unsigned short *__restrict__ col_u,
                                                 const double *__restrict__ val_u, const double *__restrict__ x,
                                                 const double *__restrict__ xdiv, double *__restrict__ y,
                                                 double *__restrict__ yn2, const double *skip) {
    extern __shared__ double smem[];
    const double over = skip_word(skip);
    double *v = smem, *spare = v + n + threadIdx.x;
    int *pl = reinterpret_cast<int *>(v + n + TH), *pu = pl + npl + 1;
    for (int k = threadIdx.x; k <= npl; k += TH) pl[k] = ppl[k];
    for (int k = threadIdx.x; k <= npu; k += TH) pu[k] = ppu[k];
    constexpr int kStage = 8;  // loads in flight per lane
    for (int i0 = threadIdx.x; i0 < n; i0 += TH * kStage) {
        double q[kStage], d[kStage];
#pragma unroll
        for (int u = 0; u < kStage; ++u) {
            const int i = min(i0 + TH * u, n - 1);
            q[u] = x[i];
            d[u] = xdiv ? xdiv[i] : 1.;
        }
#pragma unroll
        for (int u = 0; u < kStage; ++u)
            if (i0 + TH * u < n) v[i0 + TH * u] = xdiv ? q[u] / d[u] : q[u];
    }
    __syncthreads();
    if (over != 0.) return;
    ilu0_sweep<KW, TH, false>(v, spare, npl, pl, row_l, col_l, val_l, nullptr);
    __syncthreads();
    ilu0_sweep<KW, TH, true>(v, spare, npu, pu, row_u, col_u, val_u, val_u + (size_t)n * KW);
    __syncthreads();
    double q = 0.;
    for (int i = threadIdx.x; i < n; i += TH) {
        const double s = v[i];
        y[i] = s;
        q += s * s;
    }
    if (yn2) {
        q = wave_reduce(q);
        __syncthreads();
        if ((threadIdx.x & 63) == 0) v[threadIdx.x >> 6] = q;
        __syncthreads();
        if (threadIdx.x == 0) {
            double tot = 0.;
            for (int k = 0; k < TH / 64; ++k) tot += v[k];
            yn2[0] = tot;
        }
    }
}

static inline int nblk(long n, int bs) { return (int)((n + bs - 1) / bs); }

// ---- Schur-complement preconditioner (schur.c:887-981 form, :1583-1626 apply)
// Largest boundary set of one subdomain: its dense block is inverted in LDS.
constexpr int kSchurMax = 128;

__global__ void vgather(long n, const int *__restrict__ src, const double *__restrict__ in, double *__restrict__ out) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[src[i]];
}

__global__ void vscatter(long n, const int *__restrict__ dst, const double *__restrict__ in, double *__restrict__ out) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) out[dst[i]] = in[i];
}

// column c of every subdomain's E at once (schur_form_local's dense E column)
__global__ void schur_col_rhs(int nI, const int *__restrict__ e_ia, const int *__restrict__ e_loc,
                              const double *__restrict__ ev, int c, double *__restrict__ t) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nI) return;
    double v = 0.;
    for (int k = e_ia[i]; k < e_ia[i + 1]; ++k)
        if (e_loc[k] == c) v = ev[k];
    t[i] = v;
}

// S_b(:, c) = -F_b y for every subdomain with more than c boundary unknowns
__global__ void schur_col_store(int nG, const int *__restrict__ f_ia, const int *__restrict__ f_ja,
                                const double *__restrict__ fv, const double *__restrict__ y,
                                const int *__restrict__ gsub, const int *__restrict__ glocal,
                                const int *__restrict__ goff, const long *__restrict__ soff, int c,
                                double *__restrict__ S) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nG) return;
    const int b = gsub[j], n = goff[b + 1] - goff[b];
    if (c >= n) return;
    double s = 0.;
    for (int k = f_ia[j]; k < f_ia[j + 1]; ++k) s += fv[k] * y[f_ja[k]];
    S[soff[b] + (long)c * n + glocal[j]] = -s;
}

__global__ void schur_add_c(long nc, const long *__restrict__ pos, const int *__restrict__ src,
                            const double *__restrict__ a, double *__restrict__ S) {
    long k = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (k < nc) S[pos[k]] += a[src[k]];
}

// In-place Gauss-Jordan inversion of each subdomain's dense S_b (column major,
// n <= kSchurMax) in LDS, with partial pivoting: at step k the first row of
// largest |a(r, k)|, r >= k, is swapped into row k; the interchanges are undone
// as column swaps in reverse order at the end.  Waves own columns, lanes own
// rows (two rows per lane), so every LDS access of a wave is one contiguous
// column segment.  A zero pivot sets *flag.
__global__ void __launch_bounds__(256) schur_invert(const int *__restrict__ goff, const long *__restrict__ soff,
                                                    double *__restrict__ S, int *__restrict__ flag) {
    extern __shared__ double sm[];  // n x n block, pivot row, pivot column, n pivots, 2 flags
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n = goff[b + 1] - goff[b];
    if (n == 0) return;
    double *a = sm, *rk = sm + n * n, *fk = rk + n;
    int *perm = reinterpret_cast<int *>(fk + n);
    int &s_piv = perm[n], &s_bad = perm[n + 1];
    double *g = S + soff[b];
    for (int e = tid; e < n * n; e += 256) a[e] = g[e];
    if (tid == 0) s_bad = 0;
    __syncthreads();
    for (int k = 0; k < n; ++k) {
        if (wv == 0) {
            double best = -1.;
            int bi = n;
            for (int r = k + lane; r < n; r += 64) {
                const double v = fabs(a[k * n + r]);
                if (v > best) { best = v; bi = r; }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const double ob = __shfl_xor(best, off);
                const int oi = __shfl_xor(bi, off);
                if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
            }
            if (lane == 0) {
                s_piv = bi;
                perm[k] = bi;
                if (!(best > 0.)) s_bad = 1;
            }
        }
        __syncthreads();
        if (s_bad) break;
        const int p = s_piv;
        if (p != k)
            for (int c = tid; c < n; c += 256) {
                const double t = a[c * n + k];
                a[c * n + k] = a[c * n + p];
                a[c * n + p] = t;
            }
        __syncthreads();
        const double inv = 1.0 / a[k * n + k];
        for (int c = tid; c < n; c += 256) {
            rk[c] = c == k ? inv : a[c * n + k] * inv;
            fk[c] = a[k * n + c];
        }
        __syncthreads();
        const double f0 = lane < n ? fk[lane] : 0., f1 = lane + 64 < n ? fk[lane + 64] : 0.;
        for (int c = wv; c < n; c += 4) {
            const double rc = rk[c];
            double *col = a + c * n;
            if (lane < n)
                col[lane] = lane == k ? rc : (c == k ? -f0 * inv : col[lane] - f0 * rc);
            if (lane + 64 < n)
                col[lane + 64] = lane + 64 == k ? rc : (c == k ? -f1 * inv : col[lane + 64] - f1 * rc);
        }
        __syncthreads();
    }
    if (s_bad) {
        if (tid == 0) atomicOr(flag, 1);
        return;
    }
    for (int k = n - 1; k >= 0; --k) {
        const int p = perm[k];
        if (p != k)
            for (int r = tid; r < n; r += 256) {
                const double t = a[k * n + r];
                a[k * n + r] = a[p * n + r];
                a[p * n + r] = t;
            }
        __syncthreads();
    }
    for (int e = tid; e < n * n; e += 256) g[e] = a[e];
}

// Middle of the apply, one workgroup per subdomain: v = x_G - F u (u = M_B^-1 x_I),
// y_G = S_b^-1 v, written to y (original rows) and to yG (boundary numbering).
__global__ void __launch_bounds__(kSchurMax) schur_mid(const int *__restrict__ goff, const long *__restrict__ soff,
                                                       const double *__restrict__ Sinv, const int *__restrict__ grow,
                                                       const int *__restrict__ f_ia, const int *__restrict__ f_ja,
                                                       const double *__restrict__ fv, const double *__restrict__ x,
                                                       const double *__restrict__ u, double *__restrict__ y,
                                                       double *__restrict__ yG) {
    __shared__ double v[kSchurMax];
    const int b = blockIdx.x, r = threadIdx.x;
    const int g0 = goff[b], n = goff[b + 1] - g0;
    if (r < n) {
        const int j = g0 + r;
        double s = x[grow[j]];
        for (int k = f_ia[j]; k < f_ia[j + 1]; ++k) s -= fv[k] * u[f_ja[k]];
        v[r] = s;
    }
    __syncthreads();
    if (r < n) {
        const double *Sb = Sinv + soff[b];
        double s = 0.;
        for (int c = 0; c < n; ++c) s += Sb[(long)c * n + r] * v[c];
        yG[g0 + r] = s;
        y[grow[g0 + r]] = s;
    }
}

// t_I = x_I - E y_G
__global__ void schur_back(int nI, const int *__restrict__ irow, const int *__restrict__ e_ia,
                           const int *__restrict__ e_ja, const double *__restrict__ ev, const double *__restrict__ x,
                           const double *__restrict__ yG, double *__restrict__ t) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nI) return;
    double s = x[irow[i]];
    for (int k = e_ia[i]; k < e_ia[i + 1]; ++k) s -= ev[k] * yG[e_ja[k]];
    t[i] = s;
}

// ---- host helpers ---------------------------------------------------------------
static int ensure_work(fvp_csr *A, int m) {
    if (A->m_alloc >= m) return 0;
    long n = A->n;
    if (A->Q.alloc((size_t)gs_ldq(n) * (m + 1)) || A->w.alloc(n) || A->r.alloc(n) || A->z.alloc(n) ||
        A->part.alloc((size_t)kGsBlocks * (kChunk + 1)) || A->scal.alloc(16) || A->hdev.alloc(2 * (m + 2) + 2) ||
        A->Hd.alloc((size_t)(m + 1) * m) || A->gd.alloc(m + 1) || A->csd.alloc(m) || A->snd.alloc(m))
        return -1;
    if (A->hstat.alloc(m + 1)) return -1;
    A->m_alloc = m;
    return 0;
}

// out[0..nc) = Q[:, 0..nc)^T w and out[nc] = w . w (device), chunks of kChunk
// columns; the w . w term rides on the last chunk.  skip: see mdot_kernel.
static void multidot(hipStream_t s, long n, const double *w, const double *Q, long ldq, int nc, double *part,
                     double *out, const double *skip) {
    const int nb = gs_blocks(n);
    for (int c0 = 0; c0 < nc; c0 += kChunk) {
        const int k = std::min(kChunk, nc - c0);
        const int last = c0 + k == nc;
        kMdot[k - 1](s, nb, n, w, Q + c0 * ldq, ldq, last, part, skip);
        reduce_cols<<<k + last, kThreads, 0, s>>>(nb, part, out + c0, skip);
    }
}

// w -= Q[:, 0..nc) coef in chunks of kChunk columns; *norm2 = the updated w . w
// (norm2 null: left as the gs_blocks(n) partials in part)
static void multiaxpy(hipStream_t s, long n, double *w, const double *Q, long ldq, int nc, const double *coef,
                      double *part, double *norm2, const double *skip) {
    const int nb = gs_blocks(n);
    for (int c0 = 0; c0 < nc; c0 += kChunk) {
        const int k = std::min(kChunk, nc - c0);
        kAxpy[k - 1](s, nb, n, w, Q + c0 * ldq, ldq, coef + c0, part, skip);
    }
    if (norm2) reduce_cols<<<1, kThreads, 0, s>>>(nb, part, norm2, skip);
}

using Op = std::function<int(const double *, double *)>;

// Restarted right-preconditioned GMRES (gmres.c:26-201) with the host kept off
// the critical path: the Hessenberg column, the Givens rotations and the
// residual estimate are updated on the device; each Arnoldi step's estimate is
// written to pinned host memory and read one step later, while the next step
// is already queued (a cycle that has converged runs one extra, discarded
// step, whose kernels return once they have read that).  Classical
// Gram-Schmidt with a second pass only when the first one
// cancelled more than half of ||w||^2 (reorthogonalise = 1), always (2) or
// never (0).  A cycle ends early once the estimate meets tol * ||b||.
// Device and host memory of one GMRES solve: the basis Q (gs_ldq(n) x (m+1)),
// work vectors w, r, z (gs_ldq(n) each), reduction partials part
// (kGsBlocks x (kChunk+1)), scalars sc (16), per-step coefficients hdev
// (2 (m+2) + 2), the Hessenberg matrix Hd ((m+1) x m), Givens pairs and rhs;
// hstat (host, kSlot (m+1)): slot j receives step j's {estimate,
// h_{j+1,j}}, slot m the squared norms {||r||^2, ||b||^2}.
// With tag hstat is pinned memory that the kernels write, a tag last (counted
// up, so that no slot ever holds the awaited tag beforehand), and the host polls
// the tag: an event per step costs the stream a barrier packet each.  Without,
// each step's pair is copied and read right after the step (same control flow
// and results, one synchronisation per step).
// skip: set, while a step is queued, to the device word that the end of the
// cycle makes nonzero: the products and solves that look at it leave early.
// diag: the preconditioner is this diagonal, and the kernels that write a basis
// vector write z = diag q as well.
struct GmresWork {
    double *Q, *w, *r, *z, *part, *sc, *hdev, *Hd, *gd, *csd, *snd;
    double *hstat;
    double *tag;
    const double **skip;
    const double *diag;
};

// doubles of a GmresWork carved from one device buffer (each piece 256-byte aligned)
static size_t gmres_work_doubles(long n, int m) {
    auto up = [](size_t v) { return (v + 31) & ~(size_t)31; };
    const size_t ldq = (size_t)gs_ldq(n);
    return up(ldq * (m + 1)) + 3 * up(ldq) + up((size_t)kGsBlocks * (kChunk + 1)) + up(16) + up(2 * (m + 2) + 2) +
           up((size_t)(m + 1) * m) + 3 * up(m + 1);
}
static GmresWork gmres_work_carve(double *base, long n, int m) {
    auto up = [](size_t v) { return (v + 31) & ~(size_t)31; };
    const size_t ldq = (size_t)gs_ldq(n);
    GmresWork wk{};
    double *q = base;
    auto take = [&](size_t cnt) { double *r = q; q += up(cnt); return r; };
    wk.Q = take(ldq * (m + 1));
    wk.w = take(ldq);
    wk.r = take(ldq);
    wk.z = take(ldq);
    wk.part = take((size_t)kGsBlocks * (kChunk + 1));
    wk.sc = take(16);
    wk.hdev = take(2 * (m + 2) + 2);
    wk.Hd = take((size_t)(m + 1) * m);
    wk.gd = take(m + 1);
    wk.csd = take(m + 1);
    wk.snd = take(m + 1);
    return wk;
}

static int gmres_core(const GmresWork &W, hipStream_t s, long n, const Op &A, const Op &M, const double *b,
                      double *x, const fvp_gmres_params *p, fvp_gmres_stats *st, const GmresZero *zero = nullptr);

const double *gmres_skip(const fvp_csr *W) { return W->skip; }

int gmres_device(fvp_csr *W, hipStream_t s, long n, const Op &A, const Op &M, const double *b, double *x,
                 const fvp_gmres_params *p, fvp_gmres_stats *st, const GmresZero *zero, const double *diag) {
    const int m = p->dim_krylov;
    if (m < 1 || m > 63) { set_error("dim_krylov must be 1..63"); return -1; }
    if (p->reorthogonalise < 0 || p->reorthogonalise > 2) { set_error("reorthogonalise must be 0, 1 or 2"); return -1; }
    if (ensure_work(W, m)) return -1;
    GmresWork wk{W->Q.p, W->w.p, W->r.p, W->z.p, W->part.p, W->scal.p, W->hdev.p, W->Hd.p, W->gd.p, W->csd.p,
                 W->snd.p, W->hstat.p, &W->hstat.tag, &W->skip, diag};
    const int rc = gmres_core(wk, s, n, A, M, b, x, p, st, zero);
    W->skip = nullptr;
    return rc;
}

static int gmres_core(const GmresWork &W, hipStream_t s, long n, const Op &A, const Op &M, const double *b,
                      double *x, const fvp_gmres_params *p, fvp_gmres_stats *st, const GmresZero *zero) {
    const int m = p->dim_krylov;
    double *Q = W.Q, *w = W.w, *r = W.r, *z = W.z, *part = W.part, *sc = W.sc;
    // h1, h2: first / second pass coefficients (j+1 dots, then ||w||^2); stat: {estimate, h_{j+1,j}}
    double *h1 = W.hdev, *h2 = W.hdev + (m + 2), *stat = W.hdev + 2 * (m + 2);
    // device scalars: sc[0] ||r||^2, sc[1] ||b||^2; for bases past kGsCols columns sc[2] first-pass ||w||^2
    // after projection, sc[3] second-pass ||w||^2, sc[4] reorthogonalisation flag; ctl[1], ctl[2] as gs_finish has them
    double *n1 = sc + 2, *n2 = sc + 3, *flag = sc + 4, *ctl = sc + 4;
    const long ldq = gs_ldq(n);
    const int mode = p->reorthogonalise, nb = gs_nb(n);
    // the second pass's partials: the other half of part, or r (free during a cycle) where they need more
    constexpr int kHalf = kGsNb / 2 * (kGsCols + 1);
    double *part2 = nb <= kGsNb / 2 ? part + kHalf : r;
    fvp_gmres_stats stats{0, 0, 0, 0., 0.};
    double hn2[2] = {0., 0.};
    // queues r = b - r and waits for ||r||^2 and ||b||^2
    auto residual = [&]() -> int {
        gs_residual<<<nb, kGsThreads, 0, s>>>(n, b, r, part);
        double *slot = W.hstat + (size_t)kSlot * m;
        gs_post<2><<<1, kGsThreads, 0, s>>>(nb, part, sc, W.tag ? slot : nullptr, W.tag ? ++*W.tag : 0.);
        FVP_HIP(hipGetLastError());
        if (W.tag) {
            if (slot_wait(s, slot, *W.tag)) return -1;
        } else {
            FVP_HIP(hipMemcpyAsync(slot, sc, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
            FVP_HIP(hipStreamSynchronize(s));
        }
        for (int k = 0; k < 2; ++k) hn2[k] = slot[k];
        return 0;
    };
    if (zero) hn2[0] = hn2[1] = zero->norm2;
    else if (A(x, r) || residual()) return -1;
    double beta = std::sqrt(hn2[0]), normb = std::sqrt(hn2[1]);
    double error = normb > 0 ? beta / normb : 0.;
    if (beta == 0. || error < p->tol) {
        stats.converged = 1; stats.residual = beta; stats.error = error;
        if (st) *st = stats;
        return 0;
    }
    const double thr = p->tol * normb;
    int restarts = 0, converged = 0, total = 0;
    double step_tag = 0.;  // of the step before
    bool x_zero = zero;  // x is still zero, the residual still b
    while (restarts <= p->max_restarts && !converged) {
        gs_start<<<nblk(n, 256), 256, 0, s>>>(n, x_zero ? b : r, x_zero ? zero->d_norm2 : sc, beta, Q, W.diag, z, W.gd, m + 1, ctl);
        int k = m;
        for (int j = 0; j <= m; ++j) {
            const double prev_tag = step_tag;
            if (j < m) {  // queue Arnoldi step j
                const double *qj = Q + (size_t)j * ldq;
                double *slot = W.tag ? W.hstat + (size_t)kSlot * j : nullptr;
                if (W.tag) step_tag = ++*W.tag;
                if (W.skip) *W.skip = j < kGsCols ? ctl + 1 : nullptr;
                if (W.diag) { if (A(z, w)) return -1; }
                else if (M) { if (M(qj, z)) return -1; if (A(z, w)) return -1; }
                else if (A(qj, w)) return -1;
                if (j < kGsCols) {
                    const GsStep &g = kGs[j];
                    g.dots<<<nb, kGsThreads, 0, s>>>(n, w, Q, ldq, part);
                    g.update<<<nb, kGsThreads, 0, s>>>(n, w, Q, ldq, mode != 0, part, part2, h1, ctl);
                    g.finish<<<nb + 1, kGsThreads, 0, s>>>(mode, m, n, w, Q, ldq, part, part2, h1, thr, W.Hd, W.csd,
                                                           W.snd, W.gd, ctl, stat, slot, step_tag, W.diag, z);
                } else {
                    // first pass: h1 = Q^T w, ||w||^2 -> h1[j+1]; w -= Q h1, ||w||^2 -> n1
                    // (single pass: arnoldi_finish reduces ||w||^2 itself)
                    multidot(s, n, w, Q, ldq, j + 1, part, h1, nullptr);
                    multiaxpy(s, n, w, Q, ldq, j + 1, h1, part, mode ? n1 : nullptr, nullptr);
                    if (mode) {
                        reorth_decide<<<1, 64, 0, s>>>(h1 + j + 1, n1, mode, flag);
                        multidot(s, n, w, Q, ldq, j + 1, part, h2, flag);
                        multiaxpy(s, n, w, Q, ldq, j + 1, h2, part, n2, flag);
                    }
                    double *qn = Q + (size_t)(j + 1) * ldq;
                    arnoldi_finish<<<std::min(nblk(n, 256), kFinishBlocks), 256, 0, s>>>(
                        j, m, h1, h2, n1, n2, mode ? flag : nullptr, W.Hd, W.csd, W.snd, W.gd, stat, slot, step_tag, n,
                        w, qn, mode ? nullptr : part, gs_blocks(n));
                    if (W.diag) vmul<<<nblk(n, 256), 256, 0, s>>>(n, qn, W.diag, z);
                }
                FVP_HIP(hipGetLastError());
                if (!W.tag) {
                    FVP_HIP(hipMemcpyAsync(W.hstat + (size_t)kSlot * j, stat, 2 * sizeof(double),
                                           hipMemcpyDeviceToHost, s));
                    FVP_HIP(hipStreamSynchronize(s));
                }
            }
            if (j > 0) {  // read step j-1 (while step j runs, when pipelined)
                const double *slot = W.hstat + (size_t)kSlot * (j - 1);
                if (W.tag && slot_wait(s, slot, prev_tag)) return -1;
                ++total;
                const double est = slot[0], hn = slot[1];
                if (est < thr || !(hn > 1e-16)) { k = j; break; }
            }
        }
        if (W.skip) *W.skip = nullptr;
        const bool own = M && !W.diag;  // M is a call of its own
        gs_solution<<<std::min(nblk(n, 256), kFinishBlocks), 256, 0, s>>>(n, k, m, W.Hd, W.gd, Q, ldq, W.diag, !own,
                                                                         own ? w : x);
        if (own) {
            if (M(w, x_zero ? x : z)) return -1;
            if (!x_zero) vadd<<<nblk(n, 256), 256, 0, s>>>(n, z, x);
        }
        x_zero = false;
        if (A(x, r)) return -1;
        if (residual()) return -1;
        beta = std::sqrt(hn2[0]);
        error = beta / normb;
        if (error < p->tol) converged = 1;
        else ++restarts;
    }
    stats.restarts = converged ? restarts : restarts - 1;
    stats.iterations = total;
    stats.converged = converged;
    stats.residual = beta;
    stats.error = error;
    if (st) *st = stats;
    return converged ? 0 : FVP_ERR_NOCONV;
}


// Restarted GMRES with deflated restarts (gmresFH, gmres.c:212-405, with
// arnoldi, :412-511, and deflate, :527-849): each cycle runs the Arnoldi
// process for A M from column K to m (no early exit within a cycle, as there),
// solves the least-squares problem min || Q^T r - Hbar y || on the host, sets
// x += M Q y and recomputes the true residual; before the next cycle the k
// harmonic Ritz vectors of smallest magnitude (real and imaginary parts of a
// complex pair) of H = H_m + h_{m+1,m}^2 f e_m^T, f = H_m^-T e_m, are kept at
// the front of the basis, with the matching Hbar block, and the next cycle
// continues from column K (the number kept).  The Gram-Schmidt passes, the
// products and the basis updates run on the device; the small dense problems
// on the host.  k = 0 is plain restarted GMRES with convergence checked per
// cycle.
int gmres_deflated(fvp_csr *Wc, hipStream_t s, long n, const Op &A, const Op &M, const double *b, double *x,
                   const fvp_gmres_params *p, int k, fvp_gmres_stats *st) {
    const int m = p->dim_krylov;
    if (m < 2 || m > 63) { set_error("dim_krylov must be 2..63"); return -1; }
    if (k < 0 || 2 * k >= m) { set_error("deflation count k must be 0 <= 2k < dim_krylov"); return -1; }
    if (p->reorthogonalise < 0 || p->reorthogonalise > 2) { set_error("reorthogonalise must be 0, 1 or 2"); return -1; }
    if (ensure_work(Wc, m)) return -1;
    const long ldq = gs_ldq(n);
    if (k && Wc->Qk.n < (size_t)ldq * (2 * k + 1) && Wc->Qk.alloc((size_t)ldq * (2 * k + 1))) return -1;
    double *Q = Wc->Q.p, *w = Wc->w.p, *r = Wc->r.p, *z = Wc->z.p, *part = Wc->part.p, *sc = Wc->scal.p;
    double *h1 = Wc->hdev.p, *h2 = Wc->hdev.p + (m + 2), *coef = Wc->hdev.p;
    double *n1 = sc + 2, *n2 = sc + 3;
    const int nb = nblk(n, 256);
    auto host = [&](const double *d, double *hp, int cnt) -> int {
        FVP_HIP(hipMemcpyAsync(hp, d, sizeof(double) * cnt, hipMemcpyDeviceToHost, s));
        FVP_HIP(hipStreamSynchronize(s));
        return 0;
    };
    auto norm = [&](const double *v, double &out) -> int {
        if (dot_async(s, n, v, v, part, sc)) return -1;
        double q;
        if (host(sc, &q, 1)) return -1;
        out = std::sqrt(q);
        return 0;
    };
    fvp_gmres_stats stats{0, 0, 0, 0., 0.};
    // r = b - A x
    if (A(x, r)) return -1;
    vrsub<<<nb, 256, 0, s>>>(n, b, r);
    double beta, normb;
    if (norm(r, beta) || norm(b, normb)) return -1;
    double error = normb > 0 ? beta / normb : 0.;
    if (beta == 0. || error < p->tol) {
        stats.converged = 1; stats.residual = beta; stats.error = error;
        if (st) *st = stats;
        return 0;
    }
    vaxpby<<<nb, 256, 0, s>>>(n, 1. / beta, r, 0., Q);
    std::vector<double> H((size_t)(m + 1) * m, 0.);  // row-major (m+1) x m
    auto Hr = [&](int i, int j) -> double & { return H[(size_t)i * m + j]; };
    std::vector<double> hh(2 * (m + 2));
    int K = 0, restarts = 0, total = 0, converged = 0;
    while (restarts <= p->max_restarts) {
        // Arnoldi from column K
        int j = K;
        while (j < m) {
            const double *qj = Q + (size_t)j * ldq;
            if (M) { if (M(qj, z)) return -1; if (A(z, w)) return -1; }
            else if (A(qj, w)) return -1;
            multidot(s, n, w, Q, ldq, j + 1, part, h1, nullptr);
            multiaxpy(s, n, w, Q, ldq, j + 1, h1, part, n1, nullptr);
            if (p->reorthogonalise) {
                multidot(s, n, w, Q, ldq, j + 1, part, h2, nullptr);
                multiaxpy(s, n, w, Q, ldq, j + 1, h2, part, n2, nullptr);
            }
            if (host(Wc->hdev.p, hh.data(), 2 * (m + 2)) || host(sc + 2, hh.data() + 2 * (m + 2) - 2, 2)) return -1;
            for (int i = 0; i <= j; ++i) Hr(i, j) = hh[i] + (p->reorthogonalise ? hh[m + 2 + i] : 0.);
            const double ww = hh[2 * (m + 2) - 2 + (p->reorthogonalise ? 1 : 0)];
            const double hn = std::sqrt(std::max(ww, 0.));
            Hr(j + 1, j) = hn;
            ++total;
            if (hn < 1e-16) break;  // lucky breakdown: column j + 1 is not formed (gmres.c:485)
            vaxpby<<<nb, 256, 0, s>>>(n, 1. / hn, w, 0., Q + (size_t)(j + 1) * ldq);
            ++j;
        }
        // least squares on the j computed columns, right-hand side Q^T r
        multidot(s, n, r, Q, ldq, j + 1, part, h1, nullptr);
        std::vector<double> c(j + 1), y, Hs((size_t)(j + 1) * j);
        if (host(h1, c.data(), j + 1)) return -1;
        for (int a = 0; a <= j; ++a)
            for (int bcol = 0; bcol < j; ++bcol) Hs[(size_t)a * j + bcol] = Hr(a, bcol);
        if (j == 0 || !dense::lstsq(j + 1, j, Hs, c, y)) { set_error("GMRES: singular Hessenberg matrix"); return -1; }
        FVP_HIP(hipMemcpyAsync(coef, y.data(), sizeof(double) * j, hipMemcpyHostToDevice, s));
        lincomb<<<nb, 256, 0, s>>>(n, w, Q, ldq, j, coef);
        if (M) { if (M(w, z)) return -1; }
        else vcopy<<<nb, 256, 0, s>>>(n, w, z);
        vadd<<<nb, 256, 0, s>>>(n, z, x);
        if (A(x, r)) return -1;
        vrsub<<<nb, 256, 0, s>>>(n, b, r);
        if (norm(r, beta)) return -1;
        error = beta / normb;
        if (error < p->tol) { converged = 1; break; }
        if (++restarts > p->max_restarts) break;
        int Knew = 0;
        if (k && j == m) {
            // harmonic Ritz vectors of H = H_m + hb^2 f e_m^T (deflate, gmres.c:600-760)
            const double hb = Hr(m, m - 1);
            std::vector<double> Hm((size_t)m * m), HmT((size_t)m * m), f(m, 0.);
            for (int a = 0; a < m; ++a)
                for (int bcol = 0; bcol < m; ++bcol) {
                    Hm[(size_t)a * m + bcol] = Hr(a, bcol);
                    HmT[(size_t)bcol * m + a] = Hr(a, bcol);
                }
            f[m - 1] = 1.;
            bool ok = dense::lu_solve(m, HmT, f);
            std::vector<double> Hh = Hm, wr, wi;
            if (ok)
                for (int a = 0; a < m; ++a) Hh[(size_t)a * m + m - 1] += hb * hb * f[a];
            ok = ok && dense::eig(m, Hh, wr, wi);
            std::vector<int> ord(m);
            std::iota(ord.begin(), ord.end(), 0);
            if (ok)
                std::stable_sort(ord.begin(), ord.end(), [&](int a, int bcol) {
                    return wr[a] * wr[a] + wi[a] * wi[a] < wr[bcol] * wr[bcol] + wi[bcol] * wi[bcol];
                });
            std::vector<double> X;  // column-major m x jj
            for (int i = 0, q = 0; ok && i < k; ++i) {
                const int pos = ord[i + q];
                std::vector<std::complex<double>> v;
                if (wi[pos] != 0.) {
                    // the member of the pair with positive imaginary part: real and imaginary parts
                    const std::complex<double> lam(wr[pos], std::fabs(wi[pos]));
                    ok = dense::eigvec(m, Hh, lam, v);
                    for (int a = 0; a < m; ++a) X.push_back(v[a].real());
                    for (int a = 0; a < m; ++a) X.push_back(v[a].imag());
                    ++q;
                } else {
                    ok = dense::eigvec(m, Hh, std::complex<double>(wr[pos], 0.), v);
                    for (int a = 0; a < m; ++a) X.push_back(v[a].real());
                }
            }
            const int jj = (int)(X.size() / m);
            ok = ok && jj > 0 && jj + 1 <= m && dense::orthonormalise(m, jj, X);
            if (ok) {
                // Qk = Q_m X on the device; p = hb q_{m+1} - hb^2 Q_m f, orthogonalised against Qk
                double *Qk = Wc->Qk.p;
                for (int cc = 0; cc < jj; ++cc) {
                    FVP_HIP(hipMemcpyAsync(coef, &X[(size_t)cc * m], sizeof(double) * m, hipMemcpyHostToDevice, s));
                    lincomb<<<nb, 256, 0, s>>>(n, Qk + (size_t)cc * ldq, Q, ldq, m, coef);
                    FVP_HIP(hipStreamSynchronize(s));  // coef is reused by the next column
                }
                std::vector<double> pc(m + 1);
                for (int a = 0; a < m; ++a) pc[a] = -hb * hb * f[a];
                pc[m] = hb;
                FVP_HIP(hipMemcpyAsync(coef, pc.data(), sizeof(double) * (m + 1), hipMemcpyHostToDevice, s));
                double *pm = Qk + (size_t)jj * ldq;
                lincomb<<<nb, 256, 0, s>>>(n, pm, Q, ldq, m + 1, coef);
                for (int cc = 0; cc < jj; ++cc) {  // modified Gram-Schmidt
                    double dot;
                    if (dot_async(s, n, pm, Qk + (size_t)cc * ldq, part, sc) || host(sc, &dot, 1)) return -1;
                    vaxpby<<<nb, 256, 0, s>>>(n, -dot, Qk + (size_t)cc * ldq, 1., pm);
                }
                double betak;
                if (norm(pm, betak)) return -1;
                ok = betak > 0.;
                if (ok) {
                    vaxpby<<<nb, 256, 0, s>>>(n, 1. / betak, pm, 0., pm);
                    FVP_HIP(hipMemcpyAsync(Q, Qk, sizeof(double) * ldq * (jj + 1), hipMemcpyDeviceToDevice, s));
                    // the new Hbar: Omega = X^T H X - hb^2 (X^T f) s^T, row jj = betak s^T, s = X's last row
                    std::vector<double> HX((size_t)m * jj, 0.), Xf(jj, 0.);
                    for (int a = 0; a < m; ++a)
                        for (int cc = 0; cc < jj; ++cc) {
                            double acc = 0.;
                            for (int q2 = 0; q2 < m; ++q2) acc += Hh[(size_t)a * m + q2] * X[(size_t)cc * m + q2];
                            HX[(size_t)a * jj + cc] = acc;
                        }
                    for (int cc = 0; cc < jj; ++cc)
                        for (int a = 0; a < m; ++a) Xf[cc] += X[(size_t)cc * m + a] * f[a];
                    std::fill(H.begin(), H.end(), 0.);
                    for (int r1 = 0; r1 < jj; ++r1)
                        for (int cc = 0; cc < jj; ++cc) {
                            double om = 0.;
                            for (int a = 0; a < m; ++a) om += X[(size_t)r1 * m + a] * HX[(size_t)a * jj + cc];
                            Hr(r1, cc) = om - hb * hb * Xf[r1] * X[(size_t)cc * m + m - 1];
                        }
                    for (int cc = 0; cc < jj; ++cc) Hr(jj, cc) = betak * X[(size_t)cc * m + m - 1];
                    Knew = jj;
                }
            }
        }
        if (!Knew) {  // plain restart from the residual
            std::fill(H.begin(), H.end(), 0.);
            vaxpby<<<nb, 256, 0, s>>>(n, 1. / beta, r, 0., Q);
        }
        K = Knew;
        FVP_HIP(hipGetLastError());
    }
    stats.restarts = converged ? restarts : restarts - 1;
    stats.iterations = total;
    stats.converged = converged;
    stats.residual = beta;
    stats.error = error;
    if (st) *st = stats;
    return converged ? 0 : FVP_ERR_NOCONV;
}

}  // namespace fvp

// ================================================================================
// decomp-style CSR entry points
// ================================================================================
using namespace fvp;

namespace fvp {

template <int R>
static void csr_gemv_launch(fvp_csr *A, double alpha, const double *x, double beta, double *y) {
    csr_gemv_kernel<R><<<nblk(A->n, R), 256, 0, A->stream>>>(A->n, A->ia.p, A->ja.p, A->a.p, alpha, x, beta, y, A->skip);
}
static int csr_gemv_impl(fvp_csr *A, double alpha, const double *x, double beta, double *y) {
    // rows per workgroup: see csr_gemv_kernel
    const long n = A->n, nnz = A->nnz;
    if (nnz <= 9 * n && A->longest <= 256) csr_gemv_launch<128>(A, alpha, x, beta, y);
    else if (nnz <= 40 * n) csr_gemv_launch<64>(A, alpha, x, beta, y);
    else csr_gemv_launch<16>(A, alpha, x, beta, y);
    FVP_HIP(hipGetLastError());
    return 0;
}

static int build_one(fvp_csr *A, const std::vector<int> &diag, const std::vector<int> &lrows,
                     const std::vector<int> &urows);

// level sets of the L (forward) and U (backward) dependency DAGs
static int build_levels(fvp_csr *A, const std::vector<int> &diag) {
    const int n = A->n;
    std::vector<int> lev(n, 0), ulev(n, 0);
    int nl = 0, nu = 0;
    for (int i = 0; i < n; ++i) {
        int l = 0;
        for (int k = A->ia_h[i]; k < diag[i]; ++k) l = std::max(l, lev[A->ja_h[k]] + 1);
        lev[i] = l;
        nl = std::max(nl, l + 1);
    }
    for (int i = n - 1; i >= 0; --i) {
        int l = 0;
        for (int k = diag[i] + 1; k < A->ia_h[i + 1]; ++k) l = std::max(l, ulev[A->ja_h[k]] + 1);
        ulev[i] = l;
        nu = std::max(nu, l + 1);
    }
    auto group = [&](const std::vector<int> &lv, int nlev, std::vector<int> &ptr, std::vector<int> &rows) {
        ptr.assign(nlev + 1, 0);
        for (int i = 0; i < n; ++i) ptr[lv[i] + 1]++;
        for (int l = 0; l < nlev; ++l) ptr[l + 1] += ptr[l];
        rows.resize(n);
        std::vector<int> fill(ptr.begin(), ptr.end() - 1);
        for (int i = 0; i < n; ++i) rows[fill[lv[i]]++] = i;
    };
    std::vector<int> lrows, urows;
    group(lev, nl, A->lptr_h, lrows);
    group(ulev, nu, A->uptr_h, urows);
    if (build_one(A, diag, lrows, urows)) return -1;
    if (!A->one && (A->lrows.upload(lrows.data(), n) || A->urows.upload(urows.data(), n))) return -1;
    A->levels = true;
    return 0;
}

// The tables of bj_factor: roff, bia, bja, bdiag describe the blocks (local
// columns, entry positions over all blocks), rows the local rows as slots in
// level order (block b's slots are [roff[b], roff[b + 1])), out per slot its
// slots in the solve's L (x) and U (y), counted within the block, and w as in FacOut; no row is longer than
// 64 entries.
template <typename Col, typename Row>
static int factor_tables(FactorTab &F, int nb, const std::vector<int> &roff, const std::vector<int> &bia,
                         const std::vector<Col> &bja, const std::vector<int> &bdiag, const std::vector<Row> &rows,
                         int maxrow) {
    const int total = roff[nb];
    std::vector<uint4> slot(total);
    std::vector<unsigned> piv;
    size_t units = 0;  // offset batches of one 16-lane group
    for (int i = 0; i < total; ++i) {
        const int len = bia[i + 1] - bia[i], d = bdiag[i] - bia[i];
        units += (size_t)((d + 7) / 8) * ((len + kBjGroup - 1) / kBjGroup);
    }
    if (units > 0xffffffffu) { set_error("too many entries for the factorisation's tables"); return -1; }
    std::vector<unsigned char> off(units * kBjGroup * 8, (unsigned char)0);
    piv.reserve(bdiag.empty() ? 0 : (size_t)bia[total] / 2);
    int widest = 0;
    for (int b = 0; b < nb; ++b) widest = std::max(widest, roff[b + 1] - roff[b]);
    std::vector<int> pos(widest, -1);
    size_t tab = 0;
    for (int b = 0; b < nb; ++b) {
        const int base = roff[b], z0 = bia[base];
        for (int sl = base; sl < roff[b + 1]; ++sl) {
            const int i = base + (int)rows[sl];
            const int e0 = bia[i], len = bia[i + 1] - e0, d = bdiag[i] - e0;
            const int nch = (len + kBjGroup - 1) / kBjGroup;
            slot[sl] = make_uint4((unsigned)(e0 - z0), (unsigned)len | ((unsigned)d << 8), (unsigned)tab,
                                  (unsigned)piv.size());
            for (int j = 0; j < len; ++j) pos[bja[e0 + j]] = j;
            for (int k = 0; k < d; ++k) {
                const int row = base + (int)bja[e0 + k], kd = bdiag[row];
                piv.push_back((unsigned)(kd - z0));
                for (int m = kd + 1; m < bia[row + 1]; ++m) {
                    const int j = pos[bja[m]];
                    if (j < 0) continue;
                    const size_t unit = tab + (size_t)(k / 8) * nch + j / kBjGroup;
                    off[(unit * kBjGroup + j % kBjGroup) * 8 + k % 8] = (unsigned char)(m - kd);
                }
            }
            for (int j = 0; j < len; ++j) pos[bja[e0 + j]] = -1;
            tab += (size_t)((d + 7) / 8) * nch;
        }
    }
    if (piv.empty()) piv.push_back(0u);
    if (off.empty()) off.resize(8 * kBjGroup, (unsigned char)0);
    F.nc = maxrow <= kBjGroup ? 1 : maxrow <= 2 * kBjGroup ? 2 : 4;
    long longs = 0;
    for (int i = 0; i < total; ++i) longs += bia[i + 1] - bia[i] > 2 * kBjGroup;
    F.mostly_long = 8 * longs > total;
    return F.slot.upload(slot.data(), slot.size()) || F.piv.upload(piv.data(), piv.size()) ||
           F.off.upload(reinterpret_cast<const uint2 *>(off.data()), off.size() / 8);
}

// pieces of at most `width` slots of each level
static void level_pieces(const std::vector<int> &lptr, int width, std::vector<int> &pieces) {
    pieces.assign(1, lptr[0]);
    for (size_t l = 0; l + 1 < lptr.size(); ++l)
        for (int p = lptr[l]; p < lptr[l + 1]; p += width) pieces.push_back(std::min(p + width, lptr[l + 1]));
}

// Global ILU(0) in one workgroup (see ilu0_solve): the tables of its
// factorisation and of its solve, where the pattern allows them.
static int build_one(fvp_csr *A, const std::vector<int> &diag, const std::vector<int> &lrows,
                     const std::vector<int> &urows) {
    const int n = A->n;
    A->one = false;
    if (hipDeviceGetAttribute(&A->lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, A->device) != hipSuccess)
        A->lds_max = 64 * 1024;
    int maxrow = 0, maxtri = 1;
    for (int i = 0; i < n; ++i) {
        maxrow = std::max(maxrow, A->ia_h[i + 1] - A->ia_h[i]);
        maxtri = std::max({maxtri, diag[i] - A->ia_h[i], A->ia_h[i + 1] - diag[i] - 1});
    }
    const int win = maxtri <= 4 ? 4 : maxtri <= 8 ? 8 : maxtri <= 16 ? 16 : 32;
    if (maxrow > 64 || maxtri > win || n > 65536) return 0;
    // wide levels are worth a launch each (the whole device on one level); one
    // workgroup's factorisation takes 32 or 64 rows of a level at a time
    const long levels = (long)(A->lptr_h.size() - 1 + A->uptr_h.size() - 1);
    if (2L * n > kOneWidth * levels) return 0;
    // threads: the count that makes the sweep's pieces cheapest (a piece's cost
    // grows with the wavefronts that meet at its barrier)
    std::vector<int> pieces[2];
    double best = 1e300;
    for (int th : {64, 256, 1024}) {
        std::vector<int> pl, pu;
        level_pieces(A->lptr_h, th, pl);
        level_pieces(A->uptr_h, th, pu);
        const size_t lds = 8 * (size_t)(n + th) + 4 * (pl.size() + pu.size());
        const double cost = (double)(pl.size() + pu.size()) * (th == 64 ? 1.0 : th == 256 ? 1.3 : 1.8);
        if (lds > (size_t)A->lds_max || cost >= best) continue;
        best = cost;
        A->o_threads = th;
        A->o_lds = lds;
        pieces[0].swap(pl);
        pieces[1].swap(pu);
    }
    if (pieces[0].empty()) return 0;
    A->o_win = win;
    std::vector<uint4> out(n, make_uint4(0u, 0u, 0u, 0u));  // by row at first, then by slot of L's level order
    for (int t = 0; t < 2; ++t) {
        const std::vector<int> &order = t ? urows : lrows;
        std::vector<unsigned> row(n);
        std::vector<unsigned short> col((size_t)n * win, 0);
        for (int sl = 0; sl < n; ++sl) {
            const int i = order[sl], k0 = t ? diag[i] + 1 : A->ia_h[i], k1 = t ? A->ia_h[i + 1] : diag[i];
            row[sl] = (unsigned)i | ((unsigned)(k1 - k0) << 16);
            for (int k = 0; k < win; ++k) {
                const size_t q = (size_t)sl * win + k;
                col[q] = (unsigned short)(k0 + k < k1 ? A->ja_h[k0 + k] : i);
            }
            (t ? out[i].y : out[i].x) = (unsigned)sl;
        }
        IluTri &T = A->otri[t];
        T.npieces = (int)pieces[t].size() - 1;
        T.nslots = n;
        if (T.pptr.upload(pieces[t].data(), pieces[t].size()) || T.row.upload(row.data(), n) ||
            T.col.upload(col.data(), col.size()) || T.val.alloc((size_t)n * win + (t ? n : 0)))
            return -1;
        FVP_HIP(hipMemsetAsync(T.val.p, 0, sizeof(double) * T.val.n, A->stream));  // the windows' padding stays zero
    }
    std::vector<uint4> by(n);
    for (int sl = 0; sl < n; ++sl) by[sl] = out[lrows[sl]];
    std::vector<int> fp, fp1024;
    level_pieces(A->lptr_h, 512 / kBjGroup, fp);
    level_pieces(A->lptr_h, 1024 / kBjGroup, fp1024);
    A->o_fthreads = maxrow <= kBjGroup && 1.2 * fp1024.size() <= fp.size() ? 1024 : 512;
    if (A->o_fthreads == 1024) fp.swap(fp1024);
    const int head[4] = {0, n, 0, (int)fp.size() - 1};
    fp.insert(fp.begin(), head, head + 4);
    if (A->o_fptr.upload(fp.data(), fp.size()) ||
        factor_tables(A->ofac, 1, {0, n}, A->ia_h, A->ja_h, diag, lrows, maxrow) || A->ofac.out.upload(by.data(), n))
        return -1;
    for (const void *f :
         {(const void *)ilu0_solve<4, 64>, (const void *)ilu0_solve<8, 64>, (const void *)ilu0_solve<16, 64>,
          (const void *)ilu0_solve<32, 64>, (const void *)ilu0_solve<4, 256>, (const void *)ilu0_solve<8, 256>,
          (const void *)ilu0_solve<16, 256>, (const void *)ilu0_solve<32, 256>, (const void *)ilu0_solve<4, 1024>,
          (const void *)ilu0_solve<8, 1024>, (const void *)ilu0_solve<16, 1024>, (const void *)ilu0_solve<32, 1024>})
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, A->lds_max);
    A->one = true;
    return 0;
}

// The solve's packed layout with W entries to a lane, S to a slot; maxrows: of any block
static int build_pack(BjPack &P, int W, int S, int nb, int maxrows, const BjTables &t) {
    const std::vector<int> &roff = t.roff, &bia = t.bia, &bdiag = t.bdiag;
    const std::vector<unsigned short> &bja = t.bja, &rows_l = t.rows;
    const int total = roff[nb];
    std::vector<int> lev;
    std::vector<uint4> out(total, make_uint4(0u, 0u, 0u, 0u));  // by row at first, then by slot of L's level order
    std::vector<unsigned> place;
    struct Slot {
        int row, n;     // local row, entries
        int first;      // in `order`
        bool main;
    };
    std::vector<int> order, at, count, step, by, single, pair;
    std::vector<Slot> slots;
    for (int tri = 0; tri < 2; ++tri) {
        std::vector<unsigned> col;
        std::vector<unsigned short> srow;
        std::vector<int> sb(nb + 1, 0), sp(1, 0);
        int &levmax = tri ? P.levmax_u : P.levmax_l;
        levmax = 0;
        for (int b = 0; b < nb; ++b) {
            const int base = roff[b], cnt = roff[b + 1] - base;
            lev.assign(cnt, 0);
            order.clear();
            slots.clear();
            step.clear();
            // rows in dependency order: the row's entries by level, the last S in its own
            // slot; a row of further slots waits until each can precede the next
            for (int q = 0; q < cnt; ++q) {
                const int r = tri ? cnt - 1 - q : q, i = base + r;
                const int k0 = tri ? bdiag[i] + 1 : bia[i], n = (tri ? bia[i + 1] : bdiag[i]) - k0;
                const int f = (int)order.size();
                for (int k = 0; k < n; ++k) order.push_back(k0 + k);
                int l = 0;
                if (n > S)  // few entries: by insertion
                    for (int k = 1; k < n; ++k) {
                        const int e = order[f + k], le = lev[bja[e]];
                        int j = k;
                        for (; j > 0 && lev[bja[order[f + j - 1]]] > le; --j) order[f + j] = order[f + j - 1];
                        order[f + j] = e;
                    }
                for (int k = 0; k < n; ++k) l = std::max(l, lev[bja[order[f + k]]] + 1);
                for (int j = 1, e = n - S; e > 0; ++j, e -= S) l = std::max(l, lev[bja[order[f + e - 1]]] + 1 + j);
                lev[r] = l;
                slots.push_back({r, std::min(n, S), f + std::max(0, n - S), true});
                step.push_back(l);
            }
            int nl = 0;
            for (int s : step) nl = std::max(nl, s + 1);
            count.assign(nl + 1, 0);
            for (int q = 0; q < cnt; ++q) count[step[q]] += slots[q].n > W ? 2 : 1;
            for (int q = 0; q < cnt; ++q) {  // the further slots, where there is room
                const Slot m = slots[q];
                const int r = m.row, i = base + r, n = tri ? bia[i + 1] - bdiag[i] - 1 : bdiag[i] - bia[i];
                int hi = step[q];
                for (int e = n - S; e > 0; e -= S) {
                    const int f0 = m.first - (n - S) + std::max(0, e - S), ne = std::min(e, S), lanes = ne > W ? 2 : 1;
                    // not before its rows are final, nor so early that the slots before it are
                    int lo = lev[bja[order[f0 + ne - 1]]] + 1;
                    for (int k = e - S, j = 1; k > 0; k -= S, ++j)
                        lo = std::max(lo, lev[bja[order[m.first - (n - S) + k - 1]]] + 1 + j);
                    int best = hi - 1;  // the latest level with free lanes in its last piece
                    for (int s = hi - 1; s >= lo; --s)
                        if (count[s] % 64 && count[s] % 64 + lanes <= 64) { best = s; break; }
                    hi = best;
                    slots.push_back({r, ne, f0, false});
                    step.push_back(hi);
                    count[hi] += lanes;
                }
            }
            // level by level, pieces of at most 64 lanes, slots of two lanes first
            at.assign(nl + 1, 0);
            for (int l = 0; l < nl; ++l) at[l + 1] = at[l] + count[l];
            const int s0 = (int)srow.size();
            for (int l = 0; l < nl; ++l)
                for (int p = at[l]; p < at[l + 1]; p += 64) sp.push_back(s0 + std::min(p + 64, at[l + 1]));
            sb[b + 1] = (int)sp.size() - 1;
            levmax = std::max(levmax, sb[b + 1] - sb[b]);
            srow.resize(s0 + at[nl]);
            col.resize((size_t)srow.size() * (W / 2));
            by.assign(slots.size(), 0);
            single.assign(at.begin(), at.end());
            for (size_t q = 0; q < slots.size(); ++q)
                if (slots[q].n > W) single[step[q]] += 2;
            pair = at;
            for (size_t q = 0; q < slots.size(); ++q) {
                const Slot &m = slots[q];
                const bool two = m.n > W;
                const int in = two ? pair[step[q]] : single[step[q]], sl = s0 + in;
                (two ? pair : single)[step[q]] += two ? 2 : 1;
                by[q] = sl;
                srow[sl] = (unsigned short)m.row;
                if (two) srow[sl + 1] = (unsigned short)(maxrows + (in + 1 - at[step[q]]) % 64);
                for (int k = 0; k < (two ? S : W); k += 2) {
                    auto c = [&](int k) { return (unsigned)(k < m.n ? bja[order[m.first + k]] : m.row); };
                    col[(size_t)sl * (W / 2) + k / 2] = c(k) | c(k + 1) << 16;
                }
                if (m.main) (tri ? out[base + m.row].y : out[base + m.row].x) = (unsigned)(sl - s0);
            }
            // rows of several slots in either triangle: each entry's place
            for (size_t q = 0; q < slots.size(); ++q) {
                const Slot &m = slots[q];
                const int i = base + m.row, len = bia[i + 1] - bia[i];
                const bool several = std::max(bdiag[i] - bia[i], bia[i + 1] - bdiag[i] - 1) > S;
                if (!several) continue;
                if (!out[i].w) {
                    out[i].w = (unsigned)place.size() + 1;
                    place.resize(place.size() + len, 0);
                }
                for (int k = 0; k < m.n; ++k)
                    place[out[i].w - 1 + (order[m.first + k] - bia[i])] = (unsigned)((by[q] - s0) * W + k);
            }
        }
        if ((tri ? P.col_u : P.col_l).upload(col.data(), col.size()) ||
            (tri ? P.row_u : P.row_l).upload(srow.data(), srow.size()) ||
            (tri ? P.lev_u : P.lev_l).upload(sb.data(), nb + 1) ||
            (tri ? P.lptr_u : P.lptr_l).upload(sp.data(), sp.size()))
            return -1;
    }
    {
        std::vector<uint4> by(total);
        for (int b = 0; b < nb; ++b)
            for (int sl = roff[b]; sl < roff[b + 1]; ++sl) by[sl] = out[roff[b] + rows_l[sl]];
        if (P.out.upload(by.data(), by.size()) || P.place.upload(place.data(), place.size())) return -1;
    }
    P.win = W;
    return 0;
}

static void bj_attrs(int lds_max);

// The most pieces of one block, by kFacThreads
static std::array<int, 5> most_pieces(int nb, const std::vector<int> &blev, const std::vector<int> &lptr) {
    std::array<int, 5> most{};
    for (int b = 0; b < nb; ++b) {
        std::array<int, 5> m{};
        for (int l = blev[b]; l < blev[b + 1]; ++l)
            for (int w = 0; w < 5; ++w) m[w] += (lptr[l + 1] - lptr[l] + (64 >> w) - 1) >> (6 - w);
        for (int w = 0; w < 5; ++w) most[w] = std::max(most[w], m[w]);
    }
    return most;
}

// The factorisation's levels (blev per block into lptr) in pieces, at the cheapest width
static int factor_pieces(FacPieces &F, int nb, const std::vector<int> &blev, const std::vector<int> &lptr,
                         const std::array<int, 5> &pieces, int maxnz, const FactorTab &tab, size_t vb, int lds_max) {
    static_assert(sizeof(kFacThreads) == 5 * sizeof(int) && kFacThreads[0] / kBjGroup == 64 && kFacThreads[4] / kBjGroup == 4);
    const int nc = tab.nc;
    double best = 1e300;
    const char *given = getenv("FVP_BJ_FACTOR_THREADS");  // forces the threads: a tuning and test knob
    F.threads = 0;
    for (int w = 0; w < 5; ++w) {
        const int th = kFacThreads[w], most = pieces[w];
        if (given && (nc > 1 ? std::min(atoi(given), 512) : atoi(given)) != th) continue;
        // Values staged in LDS wherever a block fits, but not where many FP64 rows have
        // more than 32 entries: four registers a row spill in that form.  Whole builds,
        // staged against in place: 67 / 75 us (276 blocks of 512 rows, FP32), 200 / 307
        // (1024 with one overlap layer, FP32), 323 / 365 (the same, FP64), 517 / 549
        // (1000 blocks of 1024 with overlap, FP32); at worst 91 / 83 (276 blocks of
        // 512, FP64), all with 512 threads; FP64, one row of 41 among tridiagonal ones,
        // blocks of 1024 with overlap, 900 / 1142; all of 41, blocks of 64, 436 / 353.
        const size_t lds = (size_t)maxnz * vb + 8 * (size_t)((most + 2) / 2);
        const bool staged = lds <= (size_t)lds_max && !(vb == 8 && tab.mostly_long);
        const double cost = fac_cost(th, nc, vb, nb, maxnz, staged ? lds : 0, lds_max, most);
        if (cost >= best) continue;
        best = cost;
        F.threads = th;
        F.most = most;
        F.lds = lds;
        F.staged = staged;
    }
    if (!F.threads) { set_error("FVP_BJ_FACTOR_THREADS must be 64, 128, 256, 512 or 1024"); return -1; }
    const int width = F.threads / kBjGroup;
    std::vector<int> fb(nb + 1, 0), fp(1, 0);
    for (int b = 0; b < nb; ++b) {
        for (int l = blev[b]; l < blev[b + 1]; ++l)
            for (int p = lptr[l]; p < lptr[l + 1]; p += width) fp.push_back(std::min(p + width, lptr[l + 1]));
        fb[b + 1] = (int)fp.size() - 1;
    }
    return F.lev.upload(fb.data(), nb + 1) || F.lptr.upload(fp.data(), fp.size()) ? -1 : 0;
}

// Block-local CSR and the per-block level sets of L.  Block b owns rows
// [b bs, (b+1) bs); with overlap > 0 its local rows are the owned rows plus
// `overlap` layers of their graph neighbours (sorted by global row, so the
// local ILU(0) follows the global row order), and only the owned rows of its
// solve are kept (restricted additive Schwarz).
static int build_bj(fvp_csr *A) {
    const int n = A->n, BS = A->bs;
    const bool given = !A->bstart.empty();
    const int nb = given ? (int)A->bstart.size() - 1 : (n + BS - 1) / BS;
    A->tables.reset();
    auto tables = std::make_unique<BjTables>();
    std::vector<int> &roff = tables->roff, &bia = tables->bia, &bdiag = tables->bdiag;
    std::vector<unsigned short> &bja = tables->bja, &rows_l = tables->rows;
    roff.assign(nb + 1, 0);
    bia.assign(1, 0);
    std::vector<int> rowid, own(2 * (size_t)nb), bsrc;
    std::vector<int> stamp(n, -1), loc(n, 0), ext, frontier, next;
    for (int b = 0; b < nb; ++b) {
        const int lo = given ? A->bstart[b] : b * BS, hi = given ? A->bstart[b + 1] : std::min(n, lo + BS);
        ext.clear();
        frontier.clear();
        for (int i = lo; i < hi; ++i) { stamp[i] = b; ext.push_back(i); frontier.push_back(i); }
        for (int layer = 0; layer < A->overlap; ++layer) {
            next.clear();
            for (int i : frontier)
                for (int k = A->ia_h[i]; k < A->ia_h[i + 1]; ++k) {
                    const int j = A->ja_h[k];
                    if (stamp[j] != b) { stamp[j] = b; ext.push_back(j); next.push_back(j); }
                }
            frontier.swap(next);
        }
        std::sort(ext.begin(), ext.end());
        const int cnt = (int)ext.size();
        if (cnt > 65535) { set_error("block-Jacobi ILU(0): a block has more than 65535 rows"); return -1; }
        for (int r = 0; r < cnt; ++r) loc[ext[r]] = r;
        const int olo = (int)(std::lower_bound(ext.begin(), ext.end(), lo) - ext.begin());
        own[2 * (size_t)b] = olo;
        own[2 * (size_t)b + 1] = olo + (hi - lo);
        for (int r = 0; r < cnt; ++r) {
            const int i = ext[r];
            int d = -1;
            for (int k = A->ia_h[i]; k < A->ia_h[i + 1]; ++k) {
                const int j = A->ja_h[k];
                if (stamp[j] != b) continue;
                if (j == i) d = (int)bsrc.size();
                bsrc.push_back(k);
                bja.push_back((unsigned short)loc[j]);
            }
            if (d < 0) { set_error("zero diagonal on row " + std::to_string(i)); return FVP_ERR_PIVOT; }
            bdiag.push_back(d);
            bia.push_back((int)bsrc.size());
            rowid.push_back(i);
        }
        roff[b + 1] = roff[b] + cnt;
    }
    const int total = roff[nb];
    std::vector<int> blev_l(nb + 1, 0), lptr_l(1, 0);
    rows_l.resize(total);
    std::vector<int> lev;
    int maxnz = 0, maxrow = 0, maxrows = 0, longest = 0;
    for (int b = 0; b < nb; ++b) {
        const int base = roff[b], cnt = roff[b + 1] - base;
        maxrows = std::max(maxrows, cnt);
        maxnz = std::max(maxnz, bia[base + cnt] - bia[base]);
        for (int i = base; i < base + cnt; ++i) {
            maxrow = std::max(maxrow, bia[i + 1] - bia[i]);
            longest = std::max({longest, bdiag[i] - bia[i], bia[i + 1] - bdiag[i] - 1});
        }
        // the factorisation's levels
        lev.assign(cnt, 0);
        int nl = 0;
        for (int r = 0; r < cnt; ++r) {
            const int i = base + r;
            int l = 0;
            for (int k = bia[i]; k < bdiag[i]; ++k) l = std::max(l, lev[bja[k]] + 1);
            lev[r] = l;
            nl = std::max(nl, l + 1);
        }
        std::vector<int> c(nl + 1, 0);
        for (int r = 0; r < cnt; ++r) c[lev[r] + 1]++;
        for (int l = 0; l < nl; ++l) c[l + 1] += c[l];
        std::vector<int> fill(c.begin(), c.end() - 1);
        for (int r = 0; r < cnt; ++r) rows_l[base + fill[lev[r]]++] = (unsigned short)r;
        for (int l = 0; l < nl; ++l) lptr_l.push_back(base + c[l + 1]);
        blev_l[b + 1] = blev_l[b] + nl;
    }
    if (maxrow > 64) { set_error("block-Jacobi ILU(0) supports rows of at most 64 block entries"); return -1; }
    if (maxnz > 65535) { set_error("block-Jacobi ILU(0): more than 65535 entries in one block"); return -1; }
    const bool ident = A->overlap == 0;  // rows of block b are [b bs, ...): no row list needed
    if (A->b_ia.upload(bia.data(), total + 1) || A->b_src.upload(bsrc.data(), bsrc.size()) ||
        A->b_roff.upload(roff.data(), nb + 1) ||
        A->b_own.upload(own.data(), own.size()) || (!ident && A->b_rowid.upload(rowid.data(), total)))
        return -1;
    if (ident) A->b_rowid.release();
    if (factor_tables(A->fac, nb, roff, bia, bja, bdiag, rows_l, maxrow)) return -1;
    A->b_lu.release(); A->val_l.release(); A->val_u.release(); A->dinv.release();
    A->b_lu32.release(); A->val32_l.release(); A->val32_u.release(); A->dinv32.release();
    A->pack[0].win = A->pack[1].win = 0;
    A->b_longest = longest;
    A->b_maxnz = maxnz;
    A->b_maxrows = maxrows;
    if (hipDeviceGetAttribute(&A->lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, A->device) != hipSuccess)
        A->lds_max = 64 * 1024;
    // per-kernel attributes (shared by every matrix): allow the device maximum;
    // each build checks its own block against it
    bj_attrs(A->lds_max);
    const std::array<int, 5> pieces = most_pieces(nb, blev_l, lptr_l);
    for (int f32 = 0; f32 < 2; ++f32)
        if (factor_pieces(A->fp[f32], nb, blev_l, lptr_l, pieces, maxnz, A->fac, f32 ? sizeof(float) : sizeof(double),
                          A->lds_max))
            return -1;
    A->tables = std::move(tables);
    A->nblk = nb;
    A->bj = true;
    return 0;
}

// A precision's layout of the solve
static int bj_layout(fvp_csr *A, bool f32) {
    const int w = f32 && A->b_longest > 4;
    if (A->pack[w].win) return 0;
    if (build_pack(A->pack[w], w ? 6 : 4, w ? 12 : 4, A->nblk, A->b_maxrows, *A->tables)) return -1;
    if (A->b_longest <= 4 || A->pack[!w].win) A->tables.reset();
    return 0;
}

int csr_create_impl(int device, int n, const int *ia, const int *ja, fvp_csr **out);
static int precon_build_impl(fvp_csr *A, int type);
static int precon_apply_impl(fvp_csr *A, const double *x, double *y, const double *xdiv = nullptr,
                             double *tmp = nullptr, double *yn2 = nullptr);

static void schur_free(fvp_csr *A) {
    fvp_schur *P = A->sc;
    if (!P) return;
    if (P->B) fvp_csr_destroy(P->B);
    P->irow.release(); P->grow.release(); P->bsrc.release(); P->e_ia.release(); P->e_ja.release();
    P->e_loc.release(); P->e_src.release(); P->f_ia.release(); P->f_ja.release(); P->f_src.release();
    P->ev.release(); P->fv.release(); P->c_src.release(); P->c_pos.release(); P->goff.release();
    P->gsub.release(); P->glocal.release(); P->soff.release(); P->S.release(); P->t1.release();
    P->t2.release(); P->yG.release();
    delete P;
    A->sc = nullptr;
}

// Split of mtx_CRS_dist_split (schur.c:82-600) for subdomains of bs consecutive
// rows: a row is a boundary row when it has an entry in another subdomain or
// another subdomain has an entry in its column.  Interior unknowns keep their
// row order inside each subdomain, and so do the boundary unknowns.
static int build_schur(fvp_csr *A) {
    const int n = A->n, bs = A->bs, nsub = (n + bs - 1) / bs;
    std::vector<char> bnd(n, 0);
    for (int i = 0; i < n; ++i)
        for (int k = A->ia_h[i]; k < A->ia_h[i + 1]; ++k) {
            const int j = A->ja_h[k];
            if (i / bs != j / bs) bnd[i] = bnd[j] = 1;
        }
    std::vector<int> irow, grow, idx(n), goff(nsub + 1, 0), bstart(1, 0), gsub, glocal;
    for (int b = 0; b < nsub; ++b) {
        const int lo = b * bs, hi = std::min(n, lo + bs);
        for (int i = lo; i < hi; ++i)
            if (!bnd[i]) { idx[i] = (int)irow.size(); irow.push_back(i); }
        if ((int)irow.size() > bstart.back()) bstart.push_back((int)irow.size());  // empty interiors are skipped
        for (int i = lo; i < hi; ++i)
            if (bnd[i]) {
                idx[i] = (int)grow.size();
                glocal.push_back((int)grow.size() - goff[b]);
                grow.push_back(i);
                gsub.push_back(b);
            }
        goff[b + 1] = (int)grow.size();
        if (goff[b + 1] - goff[b] > kSchurMax) {
            set_error("Schur preconditioner: subdomain " + std::to_string(b) + " has " +
                      std::to_string(goff[b + 1] - goff[b]) + " boundary rows, at most " +
                      std::to_string(kSchurMax) + " are supported (use smaller subdomains)");
            return -1;
        }
    }
    const int nI = (int)irow.size(), nG = (int)grow.size();
    std::vector<int> bia(1, 0), bja, bsrc, eia(1, 0), eja, eloc, esrc, fia(1, 0), fja, fsrc, csrc;
    std::vector<long> cpos, soff(nsub + 1, 0);
    for (int b = 0; b < nsub; ++b) {
        const long m = goff[b + 1] - goff[b];
        soff[b + 1] = soff[b] + m * m;
    }
    for (int i : irow) {
        for (int k = A->ia_h[i]; k < A->ia_h[i + 1]; ++k) {
            const int j = A->ja_h[k];
            if (bnd[j]) { eja.push_back(idx[j]); eloc.push_back(idx[j] - goff[j / bs]); esrc.push_back(k); }
            else { bja.push_back(idx[j]); bsrc.push_back(k); }
        }
        bia.push_back((int)bja.size());
        eia.push_back((int)eja.size());
    }
    for (int i : grow) {
        const int b = i / bs;
        for (int k = A->ia_h[i]; k < A->ia_h[i + 1]; ++k) {
            const int j = A->ja_h[k];
            if (!bnd[j]) { fja.push_back(idx[j]); fsrc.push_back(k); }
            else if (j / bs == b) {  // C_ii; couplings to other subdomains' boundary rows are dropped
                const long m = goff[b + 1] - goff[b];
                cpos.push_back(soff[b] + (long)(idx[j] - goff[b]) * m + (idx[i] - goff[b]));
                csrc.push_back(k);
            }
        }
        fia.push_back((int)fja.size());
    }
    schur_free(A);
    fvp_schur *P = new fvp_schur();
    A->sc = P;
    P->nI = nI; P->nG = nG; P->nsub = nsub;
    P->maxg = 0;
    for (int b = 0; b < nsub; ++b) P->maxg = std::max(P->maxg, goff[b + 1] - goff[b]);
    if (nI > 0) {
        if (csr_create_impl(A->device, nI, bia.data(), bja.data(), &P->B)) { schur_free(A); return -1; }
        P->B->bstart = bstart;
        if (P->irow.upload(irow.data(), nI) || P->bsrc.upload(bsrc.data(), bsrc.size()) ||
            P->e_ia.upload(eia.data(), nI + 1) || P->t1.alloc(nI) || P->t2.alloc(nI) ||
            (!eja.empty() && (P->e_ja.upload(eja.data(), eja.size()) || P->e_loc.upload(eloc.data(), eloc.size()) ||
                              P->e_src.upload(esrc.data(), esrc.size()) || P->ev.alloc(eja.size())))) {
            schur_free(A);
            return -1;
        }
    }
    if (nG > 0) {
        if (P->grow.upload(grow.data(), nG) || P->f_ia.upload(fia.data(), nG + 1) || P->yG.alloc(nG) ||
            P->gsub.upload(gsub.data(), nG) || P->glocal.upload(glocal.data(), nG) ||
            P->goff.upload(goff.data(), nsub + 1) || P->soff.upload(soff.data(), nsub + 1) ||
            P->S.alloc(soff[nsub]) || P->c_src.upload(csrc.data(), csrc.size()) ||
            P->c_pos.upload(cpos.data(), cpos.size()) ||
            (!fja.empty() && (P->f_ja.upload(fja.data(), fja.size()) || P->f_src.upload(fsrc.data(), fsrc.size()) ||
                              P->fv.alloc(fja.size())))) {
            schur_free(A);
            return -1;
        }
    }
    return 0;
}

// precon_schur (schur.c:1247-1323) with schur_form_local (schur.c:887-981):
// ILU(0) of the interior blocks, then S_i = C_ii - F_i M_B^-1 E_i one column
// index at a time for every subdomain at once, then each S_i inverted.
static int schur_factor(fvp_csr *A) {
    hipStream_t s = A->stream;
    if (!A->lds_max && hipDeviceGetAttribute(&A->lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, A->device))
        A->lds_max = 64 * 1024;
    if (!A->sc && build_schur(A)) return -1;
    fvp_schur *P = A->sc;
    const size_t lds = (size_t)P->maxg * (P->maxg + 2) * sizeof(double) + (size_t)(P->maxg + 2) * sizeof(int);
    if (lds > (size_t)A->lds_max) { set_error("Schur preconditioner: a dense block does not fit the LDS"); return -1; }
    if (lds > 65536 && hipFuncSetAttribute((const void *)schur_invert, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds) != hipSuccess) {
        (void)hipGetLastError();
        set_error("Schur preconditioner: the block inversion cannot have " + std::to_string(lds) + " bytes of LDS");
        return -1;
    }
    if (P->B) {
        fvp_csr *B = P->B;
        fvp_csr_set_stream(B, s);
        vgather<<<nblk(B->nnz, 256), 256, 0, s>>>(B->nnz, P->bsrc.p, A->a.p, B->a.p);
        int rc = precon_build_impl(B, FVP_PRECON_BJILU0);
        if (rc) return rc;
        if (P->ev.n) vgather<<<nblk(P->ev.n, 256), 256, 0, s>>>(P->ev.n, P->e_src.p, A->a.p, P->ev.p);
    }
    if (P->nG == 0) return 0;
    if (P->fv.n) vgather<<<nblk(P->fv.n, 256), 256, 0, s>>>(P->fv.n, P->f_src.p, A->a.p, P->fv.p);
    for (int c = 0; c < P->maxg; ++c) {
        if (P->B) {
            schur_col_rhs<<<nblk(P->nI, 256), 256, 0, s>>>(P->nI, P->e_ia.p, P->e_loc.p, P->ev.p, c, P->t1.p);
            int rc = precon_apply_impl(P->B, P->t1.p, P->t2.p);
            if (rc) return rc;
        }
        schur_col_store<<<nblk(P->nG, 256), 256, 0, s>>>(P->nG, P->f_ia.p, P->f_ja.p, P->fv.p, P->t2.p, P->gsub.p,
                                                        P->glocal.p, P->goff.p, P->soff.p, c, P->S.p);
    }
    if (P->c_src.n)
        schur_add_c<<<nblk(P->c_src.n, 256), 256, 0, s>>>(P->c_src.n, P->c_pos.p, P->c_src.p, A->a.p, P->S.p);
    schur_invert<<<P->nsub, 256, lds, s>>>(P->goff.p, P->soff.p, P->S.p, A->flag.p);
    FVP_HIP(hipGetLastError());
    return 0;
}

// precon_schur_apply (schur.c:1583-1626): u = M_B^-1 x_I; y_G = S^-1 (x_G - F u);
// y_I = M_B^-1 (x_I - E y_G)
static int schur_apply(fvp_csr *A, const double *x, double *y) {
    hipStream_t s = A->stream;
    fvp_schur *P = A->sc;
    if (P->B) {
        fvp_csr_set_stream(P->B, s);
        vgather<<<nblk(P->nI, 256), 256, 0, s>>>(P->nI, P->irow.p, x, P->t1.p);
        int rc = precon_apply_impl(P->B, P->t1.p, P->t2.p);
        if (rc) return rc;
    }
    if (P->nG)
        schur_mid<<<P->nsub, kSchurMax, 0, s>>>(P->goff.p, P->soff.p, P->S.p, P->grow.p, P->f_ia.p, P->f_ja.p,
                                                 P->fv.p, x, P->t2.p, y, P->yG.p);
    if (P->B) {
        schur_back<<<nblk(P->nI, 256), 256, 0, s>>>(P->nI, P->irow.p, P->e_ia.p, P->e_ja.p, P->ev.p, x, P->yG.p,
                                                   P->t1.p);
        int rc = precon_apply_impl(P->B, P->t1.p, P->t2.p);
        if (rc) return rc;
        vscatter<<<nblk(P->nI, 256), 256, 0, s>>>(P->nI, P->irow.p, P->t2.p, y);
    }
    return 0;
}

// bj_factor's launch: the blocks' description, and the staged values' LDS bytes (0: in place)
struct FactorArgs {
    int nblk;
    const int *roff, *ia, *src;
    const double *a;
    const FactorTab *tab;
    const int *lev, *lptr;
    int *flag;
    FacOut out;
    const uint4 *sout;
    size_t staged;
    int npmax;  // most pieces of one block (staged form)
    int threads;
};
template <typename T, int NC, int TH>
static void bj_factor_launch_th(hipStream_t s, const FactorArgs &f, T *lu, T *vl, T *vu, T *vd) {
    const FactorTab &t = *f.tab;
    const auto kernel = f.staged ? bj_factor<T, NC, true, TH> : bj_factor<T, NC, false, TH>;
    kernel<<<f.nblk, TH, f.staged, s>>>(f.roff, f.ia, f.src, f.a, t.slot.p, f.sout, t.piv.p, t.off.p, f.lev, f.lptr, lu,
                                        vl, vu, vd, f.out, f.flag, f.npmax);
}
template <typename T, int NC>
static void bj_factor_launch_nc(hipStream_t s, const FactorArgs &f, T *lu, T *vl, T *vu, T *vd) {
    if (f.threads == 64) bj_factor_launch_th<T, NC, 64>(s, f, lu, vl, vu, vd);
    else if (f.threads == 128) bj_factor_launch_th<T, NC, 128>(s, f, lu, vl, vu, vd);
    else if (f.threads == 256) bj_factor_launch_th<T, NC, 256>(s, f, lu, vl, vu, vd);
    else if (f.threads == 512 || NC > 1) bj_factor_launch_th<T, NC, 512>(s, f, lu, vl, vu, vd);
    else bj_factor_launch_th<T, NC, NC == 1 ? 1024 : 512>(s, f, lu, vl, vu, vd);
}
template <typename T>
static void bj_factor_launch(hipStream_t s, const FactorArgs &f, T *lu, T *vl, T *vu, T *vd) {
    if (f.tab->nc == 1) bj_factor_launch_nc<T, 1>(s, f, lu, vl, vu, vd);
    else if (f.tab->nc == 2) bj_factor_launch_nc<T, 2>(s, f, lu, vl, vu, vd);
    else bj_factor_launch_nc<T, 4>(s, f, lu, vl, vu, vd);
}

template <typename T, int NC>
static void bj_factor_attrs(int lds_max) {
    for (const void *f : {(const void *)bj_factor<T, NC, true, 64>, (const void *)bj_factor<T, NC, true, 128>,
                          (const void *)bj_factor<T, NC, true, 256>, (const void *)bj_factor<T, NC, true, 512>,
                          (const void *)bj_factor<T, NC, true, NC == 1 ? 1024 : 512>})
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
}
static void bj_attrs(int lds_max) {
    bj_factor_attrs<double, 1>(lds_max); bj_factor_attrs<double, 2>(lds_max); bj_factor_attrs<double, 4>(lds_max);
    bj_factor_attrs<float, 1>(lds_max); bj_factor_attrs<float, 2>(lds_max); bj_factor_attrs<float, 4>(lds_max);
    for (const void *f : {(const void *)bj_solve<double, 4, false>, (const void *)bj_solve<float, 4, false>,
                          (const void *)bj_solve<float, 6, true>})
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max);
}

static int precon_build_impl(fvp_csr *A, int type) {
    hipStream_t s = A->stream;
    const int n = A->n;
    if (type == FVP_PRECON_NONE) { A->ptype = type; return 0; }
    if (type != FVP_PRECON_JACOBI && type != FVP_PRECON_ILU0 && type != FVP_PRECON_BJILU0 &&
        type != FVP_PRECON_BJILU0_F32 && type != FVP_PRECON_SCHUR) {
        set_error("invalid preconditioner type");
        return -1;
    }
    if (!A->flag.p) {  // cleared here and by every flag_post
        if (A->flag.alloc(1)) return -1;
        FVP_HIP(hipMemsetAsync(A->flag.p, 0, sizeof(int), s));
    }
    if (!A->hflag.p && A->hflag.alloc(1)) return -1;
    if (type == FVP_PRECON_SCHUR) {
        int rc = schur_factor(A);
        if (rc) { A->ptype = -1; return rc; }
    } else if (type == FVP_PRECON_BJILU0 || type == FVP_PRECON_BJILU0_F32) {
        const bool f32 = type == FVP_PRECON_BJILU0_F32;
        int rc = A->bj ? 0 : build_bj(A);
        if (!rc) rc = bj_layout(A, f32);
        if (rc) { A->ptype = -1; return rc; }
        const FacPieces &F = A->fp[f32];
        const BjPack &P = A->pack_of(f32);
        // FVP_BJ_FACTOR_MODE 0 / 1 forces values in place / staged where they fit the
        // workgroup: a tuning and test knob
        bool stage = F.staged;
        if (const char *e = getenv("FVP_BJ_FACTOR_MODE")) stage = atoi(e) > 0 && F.lds <= (size_t)A->lds_max;
        A->factor_mode = stage;
        const FactorArgs fa{A->nblk, A->b_roff.p, A->b_ia.p, A->b_src.p, A->a.p, &A->fac, F.lev.p, F.lptr.p, A->flag.p,
                            FacOut{(unsigned)P.win, P.place.p, P.lev_l.p, P.lptr_l.p, P.lev_u.p, P.lptr_u.p},
                            P.out.p, stage ? F.lds : 0, F.most, F.threads};
        const size_t nl = P.row_l.n * P.win, nu = P.row_u.n * P.win, nd = P.row_u.n;
        // the packed arrays' padding stays zero: only the factor's entries are written
        auto ensure = [&](auto &lu, auto &vl, auto &vu, auto &vd) {
            if (!lu.p && lu.alloc(A->b_src.n)) return -1;
            if (vd.p) return 0;  // the last of them
            // ... and a slot without a diagonal keeps d = 1
            const std::vector<std::decay_t<decltype(*vd.p)>> ones(nd, 1);
            if (vl.alloc(nl) || vu.alloc(nu)) return -1;
            FVP_HIP(hipMemsetAsync(vl.p, 0, sizeof(*vl.p) * nl, s));
            FVP_HIP(hipMemsetAsync(vu.p, 0, sizeof(*vu.p) * nu, s));
            return vd.upload(ones.data(), nd);
        };
        if (!f32) {
            if (ensure(A->b_lu, A->val_l, A->val_u, A->dinv)) return -1;
            bj_factor_launch<double>(s, fa, A->b_lu.p, A->val_l.p, A->val_u.p, A->dinv.p);
        } else {
            if (ensure(A->b_lu32, A->val32_l, A->val32_u, A->dinv32)) return -1;
            bj_factor_launch<float>(s, fa, A->b_lu32.p, A->val32_l.p, A->val32_u.p, A->dinv32.p);
        }
    } else if (type == FVP_PRECON_JACOBI) {
        if (A->jac.n != (size_t)n && A->jac.alloc(n)) return -1;
        jacobi_build<<<nblk(n, 256), 256, 0, s>>>(n, A->ia.p, A->ja.p, A->a.p, A->jac.p, A->flag.p);
    } else {
        if (!A->diag.p) {
            std::vector<int> diag(n);
            for (int i = 0; i < n; ++i) {
                int k = A->ia_h[i];
                while (k < A->ia_h[i + 1] && A->ja_h[k] != i) ++k;
                if (k == A->ia_h[i + 1]) { set_error("zero diagonal on row " + std::to_string(i)); A->ptype = -1; return FVP_ERR_PIVOT; }
                diag[i] = k;
            }
            if (A->diag.upload(diag.data(), n)) return -1;
            if (build_levels(A, diag)) return -1;
        }
        if (A->lu.n != (size_t)A->nnz && A->lu.alloc(A->nnz)) return -1;
        FVP_HIP(hipMemcpyAsync(A->lu.p, A->a.p, sizeof(double) * A->nnz, hipMemcpyDeviceToDevice, s));
        if (A->one) {
            const int *fp = A->o_fptr.p;
            double *vl = A->otri[0].val.p, *vu = A->otri[1].val.p;
            bj_factor_launch<double>(s, FactorArgs{1, fp, A->ia.p, nullptr, nullptr, &A->ofac, fp + 2, fp + 4,
                                                   A->flag.p, FacOut{(unsigned)A->o_win, nullptr, nullptr, nullptr, nullptr, nullptr},
                                                   A->ofac.out.p, 0, 0, A->o_fthreads},
                                     A->lu.p, vl, vu, vu + (size_t)n * A->o_win);
        }
        for (size_t l = 0; !A->one && l + 1 < A->lptr_h.size(); ++l) {
            int cnt = A->lptr_h[l + 1] - A->lptr_h[l];
            ilu0_factor_level<<<nblk(cnt, 64), 64, 0, s>>>(cnt, A->lrows.p + A->lptr_h[l], A->ia.p, A->ja.p,
                                                           A->diag.p, A->lu.p, A->flag.p);
        }
    }
    const double tag = ++A->hflag.tag;
    flag_post<<<1, 64, 0, s>>>(A->flag.p, A->hflag.p, tag);
    FVP_HIP(hipGetLastError());
    if (slot_wait(s, A->hflag.p, tag)) return -1;
    if (A->hflag.p[0] != 0.) { set_error("zero pivot in preconditioner factorisation"); A->ptype = -1; return FVP_ERR_PIVOT; }
    A->ptype = type;
    return 0;
}

template <int KW, int TH>
static void ilu0_one_launch_th(fvp_csr *A, const double *x, const double *xdiv, double *y, double *yn2) {
    const IluTri &L = A->otri[0], &U = A->otri[1];
    ilu0_solve<KW, TH><<<1, TH, A->o_lds, A->stream>>>(A->n, L.npieces, L.pptr.p, L.row.p, L.col.p, L.val.p,
                                                       U.npieces, U.pptr.p, U.row.p, U.col.p, U.val.p, x, xdiv, y,
                                                       yn2, A->skip);
}
template <int KW>
static void ilu0_one_launch(fvp_csr *A, const double *x, const double *xdiv, double *y, double *yn2) {
    if (A->o_threads == 64) ilu0_one_launch_th<KW, 64>(A, x, xdiv, y, yn2);
    else if (A->o_threads == 256) ilu0_one_launch_th<KW, 256>(A, x, xdiv, y, yn2);
    else ilu0_one_launch_th<KW, 1024>(A, x, xdiv, y, yn2);
}

// y = M^-1 (x / xdiv) with xdiv optional (the block solves and the one-workgroup
// ILU(0) divide as they load); yn2 (optional, at least nblk doubles): their
// partials of ||y||^2
static int precon_apply_impl(fvp_csr *A, const double *x, double *y, const double *xdiv, double *tmp,
                             double *yn2) {
    hipStream_t s = A->stream;
    const int n = A->n;
    const bool one = A->ptype == FVP_PRECON_ILU0 && A->one;
    if (xdiv && A->ptype != FVP_PRECON_BJILU0 && A->ptype != FVP_PRECON_BJILU0_F32 && !one) {
        if (!tmp) { set_error("internal: scaled preconditioner solve needs a work vector"); return -1; }
        vdiv<<<nblk(n, 256), 256, 0, s>>>(n, x, xdiv, tmp);
        x = tmp;
        xdiv = nullptr;
    }
    switch (A->ptype) {
    case FVP_PRECON_NONE:
        vcopy<<<nblk(n, 256), 256, 0, s>>>(n, x, y);
        break;
    case FVP_PRECON_JACOBI:
        vmul<<<nblk(n, 256), 256, 0, s>>>(n, x, A->jac.p, y);
        break;
    case FVP_PRECON_BJILU0:
    case FVP_PRECON_BJILU0_F32: {
        const bool f64 = A->ptype == FVP_PRECON_BJILU0;
        const BjPack &P = A->pack_of(!f64);
        const size_t lds = bj_solve_lds(f64 ? sizeof(double) : sizeof(float), A->b_maxrows, P.levmax_l, P.levmax_u);
        if (lds > (size_t)A->lds_max) {
            set_error("block-Jacobi ILU(0): a block's solution does not fit the LDS");
            return -1;
        }
#define FVP_BJ_SOLVE(T, W, PAIR, VL, VU, DI)                                                                       \
    bj_solve<T, W, PAIR><<<A->nblk, 64, lds, s>>>(A->b_roff.p, A->b_rowid.p, A->b_own.p, P.lev_l.p, P.lptr_l.p, VL,      \
                                            P.col_l.p, P.row_l.p, P.lev_u.p, P.lptr_u.p, VU, P.col_u.p, P.row_u.p, \
                                            DI, A->b_maxrows, x, xdiv, y, yn2, A->skip)
        if (f64) FVP_BJ_SOLVE(double, 4, false, A->val_l.p, A->val_u.p, A->dinv.p);
        else if (P.win == 6) FVP_BJ_SOLVE(float, 6, true, A->val32_l.p, A->val32_u.p, A->dinv32.p);
        else FVP_BJ_SOLVE(float, 4, false, A->val32_l.p, A->val32_u.p, A->dinv32.p);
#undef FVP_BJ_SOLVE
        break;
    }
    case FVP_PRECON_SCHUR: {
        int rc = schur_apply(A, x, y);
        if (rc) return rc;
        break;
    }
    case FVP_PRECON_ILU0: {
        if (one) {
            if (A->o_win == 4) ilu0_one_launch<4>(A, x, xdiv, y, yn2);
            else if (A->o_win == 8) ilu0_one_launch<8>(A, x, xdiv, y, yn2);
            else if (A->o_win == 16) ilu0_one_launch<16>(A, x, xdiv, y, yn2);
            else ilu0_one_launch<32>(A, x, xdiv, y, yn2);
            break;
        }
        const int L = 8;
        for (size_t l = 0; l + 1 < A->lptr_h.size(); ++l) {
            int cnt = A->lptr_h[l + 1] - A->lptr_h[l];
            ilu0_lower_level<L><<<nblk((long)cnt * L, 256), 256, 0, s>>>(cnt, A->lrows.p + A->lptr_h[l], A->ia.p,
                                                                        A->ja.p, A->diag.p, A->lu.p, x, y);
        }
        for (size_t l = 0; l + 1 < A->uptr_h.size(); ++l) {
            int cnt = A->uptr_h[l + 1] - A->uptr_h[l];
            ilu0_upper_level<L><<<nblk((long)cnt * L, 256), 256, 0, s>>>(cnt, A->urows.p + A->uptr_h[l], A->ia.p,
                                                                        A->ja.p, A->diag.p, A->lu.p, y);
        }
        break;
    }
    default:
        set_error("preconditioner not built");
        return -1;
    }
    FVP_HIP(hipGetLastError());
    return 0;
}

int csr_create_impl(int device, int n, const int *ia, const int *ja, fvp_csr **out) {
    if (!out || !ia || !ja || n <= 0) { set_error("invalid CSR arguments"); return -1; }
    *out = nullptr;
    int longest = 0;
    for (int i = 0; i < n; ++i) {
        if (ia[i + 1] < ia[i]) { set_error("row pointers must be non-decreasing"); return -1; }
        longest = std::max(longest, ia[i + 1] - ia[i]);
        for (int k = ia[i]; k < ia[i + 1]; ++k) {
            if (ja[k] < 0 || ja[k] >= n) { set_error("column index out of range"); return -1; }
            if (k > ia[i] && ja[k] <= ja[k - 1]) { set_error("column indices must be sorted and unique"); return -1; }
        }
    }
    FVP_HIP(hipSetDevice(device));
    fvp_csr *A = new fvp_csr();
    A->device = device;
    A->n = n;
    A->nnz = ia[n];
    A->longest = longest;
    A->ia_h.assign(ia, ia + n + 1);
    A->ja_h.assign(ja, ja + A->nnz);
    if (hipStreamCreateWithFlags(&A->own_stream, hipStreamNonBlocking) != hipSuccess) {
        delete A; set_error("hipStreamCreate failed"); return -1;
    }
    A->stream = A->own_stream;
    if (A->ia.upload(ia, n + 1) || A->ja.upload(ja, A->nnz) || A->a.alloc(A->nnz)) { fvp_csr_destroy(A); return -1; }
    *out = A;
    return 0;
}

}  // namespace fvp

extern "C" int fvp_csr_create(int device, int n, const int *ia, const int *ja, fvp_csr **out) {
    return csr_create_impl(device, n, ia, ja, out);
}

extern "C" int fvp_csr_destroy(fvp_csr *A) {
    if (!A) return 0;
    (void)hipSetDevice(A->device);
    if (A->own_stream) (void)hipStreamSynchronize(A->own_stream);
    A->ia.release(); A->ja.release(); A->a.release(); A->lu.release(); A->jac.release(); A->diag.release();
    A->lrows.release(); A->urows.release(); A->flag.release(); A->Q.release(); A->w.release(); A->r.release();
    A->z.release(); A->part.release(); A->scal.release(); A->hdev.release();
    A->Hd.release(); A->gd.release(); A->csd.release(); A->snd.release(); A->Qk.release();
    A->hstat.release();
    A->hflag.release();
    A->b_ia.release(); A->b_src.release(); A->b_lu.release(); A->b_lu32.release();
    A->b_roff.release(); A->b_rowid.release(); A->b_own.release(); A->b_zn2.release();
    A->pack[0].release(); A->pack[1].release(); A->val_l.release();
    A->val_u.release(); A->dinv.release(); A->val32_l.release(); A->val32_u.release(); A->dinv32.release();
    A->fac.release(); A->ofac.release(); A->otri[0].release(); A->otri[1].release(); A->o_fptr.release();
    A->fp[0].release(); A->fp[1].release();
    schur_free(A);
    if (A->own_stream) (void)hipStreamDestroy(A->own_stream);
    delete A;
    return 0;
}

extern "C" int fvp_csr_set_stream(fvp_csr *A, void *stream) {
    if (!A) { set_error("null matrix"); return -1; }
    A->stream = stream ? (hipStream_t)stream : A->own_stream;
    return 0;
}

extern "C" int fvp_csr_set_values(fvp_csr *A, const double *values) {
    if (!A || !values) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    FVP_HIP(hipMemcpyAsync(A->a.p, values, sizeof(double) * A->nnz, hipMemcpyDeviceToDevice, A->stream));
    A->ptype = -1;
    return 0;
}

extern "C" int fvp_csr_get_values(fvp_csr *A, double *values_host) {
    if (!A || !values_host) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    FVP_HIP(hipStreamSynchronize(A->stream));
    FVP_HIP(hipMemcpy(values_host, A->a.p, sizeof(double) * A->nnz, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int fvp_csr_gemv(fvp_csr *A, double alpha, const double *x, double beta, double *y) {
    if (!A || !x || !y) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    return csr_gemv_impl(A, alpha, x, beta, y);
}

static int set_block_rows(fvp_csr *A, int rows) {
    if (rows < 64 || rows > 4096 || (rows & (rows - 1))) {
        set_error("block rows must be a power of two in [64, 4096]");
        return -1;
    }
    if (rows != A->bs) {
        A->bs = rows;
        A->bj = false;  // block tables are rebuilt by the next block-Jacobi build
        schur_free(A);  // and the subdomains by the next Schur build
        if (A->ptype == FVP_PRECON_BJILU0 || A->ptype == FVP_PRECON_BJILU0_F32 || A->ptype == FVP_PRECON_SCHUR)
            A->ptype = -1;
    }
    return 0;
}

extern "C" int fvp_precon_block_rows(fvp_csr *A, int rows) {
    if (!A) { set_error("null matrix"); return -1; }
    return set_block_rows(A, rows);
}

static int set_overlap(fvp_csr *A, int layers) {
    if (layers < 0 || layers > 2) { set_error("overlap must be 0, 1 or 2 layers"); return -1; }
    if (layers != A->overlap) {
        A->overlap = layers;
        A->bj = false;
        if (A->ptype == FVP_PRECON_BJILU0 || A->ptype == FVP_PRECON_BJILU0_F32) A->ptype = -1;
    }
    return 0;
}

extern "C" int fvp_precon_overlap(fvp_csr *A, int layers) {
    if (!A) { set_error("null matrix"); return -1; }
    return set_overlap(A, layers);
}

extern "C" int fvp_precon_build(fvp_csr *A, int type) {
    if (!A) { set_error("null matrix"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    return precon_build_impl(A, type);
}

extern "C" int fvp_precon_apply(fvp_csr *A, const double *x, double *y) {
    if (!A || !x || !y) { set_error("null argument"); return -1; }
    if (x == y && A->ptype == FVP_PRECON_ILU0) { set_error("ILU(0) apply cannot run in place"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    return precon_apply_impl(A, x, y);
}

extern "C" int fvp_precon_values(fvp_csr *A, double *values_host) {
    if (!A || !values_host) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    FVP_HIP(hipStreamSynchronize(A->stream));
    if (A->ptype == FVP_PRECON_ILU0)
        FVP_HIP(hipMemcpy(values_host, A->lu.p, sizeof(double) * A->nnz, hipMemcpyDeviceToHost));
    else if (A->ptype == FVP_PRECON_JACOBI)
        FVP_HIP(hipMemcpy(values_host, A->jac.p, sizeof(double) * A->n, hipMemcpyDeviceToHost));
    else if ((A->ptype == FVP_PRECON_BJILU0 || A->ptype == FVP_PRECON_BJILU0_F32) && A->overlap > 0) {
        set_error("overlapping blocks share entries: their factors have no single-pattern form");
        return -1;
    } else if (A->ptype == FVP_PRECON_BJILU0 || A->ptype == FVP_PRECON_BJILU0_F32) {
        // scattered back to the full pattern, 0 off the blocks
        std::vector<double> lu(A->b_src.n);
        std::vector<int> src(A->b_src.n);
        if (A->ptype == FVP_PRECON_BJILU0)
            FVP_HIP(hipMemcpy(lu.data(), A->b_lu.p, sizeof(double) * lu.size(), hipMemcpyDeviceToHost));
        else {
            std::vector<float> lu32(lu.size());
            FVP_HIP(hipMemcpy(lu32.data(), A->b_lu32.p, sizeof(float) * lu.size(), hipMemcpyDeviceToHost));
            for (size_t k = 0; k < lu.size(); ++k) lu[k] = lu32[k];
        }
        FVP_HIP(hipMemcpy(src.data(), A->b_src.p, sizeof(int) * src.size(), hipMemcpyDeviceToHost));
        std::fill(values_host, values_host + A->nnz, 0.);
        for (size_t k = 0; k < lu.size(); ++k) values_host[src[k]] = lu[k];
    }
    else { set_error("no factored values"); return -1; }
    return 0;
}

// the preconditioner's diagonal, where it is one
static const double *diagonal_of(const fvp_csr *A) { return A->ptype == FVP_PRECON_JACOBI ? A->jac.p : nullptr; }

extern "C" int fvp_gmres_csr(fvp_csr *A, const double *b, double *x, const fvp_gmres_params *p,
                             fvp_gmres_stats *st) {
    if (!A || !b || !x || !p) { set_error("null argument"); return -1; }
    if (A->ptype < 0) { set_error("preconditioner not built"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    Op op = [A](const double *in, double *out) { return csr_gemv_impl(A, 1.0, in, 0.0, out); };
    Op pc;
    if (A->ptype != FVP_PRECON_NONE) pc = [A](const double *in, double *out) { return precon_apply_impl(A, in, out); };
    return gmres_device(A, A->stream, A->n, op, pc, b, x, p, st, nullptr, diagonal_of(A));
}

extern "C" int fvp_gmres_csr_deflated(fvp_csr *A, const double *b, double *x, const fvp_gmres_params *p, int k,
                                      fvp_gmres_stats *st) {
    if (!A || !b || !x || !p) { set_error("null argument"); return -1; }
    if (A->ptype < 0) { set_error("preconditioner not built"); return -1; }
    FVP_HIP(hipSetDevice(A->device));
    Op op = [A](const double *in, double *out) { return csr_gemv_impl(A, 1.0, in, 0.0, out); };
    Op pc;
    if (A->ptype != FVP_PRECON_NONE) pc = [A](const double *in, double *out) { return precon_apply_impl(A, in, out); };
    return gmres_deflated(A, A->stream, A->n, op, pc, b, x, p, k, st);
}

// ---- allocation-free GMRES ------------------------------------------------------
// Workspace of fvp_gmres_csr_noalloc: a static device array (32 MiB, one per
// GPU, held until the process ends).  In host code the array's name is only a
// stand-in; its device address on each GPU comes from hipGetSymbolAddress,
// taken once per device with that device current.
constexpr size_t kScratchDoubles = size_t(4) << 20;
static __device__ __align__(256) double scratch[kScratchDoubles];
constexpr int kScratchDevices = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[kScratchDevices];

__global__ void zero_fill(long n, double *__restrict__ p) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0.;
}

// the scratch array's address on `device` (which must be current)
static double *scratch_address(int device) {
    if (device < 0 || device >= kScratchDevices) { set_error("device index out of range"); return nullptr; }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[device] = static_cast<double *>(ptr);
    }
    return g_scratch_ptr[device];
}

extern "C" int fvp_gmres_csr_noalloc(fvp_csr *A, const double *b, double *x, const fvp_gmres_params *p,
                                     fvp_gmres_stats *st) {
    if (!A || !b || !x || !p) { set_error("null argument"); return -1; }
    if (A->ptype < 0) { set_error("preconditioner not built"); return -1; }
    const int m = p->dim_krylov;
    if (m < 1 || m > 63) { set_error("dim_krylov must be 1..63"); return -1; }
    if (p->reorthogonalise < 0 || p->reorthogonalise > 2) { set_error("reorthogonalise must be 0, 1 or 2"); return -1; }
    const size_t need = gmres_work_doubles(A->n, m);
    if (need > kScratchDoubles) {
        set_error("fvp_gmres_csr_noalloc: the workspace of n = " + std::to_string(A->n) + ", dim_krylov = " +
                  std::to_string(m) + " needs " + std::to_string(need) + " doubles, more than the " +
                  std::to_string(kScratchDoubles) + " of the static workspace (use fvp_gmres_csr)");
        return -1;
    }
    FVP_HIP(hipSetDevice(A->device));
    double *base = scratch_address(A->device);
    if (!base) return -1;
    GmresWork wk = gmres_work_carve(base, A->n, m);
    // the scalars, coefficients and Hessenberg data start cleared on every call
    // (the array keeps the previous call's contents); the basis, work vectors
    // and partials are written before they are read
    const long small = (long)(need - (size_t)(wk.sc - base));
    zero_fill<<<(int)std::min(1024L, (small + 255) / 256), 256, 0, A->stream>>>(small, wk.sc);
    FVP_HIP(hipGetLastError());
    double hstat[kSlot * 64];
    wk.hstat = hstat;  // pageable: each step's pair is copied and read synchronously
    wk.diag = diagonal_of(A);
    Op op = [A](const double *in, double *out) { return csr_gemv_impl(A, 1.0, in, 0.0, out); };
    Op pc;
    if (A->ptype != FVP_PRECON_NONE) pc = [A](const double *in, double *out) { return precon_apply_impl(A, in, out); };
    return gmres_core(wk, A->stream, A->n, op, pc, b, x, p, st);
}

// ================================================================================
// Coloured FD Jacobian and the Newton linear solve on a problem context
// ================================================================================
struct fvp_jacdata {
    fvp_csr *J = nullptr;
    bool coloured = false;             // colouring built (colour_init)
    int ncol = 0;
    std::vector<int> colour;           // per node
    std::vector<int> cptr;             // colour -> [cptr[c], cptr[c+1]) in cols
    std::vector<int> eptr;             // colour -> entries
    DevBuf<int> cols, erow, epos, ecol;
    DevBuf<double> shift, ys, yps, Fs;
    // element-local quotients, see FdJacobian; per row its diagonal entry
    DevBuf<int> vptr, visit, code32, dpos;
    DevBuf<unsigned> cptr2;
    DevBuf<uint16_t> code;
    int rows = 0, max_visits = 0;
    DevBuf<double> contrib, rec, dterm;
};

namespace fvp {

__global__ void shift_kernel(int n, double eps, double h, const double *__restrict__ y, const double *__restrict__ yp,
                             const double *__restrict__ ewt, double *__restrict__ shift) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    shift[j] = eps * fmax(fabs(y[j]), fmax(fabs(h * yp[j]), 1.0 / ewt[j]));
}

__global__ void perturb_kernel(int cnt, const int *__restrict__ cols, const double *__restrict__ shift, double c,
                               const double *__restrict__ y, const double *__restrict__ yp, double *__restrict__ ys,
                               double *__restrict__ yps, int restore) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= cnt) return;
    int j = cols[k];
    if (restore) { ys[j] = y[j]; yps[j] = yp[j]; }
    else { ys[j] = y[j] + shift[j]; yps[j] = yp[j] + c * shift[j]; }
}

// J[pos] = (F0[row] - Fs[row]) / shift[col]   (-(dF/dy + c dF/dy') column entries)
__global__ void fd_scatter(int cnt, const int *__restrict__ erow, const int *__restrict__ epos,
                           const int *__restrict__ ecol, const double *__restrict__ F0,
                           const double *__restrict__ Fs, const double *__restrict__ shift, double *__restrict__ J) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= cnt) return;
    int r = erow[k];
    J[epos[k]] = (F0[r] - Fs[r]) / shift[ecol[k]];
}

// Tables of fd_gather: each entry's quotients in element order, as places in
// the visits of its workgroup of rows.  A workgroup takes 64 rows (a box: about
// 1500 visits, 24 KB in FP32), fewer where their visits need more than kFdLds in
// FP64; where even 8 do, the codes are places in contrib and nothing is staged.
constexpr size_t kFdLds = 64 * 1024;
static int fd_tables(fvp_ctx *c, fvp_jacdata *jd, const std::vector<int4> &conn, const std::vector<int> &ia,
                     const std::vector<int> &ja) {
    const int N = c->N, T = c->T, npe = c->npe;
    const long nnz = ia[N];
    if ((long)16 * T > INT32_MAX) { set_error("too many elements for the FD Jacobian slots"); return -1; }
    auto at = [&](int row, int col) {
        return (int)(std::lower_bound(ja.begin() + ia[row], ja.begin() + ia[row + 1], col) - ja.begin());
    };
    // visits by row, element order within; each entry's number of quotients
    std::vector<int> rv(N + 1, 0), visit((size_t)npe * T), local((size_t)npe * T), pos((size_t)npe * npe * T), dpos(N);
    std::vector<unsigned> cp(nnz + 1, 0);
    for (int e = 0; e < T; ++e) {
        const int n[4] = {conn[e].x, conn[e].y, conn[e].z, conn[e].w};
        for (int i = 0; i < npe; ++i) {
            ++rv[n[i] + 1];
            for (int k = 0; k < npe; ++k) {
                const int p = at(n[i], n[k]);
                pos[((size_t)e * npe + i) * npe + k] = p;
                ++cp[p + 1];
            }
        }
    }
    for (int i = 0; i < N; ++i) { rv[i + 1] += rv[i]; dpos[i] = at(i, i); }
    for (long p = 0; p < nnz; ++p) cp[p + 1] += cp[p];
    {
        std::vector<int> fill(rv.begin(), rv.end() - 1);
        for (int e = 0; e < T; ++e) {
            const int n[4] = {conn[e].x, conn[e].y, conn[e].z, conn[e].w};
            for (int i = 0; i < npe; ++i) {
                const int v = fill[n[i]]++;
                visit[v] = e * npe + i;
                local[(size_t)e * npe + i] = v;
            }
        }
    }
    const int limit = (int)(kFdLds / (4 * sizeof(double)));
    auto most = [&](int rows) {
        int m = 0;
        for (int r = 0; r < N; r += rows) m = std::max(m, rv[std::min(N, r + rows)] - rv[r]);
        return m;
    };
    int rows = 64;
    while (rows > 8 && most(rows) > limit) rows /= 2;
    jd->max_visits = most(rows);
    const bool staged = jd->max_visits <= limit;
    if (!staged) rows = 64;
    jd->rows = rows;
    std::vector<uint16_t> code;
    std::vector<int> code32, vptr;
    (staged ? code.resize(cp[nnz]) : code32.resize(cp[nnz]));
    {
        std::vector<unsigned> fill(cp.begin(), cp.end() - 1);
        for (int e = 0; e < T; ++e) {
            const int n[4] = {conn[e].x, conn[e].y, conn[e].z, conn[e].w};
            for (int i = 0; i < npe; ++i)
                for (int k = 0; k < npe; ++k) {
                    const size_t v = (size_t)e * npe + i;
                    const unsigned to = fill[pos[v * npe + k]]++;
                    if (staged) code[to] = (uint16_t)(4 * (local[v] - rv[n[i] / rows * rows]) + k);
                    else code32[to] = (int)(4 * v + k);
                }
        }
    }
    for (int r = 0; r < N; r += rows) vptr.push_back(rv[r]);
    vptr.push_back(rv[N]);
    for (int i = 0; i < N; ++i) cp[dpos[i]] |= 1u << 31;
    if (staged ? jd->code.upload(code.data(), code.size()) || jd->visit.upload(visit.data(), visit.size()) ||
                     jd->vptr.upload(vptr.data(), vptr.size())
               : jd->code32.upload(code32.data(), code32.size()))
        return -1;
    return jd->cptr2.upload(cp.data(), cp.size()) || jd->dpos.upload(dpos.data(), N) ||
           jd->contrib.alloc((size_t)4 * npe * T) || jd->rec.alloc(2 * (size_t)c->nz * N) || jd->dterm.alloc(N);
}

// Node adjacency over element pairs (preconditioner_dss.cpp:107-142) and the
// greedy distance-2 colouring of preconditioner_dss.cpp:72-94.
static int jac_init(fvp_ctx *c) {
    if (c->jd) return 0;
    const int N = c->N, T = c->T, npe = c->npe;
    std::vector<int4> conn(T);
    FVP_HIP(hipMemcpy(conn.data(), c->conn.p, sizeof(int4) * T, hipMemcpyDeviceToHost));
    // node adjacency (the Jacobian pattern): every element's node pairs, counted
    // into per-row segments, then sorted and made unique row by row
    std::vector<int> off(N + 1, 0), buf;
    for (int e = 0; e < T; ++e) {
        const int n[4] = {conn[e].x, conn[e].y, conn[e].z, conn[e].w};
        for (int a = 0; a < npe; ++a) off[n[a] + 1] += npe;
    }
    for (int i = 0; i < N; ++i) off[i + 1] += off[i];
    buf.resize(off[N]);
    {
        std::vector<int> fill(off.begin(), off.end() - 1);
        for (int e = 0; e < T; ++e) {
            const int n[4] = {conn[e].x, conn[e].y, conn[e].z, conn[e].w};
            for (int a = 0; a < npe; ++a)
                for (int b = 0; b < npe; ++b) buf[fill[n[a]]++] = n[b];
        }
    }
    std::vector<int> ia(N + 1, 0), ja;
    ja.reserve(off[N] / 4);
    for (int i = 0; i < N; ++i) {
        auto b0 = buf.begin() + off[i], b1 = buf.begin() + off[i + 1];
        std::sort(b0, b1);
        ja.insert(ja.end(), b0, std::unique(b0, b1));
        ia[i + 1] = (int)ja.size();
    }
    std::vector<int>().swap(buf);
    fvp_jacdata *jd = new fvp_jacdata();
    if (csr_create_impl(c->device, N, ia.data(), ja.data(), &jd->J)) { delete jd; return -1; }
    fvp_csr_set_stream(jd->J, c->stream);
    {
        if (fd_tables(c, jd, conn, ia, ja)) {
            fvp_csr_destroy(jd->J);
            delete jd;
            return -1;
        }
    }
    if (jd->shift.alloc(N) || jd->ys.alloc(N) || jd->yps.alloc(N) || jd->Fs.alloc(N)) {
        fvp_csr_destroy(jd->J);
        delete jd;
        return -1;
    }
    c->jd = jd;
    return 0;
}

// The reference's greedy distance-2 colouring in node order and, per colour,
// the entries its columns fill (the coloured FD Jacobian and fvp_colours only;
// built on first use)
static int colour_init(fvp_ctx *c) {
    if (jac_init(c)) return -1;
    fvp_jacdata *jd = c->jd;
    if (jd->coloured) return 0;
    const int N = c->N;
    const std::vector<int> &ia = jd->J->ia_h, &ja = jd->J->ja_h;
    // greedy distance-2 colouring in node order
    std::vector<int> colour(N, N - 1), mark(N, -1);
    int maxc = 0;
    for (int i = 0; i < N; ++i) {
        for (int p = ia[i]; p < ia[i + 1]; ++p) {
            int nb = ja[p];
            for (int q = ia[nb]; q < ia[nb + 1]; ++q) mark[colour[ja[q]]] = i;
        }
        int sc = 0;
        while (sc < maxc && mark[sc] == i) ++sc;
        if (sc == maxc) ++maxc;
        colour[i] = sc;
    }
    jd->ncol = maxc;
    jd->colour = colour;
    std::vector<int> cols(N), cptr(maxc + 1, 0);
    for (int i = 0; i < N; ++i) cptr[colour[i] + 1]++;
    for (int k = 0; k < maxc; ++k) cptr[k + 1] += cptr[k];
    {
        std::vector<int> fill(cptr.begin(), cptr.end() - 1);
        for (int i = 0; i < N; ++i) cols[fill[colour[i]]++] = i;
    }
    // entries per colour: for each column j of the colour, rows = pattern of column j
    std::vector<int> erow, epos, ecol, eptr(maxc + 1, 0);
    erow.reserve(ia[N]); epos.reserve(ia[N]); ecol.reserve(ia[N]);
    for (int k = 0; k < maxc; ++k) {
        for (int q = cptr[k]; q < cptr[k + 1]; ++q) {
            int j = cols[q];
            for (int p = ia[j]; p < ia[j + 1]; ++p) {
                int row = ja[p];
                // position of (row, j) in row's sorted column list
                int lo = ia[row], hi = ia[row + 1];
                int pos = (int)(std::lower_bound(ja.begin() + lo, ja.begin() + hi, j) - ja.begin());
                erow.push_back(row); epos.push_back(pos); ecol.push_back(j);
            }
        }
        eptr[k + 1] = (int)erow.size();
    }
    jd->cptr = cptr;
    jd->eptr = eptr;
    if (jd->cols.upload(cols.data(), N) || jd->erow.upload(erow.data(), erow.size()) ||
        jd->epos.upload(epos.data(), epos.size()) || jd->ecol.upload(ecol.data(), ecol.size()))
        return -1;
    jd->coloured = true;
    return 0;
}

fvp_csr *jacobian_handle(fvp_ctx *c) {
    if (jac_init(c)) return nullptr;
    fvp_csr_set_stream(c->jd->J, c->stream);
    return c->jd->J;
}

void jac_free(fvp_ctx *c) {
    if (!c->jd) return;
    fvp_jacdata *jd = c->jd;
    fvp_csr_destroy(jd->J);
    jd->cols.release(); jd->erow.release(); jd->epos.release(); jd->ecol.release();
    jd->shift.release(); jd->ys.release(); jd->yps.release(); jd->Fs.release();
    jd->cptr2.release(); jd->vptr.release(); jd->visit.release(); jd->code.release(); jd->code32.release();
    jd->dpos.release(); jd->contrib.release(); jd->rec.release(); jd->dterm.release();
    delete jd;
    c->jd = nullptr;
}

}  // namespace fvp

extern "C" int fvp_precon_setup(fvp_ctx *c, double t, double c_j, double h, const double *psi, const double *psip,
                                const double *F0, const double *ewt, int type) {
    if (!c || !psi || !psip || !F0 || !ewt) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (jac_init(c)) return -1;
    fvp_jacdata *jd = c->jd;
    hipStream_t s = c->stream;
    fvp_csr_set_stream(jd->J, s);
    const int N = c->N;
    const double eps = 1.4901161193847656e-08;  // sqrt(2^-52)
    if (!c->averaging && c->jac_mode == FVP_JACOBIAN_ELEMENT) {
        const FdJacobian fd{eps, h, c_j, psi, psip, ewt, jd->shift.p, jd->dterm.p, jd->rec.p, jd->contrib.p,
                            jd->rows, jd->max_visits, jd->vptr.p, jd->visit.p, jd->cptr2.p, jd->code.p, jd->code32.p,
                            jd->J->ia.p, jd->dpos.p, jd->J->a.p};
        if (fd_jacobian_elem(c, fd, type == FVP_PRECON_BJILU0_F32)) return -1;
        return precon_build_impl(jd->J, type);
    }
    shift_kernel<<<nblk(N, 256), 256, 0, s>>>(N, eps, h, psi, psip, ewt, jd->shift.p);
    if (colour_init(c)) return -1;
    vcopy<<<nblk(N, 256), 256, 0, s>>>(N, psi, jd->ys.p);
    vcopy<<<nblk(N, 256), 256, 0, s>>>(N, psip, jd->yps.p);
    for (int k = 0; k < jd->ncol; ++k) {
        int nc = jd->cptr[k + 1] - jd->cptr[k];
        int ne = jd->eptr[k + 1] - jd->eptr[k];
        perturb_kernel<<<nblk(nc, 256), 256, 0, s>>>(nc, jd->cols.p + jd->cptr[k], jd->shift.p, c_j, psi, psip,
                                                     jd->ys.p, jd->yps.p, 0);
        if (residual_impl(c, t, jd->ys.p, jd->yps.p, jd->Fs.p, c->averaging)) return -1;
        fd_scatter<<<nblk(ne, 256), 256, 0, s>>>(ne, jd->erow.p + jd->eptr[k], jd->epos.p + jd->eptr[k],
                                                 jd->ecol.p + jd->eptr[k], F0, jd->Fs.p, jd->shift.p, jd->J->a.p);
        perturb_kernel<<<nblk(nc, 256), 256, 0, s>>>(nc, jd->cols.p + jd->cptr[k], jd->shift.p, c_j, psi, psip,
                                                     jd->ys.p, jd->yps.p, 1);
    }
    FVP_HIP(hipGetLastError());
    return precon_build_impl(jd->J, type);
}

namespace fvp {
// z = M^-1 (r / rdiv): the integrator's scaled solve (tmp: a work vector of N)
int precon_solve_div(fvp_ctx *c, const double *r, const double *rdiv, double *tmp, double *z, const double **zn2,
                     int *zn2_count) {
    if (!c->jd || c->jd->J->ptype < 0) { set_error("fvp_precon_setup has not run"); return -1; }
    fvp_csr *A = c->jd->J;
    fvp_csr_set_stream(A, c->stream);
    const bool bj = A->ptype == FVP_PRECON_BJILU0 || A->ptype == FVP_PRECON_BJILU0_F32;
    const bool one = A->ptype == FVP_PRECON_ILU0 && A->one;
    const int np = bj ? A->nblk : one ? 1 : 0;
    double *part = nullptr;
    if (zn2 && np) {
        if ((size_t)np > A->b_zn2.n && A->b_zn2.alloc(np)) return -1;
        part = A->b_zn2.p;
    }
    prof_mark(c, 2, 0);
    int rc = precon_apply_impl(A, r, z, rdiv, tmp, part);
    prof_mark(c, 2, 1);
    if (zn2) *zn2 = part;
    if (zn2_count) *zn2_count = part ? np : 0;
    return rc;
}
}  // namespace fvp

extern "C" int fvp_precon_solve(fvp_ctx *c, const double *r, double *z) {
    if (!c || !r || !z) { set_error("null argument"); return -1; }
    if (!c->jd || c->jd->J->ptype < 0) { set_error("fvp_precon_setup has not run"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    fvp_csr_set_stream(c->jd->J, c->stream);
    prof_mark(c, 2, 0);
    int rc = precon_apply_impl(c->jd->J, r, z);
    prof_mark(c, 2, 1);
    return rc;
}

extern "C" int fvp_set_jacobian_mode(fvp_ctx *c, int mode) {
    if (!c) { set_error("null argument"); return -1; }
    if (mode != FVP_JACOBIAN_ELEMENT && mode != FVP_JACOBIAN_COLOURED) { set_error("invalid Jacobian mode"); return -1; }
    c->jac_mode = mode;
    return 0;
}

extern "C" int fvp_jacobian(fvp_ctx *c, fvp_csr **A) {
    if (!c || !A) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (jac_init(c)) return -1;
    *A = c->jd->J;
    return 0;
}

extern "C" int fvp_set_block_rows(fvp_ctx *c, int rows) {
    if (!c) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (jac_init(c)) return -1;
    return set_block_rows(c->jd->J, rows);
}

extern "C" int fvp_set_overlap(fvp_ctx *c, int layers) {
    if (!c) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (jac_init(c)) return -1;
    return set_overlap(c->jd->J, layers);
}

extern "C" int fvp_colours(fvp_ctx *c, int *n_colours, int *colour_host) {
    if (!c || !n_colours) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (colour_init(c)) return -1;
    *n_colours = c->jd->ncol;
    if (colour_host) std::copy(c->jd->colour.begin(), c->jd->colour.end(), colour_host);
    return 0;
}

extern "C" int fvp_newton_gmres(fvp_ctx *c, double t, const double *psi, const double *psip, const double *F0,
                                double c_j, const double *b, double *x, const fvp_gmres_params *p,
                                fvp_gmres_stats *st) {
    if (!c || !psi || !psip || !F0 || !b || !x || !p) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    if (jac_init(c)) return -1;
    fvp_csr *W = c->jd->J;
    fvp_csr_set_stream(W, c->stream);
    Op op = [=](const double *in, double *out) {
        return jv_impl(c, t, psi, psip, F0, c_j, in, out, nullptr, nullptr, nullptr, 0, W->skip);
    };
    Op pc;
    if (W->ptype > 0) pc = [W](const double *in, double *out) { return precon_apply_impl(W, in, out); };
    return gmres_device(W, c->stream, c->N, op, pc, b, x, p, st, nullptr, diagonal_of(W));
}
