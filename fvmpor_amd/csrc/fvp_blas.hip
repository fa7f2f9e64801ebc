// Vector kernels of the Newton-Krylov loop: wavefront-shuffle reductions
// (norms, fused multi-dots for Gram-Schmidt), axpy forms, and the
// finite-difference Jacobian-vector product.
#include <hip/hip_runtime.h>

#include <cmath>

#include "fvp_blas.h"
#include "fvp_internal.h"
#include "fvp_sums.h"

namespace fvp {

constexpr int kRedBlocks = 512;   // partial sums per reduction (>= 2 per CU)
constexpr int kRedThreads = 256;

// partials[b] = sum over this block's grid-stride slice of x*y (x == y gives ||x||^2)
__global__ void __launch_bounds__(kRedThreads) dot_partial(long n, const double *__restrict__ x,
                                                          const double *__restrict__ y, double *__restrict__ part) {
    __shared__ double lds[kRedThreads / 64];
    double s = 0.;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        s += x[i] * y[i];
    s = block_sum(s, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// the same for ||psi||^2 (part) and ||v||^2 (part + kRedBlocks) in one launch
__global__ void __launch_bounds__(kRedThreads) norms_partial(long n, const double *__restrict__ psi,
                                                            const double *__restrict__ v, double *__restrict__ part) {
    __shared__ double lds[kRedThreads / 64];
    double a = 0., b = 0.;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const double x = psi[i], y = v[i];
        a += x * x;
        b += y * y;
    }
    a = block_sum(a, lds);
    b = block_sum(b, lds);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = a;
        part[kRedBlocks + blockIdx.x] = b;
    }
}

// out[0] = sum of np partials (fixed order: deterministic)
__global__ void __launch_bounds__(kRedThreads) sum_partials(int np, const double *__restrict__ part,
                                                           double *__restrict__ out) {
    __shared__ double lds[kRedThreads / 64];
    // each lane's partials in order, four loads in flight at a time
    double s = 0.;
    const int bd = blockDim.x;
    for (int i0 = threadIdx.x; i0 < np; i0 += 4 * bd) {
        double q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = i0 + u * bd < np ? part[i0 + u * bd] : 0.;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i0 + u * bd < np) s += q[u];
    }
    s = block_sum(s, lds);
    if (threadIdx.x == 0) out[0] = s;
}

// FD increment sigma = sqrt(eps) * ||psi|| / ||v|| from two squared norms
__global__ void __launch_bounds__(kRedThreads) jv_sigma(int np, const double *__restrict__ part_psi,
                                                       const double *__restrict__ part_v, double *__restrict__ sig) {
    __shared__ double lds[kRedThreads / 64];
    double a = 0., b = 0.;
    for (int i = threadIdx.x; i < np; i += blockDim.x) { a += part_psi[i]; b += part_v[i]; }
    a = block_sum(a, lds);
    b = block_sum(b, lds);
    if (threadIdx.x == 0) sig[0] = jv_sigma_of(a, b);
}

// the same from ||psi||^2 already reduced (psi_n2[0]) and the partials of ||v||^2
__global__ void __launch_bounds__(kRedThreads) jv_sigma_n2(int np, const double *__restrict__ psi_n2,
                                                          const double *__restrict__ part_v, double *__restrict__ sig) {
    __shared__ double lds[kRedThreads / 64];
    double b = 0.;
    for (int i = threadIdx.x; i < np; i += blockDim.x) b += part_v[i];
    b = block_sum(b, lds);
    if (threadIdx.x == 0) sig[0] = jv_sigma_of(psi_n2[0], b);
}

__global__ void jv_perturb(long n, const double *__restrict__ sig, double cj, const double *__restrict__ psi,
                           const double *__restrict__ psip, const double *__restrict__ v, double *__restrict__ y,
                           double *__restrict__ yp) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = sig[0];
    y[i] = psi[i] + s * v[i];
    yp[i] = psip[i] + cj * (s * v[i]);
}

__global__ void jv_finish(long n, const double *__restrict__ sig, const double *__restrict__ F1,
                          const double *__restrict__ F0, const double *__restrict__ osc, double *__restrict__ Jv) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double d = (F1[i] - F0[i]) / sig[0];
    Jv[i] = osc ? d * osc[i] : d;
}

static inline int nblk(long n, int bs) { return (int)((n + bs - 1) / bs); }

int dot_async(hipStream_t s, long n, const double *x, const double *y, double *part, double *out) {
    dot_partial<<<kRedBlocks, kRedThreads, 0, s>>>(n, x, y, part);
    sum_partials<<<1, kRedThreads, 0, s>>>(kRedBlocks, part, out);
    FVP_HIP(hipGetLastError());
    return 0;
}

int HostSlots::alloc(int slots) {
    release();
    const size_t bytes = sizeof(double) * kSlot * slots;
    if (hipHostMalloc((void **)&p, bytes, hipHostMallocCoherent) != hipSuccess) {
        p = nullptr;
        set_error("pinned host allocation failed");
        return -1;
    }
    std::fill(p, p + (size_t)kSlot * slots, 0.);
    tag = 0.;
    return 0;
}

void HostSlots::release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
}

// A queue that ends (or fails) without having written the tag is an error; asked
// for only now and then, since the query costs more than the reads.
int slot_wait(hipStream_t s, const double *slot, double tag) {
    auto there = [&]() {
        double v;
        __atomic_load(slot + kSlot - 1, &v, __ATOMIC_ACQUIRE);
        return v == tag;
    };
    for (long k = 1; !there(); ++k) {
        if (k & 0xfffff) continue;
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) continue;
        FVP_HIP(e);
        if (there()) break;
        set_error("the queue ended without its result");
        return -1;
    }
    return 0;
}

}  // namespace fvp

using namespace fvp;

namespace fvp {
int jv_impl(fvp_ctx *c, double t, const double *psi, const double *psip, const double *F0, double c_j,
            const double *v, double *Jv, const double *psi_n2, const double *osc, const double *v_n2,
            int v_count, const double *skip) {
    hipStream_t s = c->stream;
    const long N = c->N;
    double *part = c->red.p;  // [0, 512) psi partials, [512, 1024) v partials, [1024] sigma
    const double *pv = part + kRedBlocks;
    int np = kRedBlocks;
    if (psi_n2 && v_n2) {  // from the solve that wrote v
        pv = v_n2;
        np = v_count;
    } else if (psi_n2) {
        dot_partial<<<kRedBlocks, kRedThreads, 0, s>>>(N, v, v, part + kRedBlocks);
    } else {
        norms_partial<<<kRedBlocks, kRedThreads, 0, s>>>(N, psi, v, part);
    }
    FVP_HIP(hipGetLastError());
    if (!c->averaging) {
        // perturbation and difference quotient fused into the residual kernels, the first
        // of which forms sigma from the partials.  J v by itself, 515 747 nodes: 70.2
        // us with a launch per norm and one for sigma, 68.5 so
        JvArgs jv;
        jv.v = v; jv.sig = part + 2 * kRedBlocks; jv.F0 = F0; jv.cj = c_j; jv.osc = osc; jv.skip = skip;
        jv.psi_n2 = psi_n2; jv.part_psi = psi_n2 ? nullptr : part; jv.part_v = pv; jv.np = np;
        jv.sig_out = part + 2 * kRedBlocks;
        return residual_impl(c, t, psi, psip, Jv, 0, &jv);
    }
    if (psi_n2) jv_sigma_n2<<<1, kRedThreads, 0, s>>>(np, psi_n2, pv, part + 2 * kRedBlocks);
    else jv_sigma<<<1, kRedThreads, 0, s>>>(np, part, pv, part + 2 * kRedBlocks);
    jv_perturb<<<nblk(N, 256), 256, 0, s>>>(N, part + 2 * kRedBlocks, c_j, psi, psip, v, c->tmp1.p, c->tmp2.p);
    FVP_HIP(hipGetLastError());
    if (residual_impl(c, t, c->tmp1.p, c->tmp2.p, c->tmp3.p, c->averaging)) return -1;
    jv_finish<<<nblk(N, 256), 256, 0, s>>>(N, part + 2 * kRedBlocks, c->tmp3.p, F0, osc, Jv);
    FVP_HIP(hipGetLastError());
    return 0;
}
}  // namespace fvp

extern "C" int fvp_jv(fvp_ctx *c, double t, const double *psi, const double *psip, const double *F0, double c_j,
                      const double *v, double *Jv) {
    if (!c || !psi || !psip || !F0 || !v || !Jv) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    return jv_impl(c, t, psi, psip, F0, c_j, v, Jv, nullptr, nullptr);
}
