// CVFE Richards residual on gfx950.
//
// The reference evaluates the residual as a chain of CSR SpMVs over per-CV-face
// geometry tables plus ~13 elementwise passes over 36 M face arrays
// (fvmpor_ODE_impl.cpp:62-115, fvmpor.h:646-945).  Here the CV-face geometry
// is rebuilt per element from node coordinates: on a linear simplex the
// median-dual face between nodes a and b inside element e has the area vector
//     S_ab = |e| / (d+1) * (grad N_b - grad N_a)            (oriented a -> b)
// which equals the reference's quad / segment normal times area
// (cvface_shape.h:46-78, mesh.cpp:844-1010), so the Darcy flux across it is
//     q . S_ab = |e| / (d+1) * (g_b - g_a),   g_k = grad N_k . q,
// with q = -K (grad psi + e_gravity) constant on the element (fvmpor.h:681-717).
// Kernels:
//   vg_kernel      per node: van Genuchten Sw, dSw/dpsi, k_r for every zone the
//                  CV touches, CV-averaged capacity ahh (fvmpor.h:874-945)
//   owner_lds, owner_imports  per node tile: gradient, 3 or 6 face fluxes and
//                  upwinded k_r of the tile's elements, once each, from node records
//                  in LDS, flux sums there, then F = acc / V - psi' ahh, boundary
//                  fluxes, Dirichlet rows (fvmpor_ODE_impl.cpp:99-115); small problems
//                  with vg_kernel's pass inside
//   owner_kernel, owner_finalize  the same gathering from memory, where a tile's
//                  records do not fit the LDS
//   tile_lds_kernel  the same from staged windows, every element touching the tile
//   face_flux_kernel, edge_flux_kernel, mask_kernel  begin_step's upwind weights
//                  (fvmpor_ODE_impl.cpp:118-142)
//   fd_nodes, fd_elem_kernel, fd_gather  the element-local FD Jacobian
//   elem_kernel    per element, atomic scatter: the residual with averaged
//                  weights, before the first begin_step, then finalize
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "fvp_blas.h"
#include "fvp_internal.h"
#include "fvp_sums.h"

namespace fvp {

// a J v row, scaled by the optional row weights of the integrator's scaled solve
__device__ __forceinline__ double jv_scaled(const JvArgs &jv, int i, double d) {
    return jv.osc ? d * jv.osc[i] : d;
}

// ln x and e^x for vg_eval.  The van Genuchten pass is bound by FP64 instructions, and
// the library's pair takes about 125 of them; these take 50, to 0.92 and 1.05 ulp
// (no worse in k_r, S and dS/dh, whose errors come from the arguments' rounding).
// 1 024 000 nodes: vg_kernel 33 us with the library's, 24 to 26 with these.
// ln: x = 2^k m with m in [sqrt(1/2), sqrt(2)), f = m - 1, s = f / (2 + f), and from
// ln m = 2 atanh s = 2 s + s R, 2 s = f - s f: ln m = f - s (f - R), R = s^2 P(s^2),
// P the Chebyshev fit of degree 6 to the atanh series (1.6e-18); the published scheme of
// fdlibm's log with a polynomial of its own.  0 gives -inf, below NaN, inf gives inf (a
// head so dry that (alpha |h|)^n overflows: S = S_r, k_r = 0).
__device__ __forceinline__ double vg_log(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);
    int k = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    k = low ? k - 1 : k;
    const double f = m - 1., d = m + 1.;
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.), r);
    r = fma(r, fma(-d, r, 1.), r);
    const double s = f * r, t = s * s, kd = k;
    double p = 0.14616449685043406;
    p = fma(p, t, 0.15331721600556042);
    p = fma(p, t, 0.18182889125261723);
    p = fma(p, t, 0.2222221113479508);
    p = fma(p, t, 0.28571428625975487);
    p = fma(p, t, 0.39999999999899505);
    p = fma(p, t, 0.666666666666667);
    // ln 2 in two parts, the first times any k exact
    const double c = fma(kd, -1.9082149292705877e-10, s * (f - t * p));
    const double y = fma(kd, 0.6931471803691238, f - c);
    return x > 0. ? (x < __builtin_inf() ? y : x) : x == 0. ? -__builtin_inf() : __builtin_nan("");
}

// e^x = 2^k e^r, r = x - k ln 2 in two parts, e^r = 1 + (r + r^2 P(r)), P the Chebyshev
// fit of degree 9 on |r| <= ln 2 / 2 (1.3e-17).  Overflows to inf, underflows to 0.
__device__ __forceinline__ double vg_exp(double x) {
    x = x < -750. ? -750. : x > 720. ? 720. : x;
    const double kd = rint(x * 1.4426950408889634);
    const double r = fma(kd, -1.9082149292705877e-10, fma(kd, -0.6931471803691238, x));
    double p = 2.5100375832561234e-08;
    p = fma(p, r, 2.7620075879983367e-07);
    p = fma(p, r, 2.7557268480310024e-06);
    p = fma(p, r, 2.4801521322368692e-05);
    p = fma(p, r, 0.00019841269863040545);
    p = fma(p, r, 0.0013888888917196719);
    p = fma(p, r, 0.008333333333330065);
    p = fma(p, r, 0.041666666666624164);
    p = fma(p, r, 0.16666666666666669);
    p = fma(p, r, 0.5000000000000001);
    return __builtin_amdgcn_ldexp(1. + fma(r * r, p, r), (int)kd);
}

__device__ __forceinline__ void vg_eval(double h, const double *zp, double &Sw, double &dSw, double &krw) {
    if (h >= 0.) { Sw = 1.; dSw = 0.; krw = 1.; return; }
    // The reference's operation order, with each power x^p taken as
    // exp(p ln x) on the already-rounded base (a few ulp from pow, which keeps
    // extra precision internally and costs about twice as much in FP64).
    const double nVG = zp[Z_N], mVG = zp[Z_M], S_r = zp[Z_SR];
    double d = vg_exp(nVG * vg_log(-zp[Z_ALPHA] * h));  // a = (alpha |h|)^n
    double s = d + 1.;                            // b
    double k = -1. / s;
    d /= s;
    s = vg_exp(-mVG * vg_log(s));                       // Se = b^-m
    d *= s;
    d /= h;
    d *= -(1 - S_r) * (nVG - 1);
    k += 1.;
    k = vg_exp(mVG * vg_log(k));                        // (1 - 1/b)^m
    k -= 1.;
    k = k * k;
    k *= sqrt(s);
    s *= (1 - S_r);
    s += S_r;
    Sw = s; dSw = d; krw = k;
}

// Node i's zones (mask bits m, ascending): put(zone, rank among them, k_r) for
// each; returns the CV-averaged capacity (without CAP: 0).
template <bool CAP, typename Put>
__device__ __forceinline__ double vg_node(int N, int i, double h, unsigned m, const double *zp,
                                          const double *__restrict__ zw, double rho0, Put put) {
    double phi = 0., Sw = 0., dSw = 0., Ss = 0.;
    for (int r = 0; m; ++r) {
        const int z = __ffs(m) - 1;
        m &= m - 1;
        const double *p = zp + 10 * z;
        const double w = CAP ? zw[(size_t)z * N + i] : 0.;
        double s, d, k;
        vg_eval(h, p, s, d, k);
        put(z, r, k);
        if (CAP) {
            phi += p[Z_PHI] * w;
            Sw += s * w;
            dSw += d * w;
            Ss += p[Z_SS] * w;
        }
    }
    return (phi * dSw + Ss * Sw) * rho0;
}

// The FD increment of J v from np partials of ||v||^2 and, where given, of ||psi||^2,
// summed in the order of jv_sigma and jv_sigma_n2 (the same sigma bit for bit in every
// workgroup and thread); red: eight doubles.  Holds one barrier (five, a block sum per
// norm and a broadcast, took 17.1 us instead of 16.9 in vg_kernel, 515 747 nodes).
__device__ __forceinline__ double jv_sigma_block(const JvArgs &jv, double *red) {
    // each lane's partials in order, four loads in flight at a time
    const int bd = 256;
    auto sum = [&](const double *part) {
        double b = 0.;
        if (threadIdx.x < bd)
            for (int k0 = threadIdx.x; k0 < jv.np; k0 += 4 * bd) {
                double q[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) q[u] = k0 + u * bd < jv.np ? part[k0 + u * bd] : 0.;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k0 + u * bd < jv.np) b += q[u];
            }
        return b;
    };
    double b = sum(jv.part_v), a = jv.part_psi ? sum(jv.part_psi) : 0.;
    b = wave_sum(b);
    if (jv.part_psi) a = wave_sum(a);
    const int waves = bd / 64, w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0 && w < waves) {
        red[w] = b;
        red[waves + w] = a;
    }
    const double n2 = jv.part_psi ? 0. : jv.psi_n2[0];
    __syncthreads();
    b = a = 0.;
    for (int k = 0; k < waves; ++k) {
        b += red[k];
        a += red[waves + k];
    }
    return jv_sigma_of(jv.part_psi ? a : n2, b);
}

// One node per thread, the zone parameters in LDS.  Nodes of several zones are left to
// the first workgroups, which take them from a list (mznode, made at set-up): a per-lane
// loop over the zones made every wavefront pay for the most zones any of its nodes has
// (1 024 000 nodes, a quarter of them at layer boundaries: 41 us with the library's ln
// and e^x; 33 us with a list of the workgroup's own nodes, 24 with the ln and e^x
// above, 21 from one list, without the second phase of few lanes behind a barrier).
// Bound by FP64 instructions and the latency around them.
// JV with jv.np > 0: every workgroup reduces the np partials of ||v||^2 in the
// fixed order of jv_sigma_n2 (the same sigma bit for bit), those of ||psi||^2
// too where they come as partials, and workgroup 0 stores sigma for the
// finalisation, so no launch of its own is needed.
template <bool JV>
__global__ void __launch_bounds__(256) vg_kernel(int N, int nmz, const int *__restrict__ mznode, ZoneTable zt,
                                                 double rho0, const double *__restrict__ psi,
                                                 const uint8_t *__restrict__ zmask, const double *__restrict__ zw,
                                                 double *__restrict__ kr, double *__restrict__ cap, JvArgs jv,
                                                 double *__restrict__ nrec) {
    __shared__ double zp[kMaxZones * 10];
    __shared__ double red[8];
    if (threadIdx.x < 10 * zt.nz) zp[threadIdx.x] = zt.p[threadIdx.x / 10][threadIdx.x % 10];
    // the node's own inputs are loaded first: their latency overlaps sigma's reduction
    const int mzb = (nmz + 255) / 256;
    const bool several = (int)blockIdx.x < mzb;
    int i = ((int)blockIdx.x - (several ? 0 : mzb)) * 256 + threadIdx.x;
    bool live = i < (several ? nmz : N);
    if (several) i = live ? mznode[i] : 0;
    double h = live ? psi[i] : 0.;
    const double vi = JV && live ? jv.v[i] : 0.;
    const unsigned m = live ? zmask[i] : 0u;
    double sg = 0.;
    if (JV && jv.np > 0) {
        sg = jv_sigma_block(jv, red);  // holds a barrier, so the zone table is in place
        if (threadIdx.x == 0 && blockIdx.x == 0) jv.sig_out[0] = sg;
    } else {
        __syncthreads();
        if (JV) sg = jv.sig[0];
    }
    if (!live || (!several && (m & (m - 1)))) return;
    if (JV) h += sg * vi;
    // the head of the node record the element kernel gathers (x, y, z are
    // written once at set-up)
    if (nrec) nrec[4 * (size_t)i + 3] = h;
    cap[i] = vg_node<true>(N, i, h, m, zp, zw, rho0, [&](int z, int, double k) { kr[(size_t)z * N + i] = k; });
}

__device__ __forceinline__ void load_pt(const double *__restrict__ xyz, int i, double &x, double &y, double &z) {
    x = xyz[3 * i]; y = xyz[3 * i + 1]; z = xyz[3 * i + 2];
}

// Local edges in the element edge order of mesh.cpp:409-500: triangle edges
// (0,1) (1,2) (2,0); tetrahedron edges (0,1) (1,2) (2,0) (0,3) (1,3) (2,3).
// Compile-time functions, so that unrolled loops index registers directly.
__device__ constexpr int edge_a(int j) { return j % 3; }
__device__ constexpr int edge_b(int j) { return j < 3 ? (j + 1) % 3 : 3; }

// Face fluxes of one element, summed per element node (f[k] = net inflow into
// node k's control volume, rho0 k_r q.S over the element's CV faces).
// MODE 0: upwind k_r from the element's mask bits; MODE 1: averaged k_r
// (0.5 front + 0.5 back); MODE 2: averaged k_r, and instead of node sums the
// face fluxes (back -> front) are stored per (element, local edge) in qface
// for the edge-flux sign test.
// zk: per-zone K_xx, K_yy, K_zz in LDS.  JV: the state is psi + sig v.
// The per-element record: nodes, zone, conductivity multiplier, upwind and
// orientation bits (loaded ahead of use by the owner kernel's pipeline).
struct ElemRec {
    int4 c4;
    int z;
    double km;
    unsigned mask, orient;
};

template <int MODE>
__device__ __forceinline__ ElemRec load_elem(int e, const int4 *__restrict__ conn, const uint8_t *__restrict__ ezone,
                                             const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
                                             const uint8_t *__restrict__ eorient) {
    ElemRec r;
    r.c4 = conn[e];
    r.z = ezone[e];
    r.km = kmul[e];
    r.mask = MODE == 0 ? emask[e] : 0u;
    r.orient = MODE != 0 ? eorient[e] : 0u;
    return r;
}

// t ? x : y on the bit patterns: keeps the choice between two register
// values a choice of values (a plain conditional between two elements of a
// register array is turned into an indexed load from the stack)
__device__ __forceinline__ double bit_select(unsigned t, double x, double y) {
    const unsigned long long m = 0ULL - (unsigned long long)(t & 1u);
    return __longlong_as_double((__double_as_longlong(x) & (long long)m) | (__double_as_longlong(y) & (long long)~m));
}

// One element's node values: coordinates, head (J v: psi + sig v) and the
// relative permeability of the element's zone at each node.
template <int DIM>
struct NodeVals {
    double px[DIM + 1], py[DIM + 1], pz[DIM + 1], h[DIM + 1], k[DIM + 1];
};

template <int DIM, bool JV>
__device__ __forceinline__ void load_nodes(const ElemRec &rec, int N, const double *__restrict__ xyz,
                                           const double *__restrict__ psi, const double *__restrict__ v, double sig,
                                           const double *__restrict__ kr, NodeVals<DIM> &nv) {
    const int n[4] = {rec.c4.x, rec.c4.y, rec.c4.z, rec.c4.w};
    const double *krz = kr + (size_t)rec.z * N;
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) {
        load_pt(xyz, n[k], nv.px[k], nv.py[k], nv.pz[k]);
        nv.h[k] = JV ? psi[n[k]] + sig * v[n[k]] : psi[n[k]];
        nv.k[k] = krz[n[k]];
    }
}

// load_nodes from the packed node records (x, y, z, head; two 16-byte loads per node)
template <int DIM>
__device__ __forceinline__ void load_nodes_rec(const ElemRec &rec, int N, const double *__restrict__ nrec,
                                               const double *__restrict__ kr, NodeVals<DIM> &nv) {
    const int n[4] = {rec.c4.x, rec.c4.y, rec.c4.z, rec.c4.w};
    const double *krz = kr + (size_t)rec.z * N;
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) {
        const double2 *r = reinterpret_cast<const double2 *>(nrec + 4 * (size_t)n[k]);
        const double2 a = r[0], b = r[1];
        nv.px[k] = a.x; nv.py[k] = a.y; nv.pz[k] = b.x; nv.h[k] = b.y;
        nv.k[k] = krz[n[k]];
    }
}

// The element's face fluxes from its record and node values; f[k] = net mass
// flow into node k (n[k] its node ids).
template <int DIM, int MODE>
__device__ __forceinline__ void element_fluxes_vals(int e, const ElemRec &rec, const NodeVals<DIM> &nv,
                                                    const double *zk, double rho0, double *__restrict__ qface,
                                                    int n[4], double f[4]) {
    constexpr int NPE = DIM + 1;
    constexpr int NED = DIM == 2 ? 3 : 6;
    n[0] = rec.c4.x; n[1] = rec.c4.y; n[2] = rec.c4.z; n[3] = rec.c4.w;
    const double *px = nv.px, *py = nv.py, *pz = nv.pz, *h = nv.h;
    const int z = rec.z;
    const double km = rec.km;
    double G[NPE][3];  // adjugate rows: grad N_k * det
    double det;
    if (DIM == 3) {
        double ux = px[1] - px[0], uy = py[1] - py[0], uz = pz[1] - pz[0];
        double vx = px[2] - px[0], vy = py[2] - py[0], vz = pz[2] - pz[0];
        double wx = px[3] - px[0], wy = py[3] - py[0], wz = pz[3] - pz[0];
        G[1][0] = vy * wz - vz * wy; G[1][1] = vz * wx - vx * wz; G[1][2] = vx * wy - vy * wx;
        G[2][0] = wy * uz - wz * uy; G[2][1] = wz * ux - wx * uz; G[2][2] = wx * uy - wy * ux;
        G[3][0] = uy * vz - uz * vy; G[3][1] = uz * vx - ux * vz; G[3][2] = ux * vy - uy * vx;
        det = ux * G[1][0] + uy * G[1][1] + uz * G[1][2];
    } else {
        double ux = px[1] - px[0], uy = py[1] - py[0];
        double vx = px[2] - px[0], vy = py[2] - py[0];
        G[1][0] = vy; G[1][1] = -vx; G[1][2] = 0.;
        G[2][0] = -uy; G[2][1] = ux; G[2][2] = 0.;
        det = ux * vy - uy * vx;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) G[0][d] = -(G[1][d] + G[2][d] + (DIM == 3 ? G[NPE - 1][d] : 0.));
    const double inv = 1.0 / det;
    // gradient of psi
    double gx = 0., gy = 0., gz = 0.;
#pragma unroll
    for (int k = 1; k < NPE; ++k) {
        double dh = h[k] - h[0];
        gx += dh * G[k][0]; gy += dh * G[k][1]; gz += dh * G[k][2];
    }
    gx *= inv; gy *= inv; gz *= inv;
    // Darcy flux without k_r: q = -K (grad psi + e_gravity), gravity on y (2D) / z (3D)
    double qx = gx * -(zk[3 * z] * km);
    double qy, qz;
    if (DIM == 2) { qy = (gy + 1.) * -(zk[3 * z + 1] * km); qz = 0.; }
    else { qy = gy * -(zk[3 * z + 1] * km); qz = (gz + 1.) * -(zk[3 * z + 2] * km); }
    double g[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) g[k] = G[k][0] * qx + G[k][1] * qy + G[k][2] * qz;
    // |e|/(d+1) * (grad N_b - grad N_a) . q  =  sign(det) / (d! (d+1)) * (g_b - g_a)
    const double sc = (det > 0 ? 1.0 : -1.0) / (DIM == 3 ? 24.0 : 6.0);
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = 0.;
    const unsigned mask = rec.mask;
    const unsigned orient = rec.orient;
#pragma unroll
    for (int j = 0; j < NED; ++j) {
        const int a = edge_a(j);
        const int b = edge_b(j);
        double flux = sc * (g[b] - g[a]);  // flow a -> b
        double krf;
        if (MODE == 0) {
            krf = bit_select((mask >> j) & 1u, nv.k[a], nv.k[b]);
        } else {
            const unsigned a_front = (orient >> j) & 1u;
            double kf = bit_select(a_front, nv.k[a], nv.k[b]);
            double kb = bit_select(a_front, nv.k[b], nv.k[a]);
            krf = kf * 0.5;
            krf += kb * 0.5;
            if (MODE == 2) qface[(size_t)e * NED + j] = krf * (a_front ? -flux : flux);  // back -> front
        }
        double M = rho0 * (krf * flux);
        f[a] -= M;
        f[b] += M;
    }
}

template <int DIM, int MODE, bool JV = false>
__device__ __forceinline__ void element_fluxes_rec(int e, const ElemRec &rec, int N, const double *zk, double rho0,
                                                   const double *__restrict__ xyz, const double *__restrict__ psi,
                                                   const double *__restrict__ v, double sig,
                                                   const double *__restrict__ kr, double *__restrict__ qface,
                                                   int n[4], double f[4]) {
    NodeVals<DIM> nv;
    load_nodes<DIM, JV>(rec, N, xyz, psi, v, sig, kr, nv);
    element_fluxes_vals<DIM, MODE>(e, rec, nv, zk, rho0, qface, n, f);
}

template <int DIM, int MODE, bool JV = false>
__device__ __forceinline__ void element_fluxes(int e, int N, const double *zk, double rho0,
                                               const int4 *__restrict__ conn, const uint8_t *__restrict__ ezone,
                                               const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
                                               const uint8_t *__restrict__ eorient,
                                               const double *__restrict__ xyz, const double *__restrict__ psi,
                                               const double *__restrict__ v, double sig,
                                               const double *__restrict__ kr, double *__restrict__ qface,
                                               int n[4], double f[4]) {
    const ElemRec rec = load_elem<MODE>(e, conn, ezone, kmul, emask, eorient);
    element_fluxes_rec<DIM, MODE, JV>(e, rec, N, zk, rho0, xyz, psi, v, sig, kr, qface, n, f);
}

// Atomic scatter variant: the averaged-weight residual (before the first begin_step).
template <int DIM>
__global__ void __launch_bounds__(256) elem_kernel(int T, int N, ZoneTable zt, double rho0,
                                                   const int4 *__restrict__ conn, const uint8_t *__restrict__ ezone,
                                                   const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
                                                   const uint8_t *__restrict__ eorient,
                                                   const double *__restrict__ xyz, const double *__restrict__ psi,
                                                   const double *__restrict__ kr, double *__restrict__ acc) {
    __shared__ double zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    int n[4];
    double f[4];
    element_fluxes<DIM, 1>(e, N, zk, rho0, conn, ezone, kmul, emask, eorient, xyz, psi, nullptr, 0., kr, nullptr, n, f);
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) atomicAdd(&acc[n[k]], f[k]);
}

// begin_step's face fluxes with averaged k_r (back -> front), per local edge and
// element (one array per local edge, so that the stores are whole lines).  Nodes come
// as 32-byte records and one k_r.  1 500 000 elements: 32 us; 35 with five 8-byte
// gathers a node and the six fluxes of an element side by side (TA requests bound it).
template <int DIM>
__global__ void __launch_bounds__(256) face_flux_kernel(int T, int N, ZoneTable zt, const int4 *__restrict__ conn,
                                                        const uint8_t *__restrict__ ezone,
                                                        const double *__restrict__ kmul,
                                                        const uint8_t *__restrict__ eorient,
                                                        const double *__restrict__ nrec,
                                                        const double *__restrict__ kr, double *__restrict__ qface) {
    constexpr int NED = DIM == 2 ? 3 : 6;
    __shared__ double zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    const ElemRec rec = load_elem<2>(e, conn, ezone, kmul, nullptr, eorient);
    NodeVals<DIM> nv;
    load_nodes_rec<DIM>(rec, N, nrec, kr, nv);
    int n[4];
    double f[4], q[NED];
    element_fluxes_vals<DIM, 2>(0, rec, nv, zk, 1., q, n, f);
#pragma unroll
    for (int j = 0; j < NED; ++j) qface[(size_t)j * T + e] = q[j];
}

// Export slots of an element evaluated in tile [lo, hi): -1 for owned nodes,
// else the next slot of the element's run starting at xd[x] (foreign nodes in
// local order).
template <int DIM>
__device__ __forceinline__ void owner_exports(const ElemRec &r, int lo, int hi, const int *__restrict__ xd, int x,
                                              int d[4]) {
    const int nn[4] = {r.c4.x, r.c4.y, r.c4.z, r.c4.w};
#pragma unroll
    for (int q = 0; q < DIM + 1; ++q) d[q] = (nn[q] >= lo && nn[q] < hi) ? -1 : xd[x++];
}

// Element-owner residual: a workgroup owns the nodes of one tile and evaluates
// the tile's primary elements (lowest node in the tile; every element has
// exactly one primary tile, so each element is evaluated once), gathering node
// data through the caches.  Contributions to owned nodes accumulate in LDS
// (ds_add_f64) and are stored, with the tile's boundary fluxes, to acc; those
// to nodes of other tiles are exports (the element's first: tile base +
// xoff[e], then one per foreign node in local order), each stored to its slot
// xdst[export]; slots are grouped by target node, so the finalisation reads
// each node's imports contiguously.  No global atomics.
template <int DIM, bool JV>
__global__ void __launch_bounds__(512) owner_kernel(
    int N, int ntiles, int tile_nodes, int per_xcd, ZoneTable zt, double rho0, const int4 *__restrict__ conn,
    const uint8_t *__restrict__ ezone, const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
    const double *__restrict__ xyz, const double *__restrict__ nrec, const double *__restrict__ kr,
    const int *__restrict__ eptr, const int *__restrict__ bptr, const int *__restrict__ bnode,
    const double *__restrict__ bval, const unsigned short *__restrict__ xoff, const int *__restrict__ xptr,
    const int *__restrict__ xdst, double *__restrict__ xf, double *__restrict__ acc_g, JvArgs jv) {
    extern __shared__ double sm[];
    const int tile = per_xcd ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
    if (tile >= ntiles) return;  // uniform for the whole workgroup
    // nrec: the packed node records (x, y, z, head) written by the van Genuchten
    // pass, whose head is psi + sigma v for J v; the difference quotient is
    // formed by the finalisation (xyz is read through the records)
    (void)jv;
    (void)xyz;
    const int lo = tile * tile_nodes, hi = min(N, lo + tile_nodes), nown = hi - lo;
    for (int i = threadIdx.x; i < nown; i += blockDim.x) sm[i] = 0.;
    __shared__ double zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    const int *xd = xdst + xptr[tile];
    const int e1 = eptr[tile + 1];
    const int bs = blockDim.x;
    // Two-stage software pipeline over the thread's elements: while element e
    // is evaluated, the node values and export slots of element e + bs and the
    // record of element e + 2 bs are in flight, so the gathers' latency hides
    // behind the flux arithmetic.  Look-ahead indices past the tile's range are
    // clamped to its last element (loaded, never used).
    int e = eptr[tile] + threadIdx.x;
    if (e < e1) {
        const int last = e1 - 1;
        ElemRec cur = load_elem<0>(e, conn, ezone, kmul, emask, nullptr);
        NodeVals<DIM> vc;
        load_nodes_rec<DIM>(cur, N, nrec, kr, vc);
        int dc[4];
        owner_exports<DIM>(cur, lo, hi, xd, xoff[e], dc);
        int en = min(e + bs, last);
        ElemRec nxt = load_elem<0>(en, conn, ezone, kmul, emask, nullptr);
        int xn = xoff[en];
        for (; e < e1; e += bs) {
            NodeVals<DIM> vn;
            int dn[4];
            load_nodes_rec<DIM>(nxt, N, nrec, kr, vn);
            owner_exports<DIM>(nxt, lo, hi, xd, xn, dn);
            const int e2 = min(e + 2 * bs, last);
            const ElemRec nx2 = load_elem<0>(e2, conn, ezone, kmul, emask, nullptr);
            const int x2 = xoff[e2];
            int n[4];
            double f[4];
            element_fluxes_vals<DIM, 0>(e, cur, vc, zk, rho0, nullptr, n, f);
#pragma unroll
            for (int q = 0; q < DIM + 1; ++q) {
                if (dc[q] < 0) atomicAdd(&sm[n[q] - lo], f[q]);
                else xf[dc[q]] = f[q];
            }
            cur = nxt;
            vc = vn;
#pragma unroll
            for (int q = 0; q < 4; ++q) dc[q] = dn[q];
            nxt = nx2;
            xn = x2;
        }
    }
    __syncthreads();
    for (int k = bptr[tile] + threadIdx.x; k < bptr[tile + 1]; k += blockDim.x) sm[bnode[k] - lo] -= bval[k];
    __syncthreads();
    for (int i = threadIdx.x; i < nown; i += blockDim.x) acc_g[lo + i] = sm[i];
}

// Finalisation of the element-owner residual, one workgroup per tile: the
// tile's imports are a contiguous slot range (slots are grouped by target
// node), read coalesced and added to the nodes' own sums in LDS, then
// F = acc / V - psi' ahh (JV: the difference quotient) and the Dirichlet rows.
template <bool JV>
__global__ void __launch_bounds__(1024) owner_finalize(
    int N, int ntiles, int tile_nodes, const double *__restrict__ acc, const int *__restrict__ iptr,
    const int *__restrict__ xtgt, const double *__restrict__ xf, const double *__restrict__ invV,
    const double *__restrict__ psi, const double *__restrict__ psip, const double *__restrict__ cap,
    const int *__restrict__ dptr, const int *__restrict__ dnode, const double *__restrict__ dval,
    double *__restrict__ F, JvArgs jv) {
    extern __shared__ double sm[];
    const int tile = blockIdx.x;
    const int lo = tile * tile_nodes, hi = min(N, lo + tile_nodes), nown = hi - lo;
    for (int i = threadIdx.x; i < nown; i += blockDim.x) sm[i] = acc[lo + i];
    __syncthreads();
    for (int k = iptr[lo] + threadIdx.x; k < iptr[hi]; k += blockDim.x) atomicAdd(&sm[xtgt[k] - lo], xf[k]);
    __syncthreads();
    const double sig = JV ? jv.sig[0] : 0.;
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        const double a = sm[i - lo];
        if (JV) {
            const double yp = psip[i] + jv.cj * (sig * jv.v[i]);
            const double F1 = a * invV[i] - yp * cap[i];
            F[i] = jv_scaled(jv, i, (F1 - jv.F0[i]) / sig);
        } else
            F[i] = a * invV[i] - psip[i] * cap[i];
    }
    __syncthreads();
    for (int k = dptr[tile] + threadIdx.x; k < dptr[tile + 1]; k += blockDim.x) {
        const int i = dnode[k];
        if (JV) {
            const double y = psi[i] + sig * jv.v[i];
            F[i] = jv_scaled(jv, i, ((dval[k] - y) - jv.F0[i]) / sig);
        } else
            F[i] = dval[k] - psi[i];
    }
}

// t ? x : y for the sign-extended bit t (0 or ~0), on the two halves
__device__ __forceinline__ double half_select(unsigned t, double x, double y) {
    const long long a = __double_as_longlong(x), b = __double_as_longlong(y);
    const unsigned lo = ((unsigned)a & t) | ((unsigned)b & ~t);
    const unsigned hi = ((unsigned)(a >> 32) & t) | ((unsigned)(b >> 32) & ~t);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The face fluxes of element_fluxes_vals<DIM, 0>, with fewer operations: gravity is
// added to the head differences (so a hydrostatic element cancels before the
// gradient is formed), rho0 / (d! (d + 1)) comes with the conductivities (kz), the
// sign of det cancels, and node 0's gradient and flux are minus the others' sums.
template <int DIM>
__device__ __forceinline__ void upwind_fluxes(const NodeVals<DIM> &nv, const double *kz, double km, unsigned mask,
                                              double (&f)[DIM + 1]) {
    const double *px = nv.px, *py = nv.py, *pz = nv.pz, *h = nv.h;
    double g[DIM + 1];
    const double ux = px[1] - px[0], uy = py[1] - py[0], vx = px[2] - px[0], vy = py[2] - py[0];
    if (DIM == 3) {
        const double uz = pz[1] - pz[0], vz = pz[2] - pz[0];
        const double wx = px[3] - px[0], wy = py[3] - py[0], wz = pz[3] - pz[0];
        const double a1 = vy * wz - vz * wy, b1 = vz * wx - vx * wz, c1 = vx * wy - vy * wx;
        const double a2 = wy * uz - wz * uy, b2 = wz * ux - wx * uz, c2 = wx * uy - wy * ux;
        const double a3 = uy * vz - uz * vy, b3 = uz * vx - ux * vz, c3 = ux * vy - uy * vx;
        const double det = ux * a1 + uy * b1 + uz * c1;
        const double d1 = (h[1] - h[0]) + uz, d2 = (h[2] - h[0]) + vz, d3 = (h[3] - h[0]) + wz;
        const double t = km / fabs(det);
        const double qx = (d1 * a1 + d2 * a2 + d3 * a3) * (kz[0] * t);
        const double qy = (d1 * b1 + d2 * b2 + d3 * b3) * (kz[1] * t);
        const double qz = (d1 * c1 + d2 * c2 + d3 * c3) * (kz[2] * t);
        g[1] = a1 * qx + b1 * qy + c1 * qz;
        g[2] = a2 * qx + b2 * qy + c2 * qz;
        g[DIM] = a3 * qx + b3 * qy + c3 * qz;
        g[0] = -(g[1] + g[2] + g[DIM]);
    } else {
        const double det = ux * vy - uy * vx;
        const double d1 = (h[1] - h[0]) + uy, d2 = (h[2] - h[0]) + vy;
        const double t = km / fabs(det);
        // gradients of N_1, N_2 times det: (vy, -vx), (-uy, ux)
        const double qx = (d1 * vy - d2 * uy) * (kz[0] * t), qy = (d2 * ux - d1 * vx) * (kz[1] * t);
        g[1] = vy * qx - vx * qy;
        g[2] = ux * qy - uy * qx;
        g[0] = -(g[1] + g[2]);
    }
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) f[k] = 0.;
#pragma unroll
    for (int j = 0; j < (DIM == 2 ? 3 : 6); ++j) {
        const int a = edge_a(j), b = edge_b(j);
        const double kr = half_select((unsigned)((int)(mask << (31 - j)) >> 31), nv.k[a], nv.k[b]);
        const double d = g[b] - g[a];
        f[a] += kr * d;
        f[b] -= kr * d;
    }
}

// Element-owner residual from LDS windows.  A workgroup owns the nodes of one tile
// and evaluates the tile's primary elements (lowest node in the tile), once each.
// It stages one LDS record per node of those elements' window (owned nodes, then
// the halo: higher nodes of other tiles): coordinates, head, flux sum and k_r per
// rank of the node's zones.  Elements then need 18 streamed bytes each and take the
// rest from LDS (per corner the record's place in 14 bits, the rank of the element's
// zone there in 2).  Halo sums leave as one export per (tile, halo node), its slot
// grouped by target node.  An owned node without imports is finished here; the
// others' sums go to acc and owner_imports.
// VG: the van Genuchten pass is part of the staging (owned nodes write the capacity,
// halo nodes are evaluated again); otherwise k_r comes from vg_kernel.  Nodes of
// several zones are set aside in a list and done afterwards, as there.
// Bound by the LDS (268 cycles per 64 elements: 16-byte record reads and four sums)
// and the phases' latency.  1 024 000 nodes, 512-node tiles: 76 us, with vg_kernel 21
// and owner_imports 8 us more.  Gathering from memory through the L1 (owner_kernel,
// kept for windows that do not fit) with a finalisation of its own: 120 + 41 + 33 us.
constexpr int kRecBits = 14, kRecRanks = 4;

// doubles per window record: DIM coordinates, head, sum, k_r per rank; odd, so that
// records start in all banks
__host__ __device__ inline int win_stride(int dim, int nr) { return (dim + 2 + nr) | 1; }

template <int DIM, bool JV, bool VG, int TH>
__global__ void __launch_bounds__(TH) owner_lds(
    int N, int ntiles, int tile_nodes, int per_xcd, int wmax, int nr, ZoneTable zt, double rho0,
    const uint8_t *__restrict__ ezone, const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
    const ushort4 *__restrict__ lconn, const double *__restrict__ xyz, const double *__restrict__ psi,
    const uint8_t *__restrict__ zmask, const double *__restrict__ zw, const double *__restrict__ kr,
    const int *__restrict__ eptr, const int *__restrict__ wptr, const int *__restrict__ whalo,
    const int *__restrict__ xdst,
    double *__restrict__ xf, const int *__restrict__ iptr, const int *__restrict__ bptr,
    const int *__restrict__ bnode, const double *__restrict__ bval, const double *__restrict__ invV,
    const double *__restrict__ psip, double *__restrict__ cap, double *__restrict__ acc_g, double *__restrict__ F,
    JvArgs jv) {
    constexpr int kH = DIM, kAcc = DIM + 1, kK = DIM + 2;
    extern __shared__ __align__(16) double sm[];
    __shared__ double zk[3 * kMaxZones], zp[VG ? 10 * kMaxZones : 1];
    __shared__ double red[16];
    __shared__ int nlist;
    const int tile = per_xcd ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
    if (tile >= ntiles) return;  // uniform for the whole workgroup
    const int lo = tile * tile_nodes, hi = min(N, lo + tile_nodes), nown = hi - lo;
    const int w0 = wptr[tile], win = nown + wptr[tile + 1] - w0;
    const int stride = win_stride(DIM, nr);
    unsigned short *const list = reinterpret_cast<unsigned short *>(sm + wmax * stride);
    const double over = JV ? skip_word(jv.skip) : 0.;
    const double c0 = rho0 / (DIM == 3 ? 24.0 : 6.0);
    for (int k = threadIdx.x; k < 3 * zt.nz; k += TH) zk[k] = zt.p[k / 3][ZK_X + k % 3] * c0;
    if (VG)
        for (int k = threadIdx.x; k < 10 * zt.nz; k += TH) zp[k] = zt.p[k / 10][k % 10];
    if (threadIdx.x == 0) nlist = 0;
    double sig = 0.;
    if (JV && VG && jv.np > 0) {
        sig = jv_sigma_block(jv, red);  // holds a barrier
        if (threadIdx.x == 0 && blockIdx.x == 0) jv.sig_out[0] = sig;
    } else {
        __syncthreads();  // the zone tables
        if (JV) sig = jv.sig[0];
    }
    auto node_of = [&](int i) { return i < nown ? lo + i : whalo[w0 + i - nown]; };
    auto evaluate = [&](int i, int g, double h, unsigned m) {
        double *const rec = sm + i * stride;
        auto put = [&](int, int r, double k) { rec[kK + r] = k; };
        if (i < nown) cap[g] = vg_node<true>(N, g, h, m, zp, zw, rho0, put);
        else vg_node<false>(N, g, h, m, zp, zw, rho0, put);
    };
    for (int i = threadIdx.x; i < win; i += TH) {
        const int g = node_of(i);
        double h = psi[g];
        if (JV) h += sig * jv.v[g];
        const unsigned m = zmask[g];
        double *const rec = sm + i * stride;
        double x, y, z;
        load_pt(xyz, g, x, y, z);
        rec[0] = x;
        rec[1] = y;
        if (DIM == 3) rec[2] = z;
        rec[kH] = h;
        rec[kAcc] = 0.;
        if (VG) {
            if (m & (m - 1)) list[atomicAdd(&nlist, 1)] = (unsigned short)i;
            else evaluate(i, g, h, m);
        } else {
            unsigned q = m;
            for (int r = 0; q; ++r, q &= q - 1) rec[kK + r] = kr[(size_t)(__ffs(q) - 1) * N + g];
        }
    }
    __syncthreads();
    if (JV && over != 0.) return;
    if (VG) {
        for (int k = threadIdx.x; k < nlist; k += TH) {
            const int i = list[k], g = node_of(i);
            evaluate(i, g, sm[i * stride + kH], zmask[g]);
        }
        __syncthreads();
    }
    constexpr int NPE = DIM + 1;
    const int e1 = eptr[tile + 1];
    int e = eptr[tile] + threadIdx.x;
    if (e < e1) {
        // the next element's stream is in flight while this one is evaluated
        ushort4 lc = lconn[e];
        int z = ezone[e];
        double km = kmul[e];
        unsigned mask = emask[e];
        for (; e < e1; e += TH) {
            const int en = min(e + TH, e1 - 1);
            const ushort4 ln = lconn[en];
            const int zn = ezone[en];
            const double kn = kmul[en];
            const unsigned mn = emask[en];
            const unsigned l[4] = {lc.x, lc.y, lc.z, lc.w};
            NodeVals<DIM> nv;
            double *rec[NPE];
#pragma unroll
            for (int q = 0; q < NPE; ++q) {
                rec[q] = sm + (l[q] & ((1u << kRecBits) - 1));
                nv.px[q] = rec[q][0];
                nv.py[q] = rec[q][1];
                nv.pz[q] = DIM == 3 ? rec[q][2] : 0.;
                nv.h[q] = rec[q][kH];
                nv.k[q] = rec[q][kK + (l[q] >> kRecBits)];
            }
            double f[NPE];
            upwind_fluxes<DIM>(nv, zk + 3 * z, km, mask, f);
#pragma unroll
            for (int q = 0; q < NPE; ++q) atomicAdd(rec[q] + kAcc, f[q]);
            lc = ln;
            z = zn;
            km = kn;
            mask = mn;
        }
    }
    __syncthreads();
    for (int k = bptr[tile] + threadIdx.x; k < bptr[tile + 1]; k += TH)
        sm[(bnode[k] - lo) * stride + kAcc] -= bval[k];
    __syncthreads();
    for (int i = threadIdx.x; i < nown; i += TH) {
        const int g = lo + i;
        const double a = sm[i * stride + kAcc];
        if (iptr[g] != iptr[g + 1]) {
            acc_g[g] = a;
            continue;
        }
        if (JV) {
            const double yp = psip[g] + jv.cj * (sig * jv.v[g]);
            const double F1 = a * invV[g] - yp * cap[g];
            F[g] = jv_scaled(jv, g, (F1 - jv.F0[g]) / sig);
        } else
            F[g] = a * invV[g] - psip[g] * cap[g];
    }
    for (int i = nown + threadIdx.x; i < win; i += TH) xf[xdst[w0 + i - nown]] = sm[i * stride + kAcc];
}

// The nodes with imports (inode, ascending): their own sums plus their slots in
// order, then the finalisation.
template <bool JV>
__global__ void __launch_bounds__(256) owner_imports(int nimp, const int *__restrict__ inode,
                                                     const double *__restrict__ acc, const int *__restrict__ iptr,
                                                     const double *__restrict__ xf, const double *__restrict__ invV,
                                                     const double *__restrict__ psip, const double *__restrict__ cap,
                                                     double *__restrict__ F, JvArgs jv) {
    const double over = JV ? skip_word(jv.skip) : 0.;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nimp) return;
    const int i = inode[k];
    const int s0 = iptr[i], s1 = iptr[i + 1];
    if (over != 0.) return;
    double a = acc[i];
    const double iv = invV[i], p = psip[i], c = cap[i];
    const double sig = JV ? jv.sig[0] : 0., v = JV ? jv.v[i] : 0., f0 = JV ? jv.F0[i] : 0.;
    // four slots in flight at a time
    for (int s = s0; s < s1; s += 4) {
        double q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = xf[min(s + u, s1 - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s + u < s1) a += q[u];
    }
    if (JV) {
        const double yp = p + jv.cj * (sig * v);
        const double F1 = a * iv - yp * c;
        F[i] = jv_scaled(jv, i, (F1 - f0) / sig);
    } else
        F[i] = a * iv - p * c;
}

// LDS-staged owner-computes residual.  A workgroup owns tile_nodes nodes; it
// stages the coordinates, heads and relative permeabilities of its window (owned
// nodes plus the halo nodes its elements reach) in LDS with coalesced loads for
// the owned range and one gather per halo node, then evaluates every element
// touching the tile from LDS using the window-local connectivity (8 B per
// element visit), accumulates the flux sums of owned nodes in LDS (ds_add_f64),
// and finishes F = acc / V - psi' ahh, boundary fluxes and Dirichlet rows.
// Elements shared by several tiles are evaluated once per tile and only the
// contributions to owned nodes are kept, so no global atomics are issued; the
// tiles of one XCD are contiguous so their halo nodes share that XCD's L2.
// JV: directional-derivative mode (state psi + sig v, output (F - F0) / sig).
template <int DIM, bool JV>
__global__ void __launch_bounds__(256) tile_lds_kernel(
    int N, int ntiles, int tile_nodes, int per_xcd, int wmax, int ntzmax, ZoneTable zt, double rho0, const uint8_t *__restrict__ ezone,
    const double *__restrict__ kmul, const uint8_t *__restrict__ emask, const double *__restrict__ xyz,
    const double *__restrict__ psi, const double *__restrict__ kr, const int *__restrict__ eptr,
    const int *__restrict__ hptr, const int *__restrict__ hlist, const int *__restrict__ wptr,
    const int *__restrict__ whalo, const int *__restrict__ vptr, const ushort4 *__restrict__ lconn,
    const int *__restrict__ tzone, const double *__restrict__ invV, const double *__restrict__ psip,
    const double *__restrict__ cap, const int *__restrict__ bptr, const int *__restrict__ bnode,
    const double *__restrict__ bval, const int *__restrict__ dptr, const int *__restrict__ dnode,
    const double *__restrict__ dval, double *__restrict__ F, JvArgs jv) {
    extern __shared__ double sm[];
    // workgroups are dealt to the 8 XCDs round-robin: with per_xcd > 0 the
    // tiles of one XCD are contiguous (their halos share its L2)
    const int tile = per_xcd ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
    if (tile >= ntiles) return;  // uniform for the whole workgroup
    const double sig = JV ? jv.sig[0] : 0.;
    const int lo = tile * tile_nodes, hi = min(N, lo + tile_nodes), nown = hi - lo;
    const int w0 = wptr[tile], win = nown + wptr[tile + 1] - w0;
    int tz[4], ntz = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        tz[q] = tzone[tile * 4 + q];
        ntz += tz[q] >= 0;
    }
    double *sx = sm, *sy = sx + wmax, *sz = sy + wmax, *sp = sz + wmax, *sk = sp + wmax;
    double *acc = sk + ntzmax * wmax;
    for (int i = threadIdx.x; i < win; i += blockDim.x) {
        const int g = i < nown ? lo + i : whalo[w0 + i - nown];
        sx[i] = xyz[3 * g];
        sy[i] = xyz[3 * g + 1];
        sz[i] = xyz[3 * g + 2];
        sp[i] = JV ? psi[g] + sig * jv.v[g] : psi[g];
        for (int q = 0; q < ntz; ++q) sk[q * wmax + i] = kr[(size_t)tz[q] * N + g];
    }
    for (int i = threadIdx.x; i < nown; i += blockDim.x) acc[i] = 0.;
    // per-zone conductivity tensor diagonal in LDS: elements of one wavefront
    // index it with their own zone, which a kernel-argument table would turn
    // into select chains over every zone
    __shared__ double zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    constexpr int NPE = DIM + 1;
    constexpr int NED = DIM == 2 ? 3 : 6;
    const int e0 = eptr[tile], np = eptr[tile + 1] - e0, h0 = hptr[tile];
    const int v0 = vptr[tile], nv = vptr[tile + 1] - v0;
    for (int k = threadIdx.x; k < nv; k += blockDim.x) {
        const int e = k < np ? e0 + k : hlist[h0 + k - np];
        const ushort4 lc = lconn[v0 + k];
        const int l[4] = {lc.x, lc.y, lc.z, lc.w};
        const int z = ezone[e];
        const double km = kmul[e];
        const unsigned mask = emask[e];
        const int slot = z == tz[0] ? 0 : z == tz[1] ? 1 : z == tz[2] ? 2 : 3;
        double px[NPE], py[NPE], pz[NPE], h[NPE];
#pragma unroll
        for (int q = 0; q < NPE; ++q) {
            px[q] = sx[l[q]]; py[q] = sy[l[q]]; pz[q] = sz[l[q]]; h[q] = sp[l[q]];
        }
        double G[NPE][3];
        double det;
        if (DIM == 3) {
            double ux = px[1] - px[0], uy = py[1] - py[0], uz = pz[1] - pz[0];
            double vx = px[2] - px[0], vy = py[2] - py[0], vz = pz[2] - pz[0];
            double wx = px[3] - px[0], wy = py[3] - py[0], wz = pz[3] - pz[0];
            G[1][0] = vy * wz - vz * wy; G[1][1] = vz * wx - vx * wz; G[1][2] = vx * wy - vy * wx;
            G[2][0] = wy * uz - wz * uy; G[2][1] = wz * ux - wx * uz; G[2][2] = wx * uy - wy * ux;
            G[3][0] = uy * vz - uz * vy; G[3][1] = uz * vx - ux * vz; G[3][2] = ux * vy - uy * vx;
            det = ux * G[1][0] + uy * G[1][1] + uz * G[1][2];
        } else {
            double ux = px[1] - px[0], uy = py[1] - py[0];
            double vx = px[2] - px[0], vy = py[2] - py[0];
            G[1][0] = vy; G[1][1] = -vx; G[1][2] = 0.;
            G[2][0] = -uy; G[2][1] = ux; G[2][2] = 0.;
            det = ux * vy - uy * vx;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) G[0][d] = -(G[1][d] + G[2][d] + (DIM == 3 ? G[NPE - 1][d] : 0.));
        const double inv = 1.0 / det;
        double gx = 0., gy = 0., gz = 0.;
#pragma unroll
        for (int q = 1; q < NPE; ++q) {
            double dh = h[q] - h[0];
            gx += dh * G[q][0]; gy += dh * G[q][1]; gz += dh * G[q][2];
        }
        gx *= inv; gy *= inv; gz *= inv;
        double qx = gx * -(zk[3 * z] * km);
        double qy, qzz;
        if (DIM == 2) { qy = (gy + 1.) * -(zk[3 * z + 1] * km); qzz = 0.; }
        else { qy = gy * -(zk[3 * z + 1] * km); qzz = (gz + 1.) * -(zk[3 * z + 2] * km); }
        double g[NPE];
#pragma unroll
        for (int q = 0; q < NPE; ++q) g[q] = G[q][0] * qx + G[q][1] * qy + G[q][2] * qzz;
        const double sc = (det > 0 ? 1.0 : -1.0) / (DIM == 3 ? 24.0 : 6.0);
        double f[NPE];
#pragma unroll
        for (int q = 0; q < NPE; ++q) f[q] = 0.;
        const double *krs = sk + slot * wmax;
#pragma unroll
        for (int j = 0; j < NED; ++j) {
            const int a = edge_a(j);
            const int b = edge_b(j);
            const double flux = sc * (g[b] - g[a]);
            const double krf = krs[(mask >> j) & 1u ? l[a] : l[b]];
            const double M = rho0 * (krf * flux);
            f[a] -= M;
            f[b] += M;
        }
#pragma unroll
        for (int q = 0; q < NPE; ++q)
            if (l[q] < nown) atomicAdd(&acc[l[q]], f[q]);
    }
    __syncthreads();
    for (int k = bptr[tile] + threadIdx.x; k < bptr[tile + 1]; k += blockDim.x) acc[bnode[k] - lo] -= bval[k];
    __syncthreads();
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        if (JV) {
            const double yp = psip[i] + jv.cj * (sig * jv.v[i]);
            const double F1 = acc[i - lo] * invV[i] - yp * cap[i];
            F[i] = jv_scaled(jv, i, (F1 - jv.F0[i]) / sig);
        } else
            F[i] = acc[i - lo] * invV[i] - psip[i] * cap[i];
    }
    __syncthreads();
    for (int k = dptr[tile] + threadIdx.x; k < dptr[tile + 1]; k += blockDim.x) {
        const int i = dnode[k];
        if (JV) {
            const double y = psi[i] + sig * jv.v[i];
            F[i] = jv_scaled(jv, i, ((dval[k] - y) - jv.F0[i]) / sig);
        } else
            F[i] = dval[k] - psi[i];
    }
}

__global__ void boundary_kernel(int nb, const int *__restrict__ bnode, const double *__restrict__ bval,
                                double *__restrict__ acc) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nb) acc[bnode[k]] -= bval[k];
}

template <bool JV = false>
__global__ void finalize_kernel(int N, const double *__restrict__ acc, const double *__restrict__ invV,
                                const double *__restrict__ psip, const double *__restrict__ cap,
                                double *__restrict__ F, JvArgs jv = JvArgs()) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    if (JV) {
        const double sig = jv.sig[0];
        const double yp = psip[i] + jv.cj * (sig * jv.v[i]);
        const double F1 = acc[i] * invV[i] - yp * cap[i];
        F[i] = jv_scaled(jv, i, (F1 - jv.F0[i]) / sig);
    } else
        F[i] = acc[i] * invV[i] - psip[i] * cap[i];
}

template <bool JV = false>
__global__ void dirichlet_kernel(int nd, const int *__restrict__ dnode, const double *__restrict__ dval,
                                 const double *__restrict__ psi, double *__restrict__ F, JvArgs jv = JvArgs()) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nd) {
        int i = dnode[k];
        if (JV) {
            const double sig = jv.sig[0];
            const double y = psi[i] + sig * jv.v[i];
            F[i] = jv_scaled(jv, i, ((dval[k] - y) - jv.F0[i]) / sig);
        } else
            F[i] = dval[k] - psi[i];
    }
}

// edge flux = sum over the edge's CV faces of q.n / sum of their areas
// (flux_lim_matrix, fvmpor.h:1033-1071; the faces in the reference's (edge,
// element) order), then the upwind test (fvmpor.h:783-794)
// A workgroup's edges own one contiguous range of slots, which its threads load
// slot by slot (whole lines, every lane in use) and stage in the LDS kEdgeChunk at a
// time; each edge then sums its own in slot order.  9 million faces, 1.79 million
// edges: 36 us; 40 with a thread gathering its own edge's faces (five of eight lanes in
// use, 42 lines a load) and writing the weights as doubles.  Bound by its bytes.
constexpr int kEdgeBatch = 8;  // loads in flight per thread
constexpr int kEdgeChunk = 256 * kEdgeBatch;
__global__ void __launch_bounds__(256) edge_flux_kernel(int NE, const int *__restrict__ slot_ptr,
                                                        const int *__restrict__ slot,
                                                        const double *__restrict__ qface,
                                                        const double *__restrict__ ea, double *__restrict__ eflux,
                                                        uint8_t *__restrict__ front) {
    __shared__ double q[kEdgeChunk];
    const int ed = blockIdx.x * 256 + threadIdx.x, last = min(NE, (int)(blockIdx.x + 1) * 256);
    const int b0 = slot_ptr[blockIdx.x * 256], b1 = slot_ptr[last];
    const int s0 = ed < NE ? slot_ptr[ed] : b1, s1 = ed < NE ? slot_ptr[ed + 1] : b1;
    const double w = ed < NE ? 1. / ea[ed] : 0.;
    double sum = 0.;
    for (int c0 = b0; c0 < b1; c0 += kEdgeChunk) {
        int sl[kEdgeBatch];
        double v[kEdgeBatch];
#pragma unroll
        for (int u = 0; u < kEdgeBatch; ++u) {
            const int k = c0 + 256 * u + threadIdx.x;
            if (k < b1) sl[u] = slot[k];
        }
#pragma unroll
        for (int u = 0; u < kEdgeBatch; ++u)
            if (c0 + 256 * u + (int)threadIdx.x < b1) v[u] = qface[sl[u]];
#pragma unroll
        for (int u = 0; u < kEdgeBatch; ++u)
            if (c0 + 256 * u + (int)threadIdx.x < b1) q[256 * u + threadIdx.x] = v[u];
        __syncthreads();
        const int k1 = min(s1, c0 + kEdgeChunk);
        for (int k = max(s0, c0); k < k1; ++k) sum += w * q[k - c0];
        __syncthreads();
    }
    if (ed >= NE) return;
    eflux[ed] = sum;
    front[ed] = sum < 0.;
}

// CV face areas |S_ab| = |e| / (d+1) |grad N_b - grad N_a| per (local edge, element)
template <int DIM>
__global__ void face_area_kernel(int T, const int4 *__restrict__ conn, const double *__restrict__ xyz,
                                 double *__restrict__ aface) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    constexpr int NPE = DIM + 1;
    constexpr int NED = DIM == 2 ? 3 : 6;
    const int4 c4 = conn[e];
    const int n[4] = {c4.x, c4.y, c4.z, c4.w};
    double px[NPE], py[NPE], pz[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) load_pt(xyz, n[k], px[k], py[k], pz[k]);
    double G[NPE][3];
    if (DIM == 3) {
        double ux = px[1] - px[0], uy = py[1] - py[0], uz = pz[1] - pz[0];
        double vx = px[2] - px[0], vy = py[2] - py[0], vz = pz[2] - pz[0];
        double wx = px[3] - px[0], wy = py[3] - py[0], wz = pz[3] - pz[0];
        G[1][0] = vy * wz - vz * wy; G[1][1] = vz * wx - vx * wz; G[1][2] = vx * wy - vy * wx;
        G[2][0] = wy * uz - wz * uy; G[2][1] = wz * ux - wx * uz; G[2][2] = wx * uy - wy * ux;
        G[3][0] = uy * vz - uz * vy; G[3][1] = uz * vx - ux * vz; G[3][2] = ux * vy - uy * vx;
    } else {
        double ux = px[1] - px[0], uy = py[1] - py[0];
        double vx = px[2] - px[0], vy = py[2] - py[0];
        G[1][0] = vy; G[1][1] = -vx; G[1][2] = 0.;
        G[2][0] = -uy; G[2][1] = ux; G[2][2] = 0.;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) G[0][d] = -(G[1][d] + G[2][d] + (DIM == 3 ? G[NPE - 1][d] : 0.));
    const double sc = 1.0 / (DIM == 3 ? 24.0 : 6.0);
#pragma unroll
    for (int j = 0; j < NED; ++j) {
        const int a = edge_a(j), b = edge_b(j);
        const double sx = G[b][0] - G[a][0], sy = G[b][1] - G[a][1], sz = G[b][2] - G[a][2];
        aface[(size_t)j * T + e] = sc * sqrt(sx * sx + sy * sy + sz * sz);
    }
}

__global__ void edge_area_kernel(int NE, const int *__restrict__ slot_ptr, const int *__restrict__ slot,
                                 const double *__restrict__ aface, double *__restrict__ ea) {
    int ed = blockIdx.x * blockDim.x + threadIdx.x;
    if (ed >= NE) return;
    double tot = 0.;
    for (int s = slot_ptr[ed]; s < slot_ptr[ed + 1]; ++s) tot += aface[slot[s]];
    ea[ed] = tot;
}

// per-element upwind bits: bit j set when the first local node of edge j is upwind
// (front: the edges' front nodes as bytes, so that neighbouring edges share the
// lines that the elements gather; 1 500 000 elements: 11 us, 13 from the weights)
template <int DIM>
__global__ void mask_kernel(int T, const int *__restrict__ eedge, const uint8_t *__restrict__ eorient,
                            const uint8_t *__restrict__ front, uint8_t *__restrict__ emask) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    constexpr int NED = DIM == 2 ? 3 : 6;
    unsigned o = eorient[e], m = 0;
#pragma unroll
    for (int j = 0; j < NED; ++j) {
        bool front_up = front[eedge[(size_t)j * T + e]];
        bool a_front = (o >> j) & 1u;
        if (front_up == a_front) m |= 1u << j;
    }
    emask[e] = (uint8_t)m;
}

static inline int blocks(long n, int bs) { return (int)((n + bs - 1) / bs); }

template <bool JV>
static void launch_vg(fvp_ctx *c, const double *psi, const JvArgs &jv, double *nrec) {
    vg_kernel<JV><<<blocks(c->nmz, 256) + blocks(c->N, 256), 256, 0, c->stream>>>(
        c->N, c->nmz, c->mznode.p, c->zt, c->rho0, psi, c->zmask.p, c->zw.p, c->kr.p, c->cap.p, jv, nrec);
}

// Dynamic LDS of owner_lds for windows of wmax nodes with up to nr zones per node
// (0: not used): the records have to fit the elements' 14 + 2 bits and half of the LDS
// (two workgroups per CU).
size_t owner_window_lds(int dim, int wmax, int nr) {
    const long recs = (long)wmax * win_stride(dim, nr);
    const size_t bytes = sizeof(double) * recs + 2 * (size_t)((wmax + 3) & ~3);
    return nr <= kRecRanks && recs <= 1 << kRecBits && bytes <= kOwnerLdsMax ? bytes : 0;
}
int owner_window_code(int dim, int nr, int local, int rank) { return local * win_stride(dim, nr) | (rank << kRecBits); }

// Allow the tile kernel's dynamic LDS beyond the default limit; fails cleanly if
// the device cannot provide it.
int tile_kernel_attrs(fvp_ctx *c) {
    int lds_max = 0;
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device) != hipSuccess)
        lds_max = 64 * 1024;
    // the static zone table shares the workgroup's LDS with the dynamic window
    const size_t static_lds = sizeof(double) * 3 * kMaxZones;
    if (c->tile_lds + static_lds > (size_t)lds_max) {
        set_error("residual tile window needs " + std::to_string(c->tile_lds) + " B of LDS, device allows " +
                  std::to_string(lds_max));
        return -1;
    }
    // the attribute is per kernel, not per context: allow the device maximum so
    // that contexts with different windows can coexist
    const int dyn = lds_max - (int)static_lds;
    FVP_HIP(hipFuncSetAttribute((const void *)tile_lds_kernel<3, false>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn));
    FVP_HIP(hipFuncSetAttribute((const void *)tile_lds_kernel<2, false>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn));
    FVP_HIP(hipFuncSetAttribute((const void *)tile_lds_kernel<3, true>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn));
    FVP_HIP(hipFuncSetAttribute((const void *)tile_lds_kernel<2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, dyn));
    for (const void *f : {(const void *)owner_lds<2, false, false, 256>, (const void *)owner_lds<2, false, true, 256>,
                          (const void *)owner_lds<2, true, false, 256>, (const void *)owner_lds<2, true, true, 256>,
                          (const void *)owner_lds<3, false, false, 256>, (const void *)owner_lds<3, false, true, 256>,
                          (const void *)owner_lds<3, true, false, 256>, (const void *)owner_lds<3, true, true, 256>,
                          (const void *)owner_lds<2, false, false, 512>, (const void *)owner_lds<2, false, true, 512>,
                          (const void *)owner_lds<2, true, false, 512>, (const void *)owner_lds<2, true, true, 512>,
                          (const void *)owner_lds<3, false, false, 512>, (const void *)owner_lds<3, false, true, 512>,
                          (const void *)owner_lds<3, true, false, 512>, (const void *)owner_lds<3, true, true, 512>})
        FVP_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max - kOwnerStaticLds));
    return 0;
}

template <int DIM, bool JV>
static void launch_owner_lds(fvp_ctx *c, const double *psi, const double *psip, double *F, const JvArgs &jv) {
    const int per = (c->ntiles + 7) / 8;
    hipStream_t s = c->stream;
    hipEvent_t ea, eb;
    prof_pair(c, JV ? 3 : 0, &ea, &eb);
    // 512 threads (31 000 nodes in tiles of 128: 15.7 us against 16.8 with 256; 1 024 000
    // in tiles of 256: 106 against 122), 256 for the smallest tiles
    const int threads = c->tile_nodes >= 128 ? 512 : 256;
    const auto kernel = threads == 512 ? (c->owner_vg ? owner_lds<DIM, JV, true, 512> : owner_lds<DIM, JV, false, 512>)
                                       : (c->owner_vg ? owner_lds<DIM, JV, true, 256> : owner_lds<DIM, JV, false, 256>);
    hipExtLaunchKernelGGL(kernel, dim3(c->xcd_map ? per * 8 : c->ntiles), dim3(threads), c->tile_lds, s, ea,
                          eb, 0, c->N, c->ntiles, c->tile_nodes, c->xcd_map ? per : 0, c->win_max, c->ntz_max, c->zt,
                          c->rho0, (const uint8_t *)c->ezone.p, (const double *)c->kmul.p,
                          (const uint8_t *)c->emask.p, (const ushort4 *)c->t_lconn.p, (const double *)c->xyz.p, psi,
                          (const uint8_t *)c->zmask.p, (const double *)c->zw.p, (const double *)c->kr.p,
                          (const int *)c->t_eptr.p, (const int *)c->t_wptr.p, (const int *)c->t_whalo.p, (const int *)c->x_ilist.p, c->xf.p,
                          (const int *)c->x_iptr.p, (const int *)c->t_bptr.p, (const int *)c->bnode.p,
                          (const double *)c->bval.p, (const double *)c->invV.p, psip, c->cap.p, c->acc.p, F, jv);
    if (c->nimp)
        owner_imports<JV><<<blocks(c->nimp, 256), 256, 0, s>>>(c->nimp, c->x_inode.p, c->acc.p, c->x_iptr.p, c->xf.p,
                                                               c->invV.p, psip, c->cap.p, F, jv);
    if (c->ndir)
        dirichlet_kernel<JV><<<blocks(c->ndir, 256), 256, 0, s>>>(c->ndir, c->dnode.p, c->dval.p, psi, F, jv);
}

template <int DIM, bool JV>
static void launch_tile(fvp_ctx *c, const double *psi, const double *psip, double *F, const JvArgs &jv) {
    const int per = (c->ntiles + 7) / 8;  // tiles per XCD: consecutive tiles share an XCD's L2
    hipStream_t s = c->stream;
    if (c->owner_win) {
        // the tiles read their halo's psi and v while others write F: a result in place
        // of either goes through a work vector
        auto meets = [&](const double *p) { return p && F < p + c->N && p < F + c->N; };
        const bool in_place = meets(psi) || meets(jv.v);
        launch_owner_lds<DIM, JV>(c, psi, psip, in_place ? c->tmp1.p : F, jv);
        if (in_place) (void)hipMemcpyAsync(F, c->tmp1.p, sizeof(double) * c->N, hipMemcpyDeviceToDevice, s);
        return;
    }
    if (c->rvariant == FVP_RESIDUAL_OWNER) {
        const int N = c->N;
        // one workgroup per tile, wide enough that large tiles still fill the CUs; when
        // profiling, the events are part of the dispatch (the kernel's own duration)
        const int threads = c->tile_nodes >= 1024 ? 512 : 256;
        hipEvent_t ea, eb;
        prof_pair(c, JV ? 3 : 0, &ea, &eb);
        hipExtLaunchKernelGGL(owner_kernel<DIM, JV>, dim3(c->xcd_map ? per * 8 : c->ntiles), dim3(threads),
                              sizeof(double) * c->tile_nodes, s, ea, eb, 0, N, c->ntiles, c->tile_nodes,
                              c->xcd_map ? per : 0, c->zt, c->rho0, (const int4 *)c->conn.p,
                              (const uint8_t *)c->ezone.p, (const double *)c->kmul.p, (const uint8_t *)c->emask.p,
                              (const double *)c->xyz.p, (const double *)c->nrec.p,
                              (const double *)c->kr.p, (const int *)c->t_eptr.p,
                              (const int *)c->t_bptr.p, (const int *)c->bnode.p, (const double *)c->bval.p,
                              (const unsigned short *)c->t_xoff.p, (const int *)c->t_xptr.p,
                              (const int *)c->x_ilist.p, c->xf.p, c->acc.p, jv);
        owner_finalize<JV><<<c->ntiles, 1024, sizeof(double) * c->tile_nodes, s>>>(
            N, c->ntiles, c->tile_nodes, c->acc.p, c->x_iptr.p, c->x_tgt.p, c->xf.p, c->invV.p, psi, psip, c->cap.p,
            c->t_dptr.p, c->dnode.p, c->dval.p, F, jv);
        return;
    }
    hipEvent_t ea, eb;
    prof_pair(c, JV ? 3 : 0, &ea, &eb);
    if (ea) (void)hipEventRecord(ea, s);
    tile_lds_kernel<DIM, JV><<<c->xcd_map ? per * 8 : c->ntiles, 256, c->tile_lds, c->stream>>>(
        c->N, c->ntiles, c->tile_nodes, c->xcd_map ? per : 0, c->win_max, c->ntz_max, c->zt, c->rho0, c->ezone.p, c->kmul.p, c->emask.p, c->xyz.p,
        psi, c->kr.p, c->t_eptr.p, c->t_hptr.p, c->t_hlist.p, c->t_wptr.p, c->t_whalo.p, c->t_vptr.p,
        (const ushort4 *)c->t_lconn.p, c->t_tz.p, c->invV.p, psip, c->cap.p, c->t_bptr.p, c->bnode.p, c->bval.p,
        c->t_dptr.p, c->dnode.p, c->dval.p, F, jv);
    if (eb) (void)hipEventRecord(eb, s);
}

// The node side of the element-local Jacobian, one pass: the increment of each node
// (IDA's), k_r and capacity at the base state and with the node moved by its
// increment, and what the elements gather of them: per zone and node one 16-byte
// record, {V^-1, k_r, k_r moved, dk_r / shift} in FP32 or the two k_r in FP64; the
// diagonal's capacity term -psi' a_hh(psi) moved with psi_i and psi'_i + c_j shift_i.
// Nodes of several zones come first, from the list, as in vg_kernel.  Bound by FP64
// instructions (two evaluations per node and zone) and the latency around them: a
// workgroup's own list behind a barrier, and inputs loaded once the zones were known,
// took 19 us on 141 000 nodes, this 13; five launches (increments, base, sum, moved,
// capacity term) took 42, and the elements' four 8-byte gathers per node become one of 16.
template <typename C>
__global__ void __launch_bounds__(256) fd_nodes(int N, int nmz, const int *__restrict__ mznode, ZoneTable zt,
                                                double rho0, FdJacobian fd, const uint8_t *__restrict__ zmask,
                                                const double *__restrict__ zw, const double *__restrict__ invV,
                                                double *__restrict__ kr, double *__restrict__ cap,
                                                double *__restrict__ nrec) {
    __shared__ double zp[kMaxZones * 10];
    if (threadIdx.x < 10 * zt.nz) zp[threadIdx.x] = zt.p[threadIdx.x / 10][threadIdx.x % 10];
    const int mzb = (nmz + 255) / 256;
    const bool several = (int)blockIdx.x < mzb;
    int g = ((int)blockIdx.x - (several ? 0 : mzb)) * 256 + threadIdx.x;
    const bool live = g < (several ? nmz : N);
    if (several) g = live ? mznode[g] : 0;
    else if (!live) g = 0;
    const unsigned m = zmask[g];
    const double y = fd.psi[g], yp = fd.psip[g], ew = fd.ewt[g], iv = invV[g];
    __syncthreads();
    if (!live || (!several && (m & (m - 1)))) return;
    const double sh = fd.eps * fmax(fabs(y), fmax(fabs(fd.h * yp), 1.0 / ew));
    const float w = (float)iv;
    double one = 0.;
    const double c0 = vg_node<true>(N, g, y, m, zp, zw, rho0, [&](int z, int, double k) {
        one = k;
        if (several) kr[(size_t)z * N + g] = k;
    });
    const double c1 = vg_node<true>(N, g, y + sh, m, zp, zw, rho0, [&](int z, int, double k1) {
        const double k0 = several ? kr[(size_t)z * N + g] : one;
        if constexpr (sizeof(C) == 4)
            reinterpret_cast<float4 *>(fd.rec)[(size_t)z * N + g] = make_float4(w, (float)k0, (float)k1, (float)((k1 - k0) / sh));
        else
            reinterpret_cast<double2 *>(fd.rec)[(size_t)z * N + g] = make_double2(k0, k1);
    });
    cap[g] = c0;
    fd.dterm[g] = ((yp + fd.cj * sh) * c1 - yp * c0) / sh;
    fd.shift[g] = sh;
    nrec[4 * (size_t)g + 3] = y;
}

// node values of an element from the packed records (x, y, z, head: two 16-byte loads)
template <int DIM>
__device__ __forceinline__ void load_geometry(const ElemRec &rec, const double *__restrict__ nrec,
                                              NodeVals<DIM> &nv) {
    const int n[4] = {rec.c4.x, rec.c4.y, rec.c4.z, rec.c4.w};
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) {
        const double2 *r = reinterpret_cast<const double2 *>(nrec + 4 * (size_t)n[k]);
        const double2 a = r[0], b = r[1];
        nv.px[k] = a.x; nv.py[k] = a.y; nv.pz[k] = b.x; nv.h[k] = b.y;
    }
}

// Element-local finite-difference Jacobian, -(dF/dpsi + c_j dF/dpsi') with
// the coloured method's increments (shift) and upwind bits: every element is
// evaluated at the base state and once per node with that node's head moved
// by its shift (k_r from the second van Genuchten pass, kr2), and
// (f_base - f_moved) V^-1 / shift for (row node i, moved node k) is stored at
// contrib[4 (npe e + i) + k], an element's quotients in one piece; fd_gather
// sums each entry's (in a fixed order without atomics, so the Jacobian is
// repeatable bit for bit) and adds fd_nodes' capacity term to the diagonal.  The
// Dirichlet rows are set by fd_dirichlet.  The residual is a sum of element terms, so these are the
// coloured quotients up to the rounding of the sums.
template <int DIM>
__global__ void __launch_bounds__(256) fd_elem_kernel(int T, int N, ZoneTable zt, double rho0,
                                                      const int4 *__restrict__ conn, const uint8_t *__restrict__ ezone,
                                                      const double *__restrict__ kmul, const uint8_t *__restrict__ emask,
                                                      const double *__restrict__ nrec, const double2 *__restrict__ kk,
                                                      const double *__restrict__ shift,
                                                      const double *__restrict__ invV,
                                                      double2 *__restrict__ contrib) {
    __shared__ double zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    const ElemRec rec = load_elem<0>(e, conn, ezone, kmul, emask, nullptr);
    NodeVals<DIM> nv;
    load_geometry<DIM>(rec, nrec, nv);
    int n[4] = {rec.c4.x, rec.c4.y, rec.c4.z, rec.c4.w};
    double w[DIM + 1], sh[DIM + 1], km[DIM + 1], d[DIM + 1][4];
#pragma unroll
    for (int i = 0; i < DIM + 1; ++i) {
        const double2 k2 = kk[(size_t)rec.z * N + n[i]];
        nv.k[i] = k2.x;
        km[i] = k2.y;
        w[i] = invV[n[i]];
        sh[i] = shift[n[i]];
        d[i][3] = 0.;
    }
    double f0[4];
    element_fluxes_vals<DIM, 0>(e, rec, nv, zk, rho0, nullptr, n, f0);
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) {
        const double sk = sh[k], hk = nv.h[k], k0 = nv.k[k];
        nv.h[k] = hk + sk;
        nv.k[k] = km[k];
        int n1[4];
        double f1[4];
        element_fluxes_vals<DIM, 0>(e, rec, nv, zk, rho0, nullptr, n1, f1);
        nv.h[k] = hk;
        nv.k[k] = k0;
#pragma unroll
        for (int i = 0; i < DIM + 1; ++i) d[i][k] = (f0[i] - f1[i]) * w[i] / sk;
    }
    double2 *const out = contrib + 2 * (DIM + 1) * (size_t)e;
#pragma unroll
    for (int i = 0; i < DIM + 1; ++i) {
        out[2 * i] = make_double2(d[i][0], d[i][1]);
        out[2 * i + 1] = make_double2(d[i][2], d[i][3]);
    }
}

// The same element-local quotients in FP32 arithmetic (the FP32
// preconditioner's input).  For a fixed k_r a face flux is linear in the
// heads, so with node k moved by s_k the difference quotient of the face's
// mass flow M = rho0 k_r flux is, exactly,
//   (M1 - M0) / s_k = rho0 [ (k_r1 - k_r0) / s_k * flux + k_r1 * dflux/dh_k ],
// k_r1 differing from k_r0 only when node k is the face's upwind node.  Each
// term is formed directly (dflux/dh_k from the adjugate, (k_r1 - k_r0) / s_k
// in FP64 from the two van Genuchten passes), so nothing cancels and FP32
// carries the quotient to its rounding; the geometry is built once per
// element, relative to its first node.  Same increments, same upwind bits,
// same places as fd_elem_kernel.  787 000 elements: 27 us; scattering the 16
// quotients to their entries, one 4-byte store each, took 67 (bound by the L2's
// requests).
template <int DIM>
__global__ void __launch_bounds__(256) fd_elem_kernel32(int T, int N, ZoneTable zt, double rho0,
                                                        const int4 *__restrict__ conn,
                                                        const uint8_t *__restrict__ ezone,
                                                        const double *__restrict__ kmul,
                                                        const uint8_t *__restrict__ emask,
                                                        const double *__restrict__ nrec, const float4 *__restrict__ kk,
                                                        float4 *__restrict__ contrib) {
    constexpr int NPE = DIM + 1;
    constexpr int NED = DIM == 2 ? 3 : 6;
    __shared__ float zk[3 * kMaxZones];
    if (threadIdx.x < 3 * zt.nz) zk[threadIdx.x] = (float)zt.p[threadIdx.x / 3][ZK_X + threadIdx.x % 3];
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= T) return;
    const ElemRec rec = load_elem<0>(e, conn, ezone, kmul, emask, nullptr);
    NodeVals<DIM> nv;
    load_geometry<DIM>(rec, nrec, nv);
    const int n[4] = {rec.c4.x, rec.c4.y, rec.c4.z, rec.c4.w};
    float w[NPE], kb[NPE], km1[NPE], dkr[NPE];
#pragma unroll
    for (int i = 0; i < NPE; ++i) {
        const float4 q = kk[(size_t)rec.z * N + n[i]];
        w[i] = q.x; kb[i] = q.y; km1[i] = q.z; dkr[i] = q.w;
    }
    float G[NPE][3], det;
    if (DIM == 3) {
        const float ux = (float)(nv.px[1] - nv.px[0]), uy = (float)(nv.py[1] - nv.py[0]), uz = (float)(nv.pz[1] - nv.pz[0]);
        const float vx = (float)(nv.px[2] - nv.px[0]), vy = (float)(nv.py[2] - nv.py[0]), vz = (float)(nv.pz[2] - nv.pz[0]);
        const float wx = (float)(nv.px[3] - nv.px[0]), wy = (float)(nv.py[3] - nv.py[0]), wz = (float)(nv.pz[3] - nv.pz[0]);
        G[1][0] = vy * wz - vz * wy; G[1][1] = vz * wx - vx * wz; G[1][2] = vx * wy - vy * wx;
        G[2][0] = wy * uz - wz * uy; G[2][1] = wz * ux - wx * uz; G[2][2] = wx * uy - wy * ux;
        G[3][0] = uy * vz - uz * vy; G[3][1] = uz * vx - ux * vz; G[3][2] = ux * vy - uy * vx;
        det = ux * G[1][0] + uy * G[1][1] + uz * G[1][2];
    } else {
        const float ux = (float)(nv.px[1] - nv.px[0]), uy = (float)(nv.py[1] - nv.py[0]);
        const float vx = (float)(nv.px[2] - nv.px[0]), vy = (float)(nv.py[2] - nv.py[0]);
        G[1][0] = vy; G[1][1] = -vx; G[1][2] = 0.f;
        G[2][0] = -uy; G[2][1] = ux; G[2][2] = 0.f;
        det = ux * vy - uy * vx;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) G[0][d] = -(G[1][d] + G[2][d] + (DIM == 3 ? G[NPE - 1][d] : 0.f));
    const float inv = 1.f / det;
    const float km = (float)rec.km;
    const float Kx = -(zk[3 * rec.z] * km), Ky = -(zk[3 * rec.z + 1] * km), Kz = -(zk[3 * rec.z + 2] * km);
    // base state: head gradient, Darcy flux without k_r, face fluxes
    float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
    for (int k = 1; k < NPE; ++k) {
        const float dh = (float)(nv.h[k] - nv.h[0]);
        gx += dh * G[k][0]; gy += dh * G[k][1]; gz += dh * G[k][2];
    }
    gx *= inv; gy *= inv; gz *= inv;
    float qx = gx * Kx, qy, qz;
    if (DIM == 2) { qy = (gy + 1.f) * Ky; qz = 0.f; }
    else { qy = gy * Ky; qz = (gz + 1.f) * Kz; }
    float g[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) g[k] = G[k][0] * qx + G[k][1] * qy + G[k][2] * qz;
    const float sc = (det > 0.f ? 1.f : -1.f) / (DIM == 3 ? 24.f : 6.f);
    const float r0 = (float)rho0;
    float out[NPE][4];
#pragma unroll
    for (int i = 0; i < NPE; ++i) out[i][3] = 0.f;
#pragma unroll
    for (int k = 0; k < NPE; ++k) {
        // d(grad h)/dh_k = G[k] / det, so dq/dh_k = K (G[k] / det) (no gravity term)
        const float dqx = G[k][0] * inv * Kx, dqy = G[k][1] * inv * Ky, dqz = G[k][2] * inv * Kz;
        float dg[NPE];
#pragma unroll
        for (int m = 0; m < NPE; ++m) dg[m] = G[m][0] * dqx + G[m][1] * dqy + G[m][2] * dqz;
        float d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NED; ++j) {
            const int a = edge_a(j), b = edge_b(j);
            const unsigned up_a = (rec.mask >> j) & 1u;  // 1: node a is upwind
            const int u = up_a ? a : b;
            const float flux = sc * (g[b] - g[a]);
            const float dflux = sc * (dg[b] - dg[a]);
            const float kr1 = u == k ? km1[k] : (up_a ? kb[a] : kb[b]);
            const float dM = r0 * ((u == k ? dkr[k] : 0.f) * flux + kr1 * dflux);
            d[a] += dM;  // (f0 - f1) / s_k at a: f[a] -= M
            d[b] -= dM;
        }
#pragma unroll
        for (int i = 0; i < NPE; ++i) out[i][k] = d[i] * w[i];
    }
#pragma unroll
    for (int i = 0; i < NPE; ++i)
        contrib[NPE * (size_t)e + i] = make_float4(out[i][0], out[i][1], out[i][2], out[i][3]);
}

// The entries of a block of rows: per entry the sum of its quotients, accumulated in
// FP64 in a fixed order, the capacity term added on the diagonal.  A row's quotients
// lie four to an element (its visit); the block's visits are staged in the LDS with
// 16- or 32-byte loads, which both the requests and the lines are few for, and the
// entries pick their 2-byte codes (visit, place) there.  Diagonals have a quotient of
// every visit, so kDiagLanes lanes share one.  Without STAGED (more visits than the
// LDS holds) the codes are places in contrib.  787 000 elements, 2 million entries,
// FP32: 37 us (46 with 256 threads and no loads ahead of the barrier); bound by the
// latency of its chain of loads (entry, code; visit, quotients) and then the bytes.
constexpr int kFdThreads = 512;
constexpr int kDiagLanes = 8;  // x 64 rows
template <typename C, bool STAGED>
__global__ void __launch_bounds__(kFdThreads) fd_gather(int N, FdJacobian fd) {
    using V = std::conditional_t<sizeof(C) == 4, float4, double4>;
    extern __shared__ __align__(16) char fd_lds[];
    constexpr unsigned kDiag = 1u << 31;
    const V *const contrib = reinterpret_cast<const V *>(fd.contrib);
    const C *const q = STAGED ? reinterpret_cast<const C *>(fd_lds) : reinterpret_cast<const C *>(fd.contrib);
    const int r0 = blockIdx.x * fd.rows, r1 = min(N, r0 + fd.rows), p1 = fd.ia[r1];
    // an entry's codes [k0, k1), every step-th from k0 + l; the first kEdgeBatch of them
    struct Codes {
        unsigned k0, k1;
        int at[kEdgeBatch];
    };
    auto place = [&](unsigned k) { return STAGED ? (int)fd.code[k] : fd.code32[k]; };
    auto fetch = [&](int p, unsigned l, unsigned step, Codes &e) {
        e.k0 = fd.cptr[p];
        e.k1 = fd.cptr[p + 1] & ~kDiag;
        const unsigned k = (e.k0 & ~kDiag) + l;
#pragma unroll
        for (int u = 0; u < kEdgeBatch; ++u) e.at[u] = place(min(k + u * step, e.k1 - 1));
    };
    auto sum = [&](const Codes &e, unsigned l, unsigned step) {
        double s = 0.;
        unsigned k = (e.k0 & ~kDiag) + l;
        int at[kEdgeBatch];
#pragma unroll
        for (int u = 0; u < kEdgeBatch; ++u) at[u] = e.at[u];
        while (k < e.k1) {
            C c[kEdgeBatch];
#pragma unroll
            for (int u = 0; u < kEdgeBatch; ++u) c[u] = q[at[u]];
#pragma unroll
            for (int u = 0; u < kEdgeBatch; ++u)
                if (k + u * step < e.k1) s += (double)c[u];
            k += kEdgeBatch * step;
            if (k >= e.k1) break;
#pragma unroll
            for (int u = 0; u < kEdgeBatch; ++u) at[u] = place(min(k + u * step, e.k1 - 1));
        }
        return s;
    };
    int p = fd.ia[r0] + threadIdx.x;
    const int r = r0 + threadIdx.x / kDiagLanes, pd = fd.dpos[min(r, r1 - 1)], l = threadIdx.x % kDiagLanes;
    Codes e{}, d;
    if (p < p1) fetch(p, 0, 1, e);
    fetch(pd, l, kDiagLanes, d);
    if (STAGED) {
        const int v0 = fd.vptr[blockIdx.x], nv = fd.vptr[blockIdx.x + 1] - v0;
        constexpr int kU = 4;
        for (int k0 = threadIdx.x; k0 < nv; k0 += kFdThreads * kU) {
            int at[kU];
            V c[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) at[u] = fd.visit[v0 + min(k0 + kFdThreads * u, nv - 1)];
#pragma unroll
            for (int u = 0; u < kU; ++u) c[u] = contrib[at[u]];
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (k0 + kFdThreads * u < nv) reinterpret_cast<V *>(fd_lds)[k0 + kFdThreads * u] = c[u];
        }
        __syncthreads();
    }
    double s = sum(d, l, kDiagLanes);
#pragma unroll
    for (int m = 1; m < kDiagLanes; m *= 2) s += __shfl_xor(s, m, 64);
    if (l == 0 && r < r1) fd.J[pd] = s + fd.dterm[r];
    while (p < p1) {
        Codes n{};
        if (p + kFdThreads < p1) fetch(p + kFdThreads, 0, 1, n);
        if (!(e.k0 & kDiag)) fd.J[p] = sum(e, 0, 1);
        e = n;
        p += kFdThreads;
    }
}

// Dirichlet rows F = psi_D - psi: zero off the diagonal, the quotient on it
__global__ void fd_dirichlet(int nd, const int *__restrict__ dnode, const double *__restrict__ dval,
                             const double *__restrict__ psi, const double *__restrict__ shift,
                             const int *__restrict__ ia, const int *__restrict__ dpos, double *__restrict__ J) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nd) return;
    const int i = dnode[k];
    for (int p = ia[i]; p < ia[i + 1]; ++p) J[p] = 0.;
    J[dpos[i]] = ((dval[k] - psi[i]) - (dval[k] - (psi[i] + shift[i]))) / shift[i];
}

template <typename C>
static void fd_launch(fvp_ctx *c, const FdJacobian &fd) {
    hipStream_t s = c->stream;
    const int N = c->N, T = c->T;
    fd_nodes<C><<<blocks(c->nmz, 256) + blocks(N, 256), 256, 0, s>>>(N, c->nmz, c->mznode.p, c->zt, c->rho0, fd,
                                                                    c->zmask.p, c->zw.p, c->invV.p, c->kr.p, c->cap.p,
                                                                    c->nrec.p);
    const int4 *conn = (const int4 *)c->conn.p;
    const uint8_t *ezone = c->ezone.p, *emask = c->emask.p;
    if constexpr (sizeof(C) == 4) {
        const auto elem = c->dim == 3 ? fd_elem_kernel32<3> : fd_elem_kernel32<2>;
        elem<<<blocks(T, 256), 256, 0, s>>>(T, N, c->zt, c->rho0, conn, ezone, c->kmul.p, emask, c->nrec.p,
                                            (const float4 *)fd.rec, (float4 *)fd.contrib);
    } else {
        const auto elem = c->dim == 3 ? fd_elem_kernel<3> : fd_elem_kernel<2>;
        elem<<<blocks(T, 256), 256, 0, s>>>(T, N, c->zt, c->rho0, conn, ezone, c->kmul.p, emask, c->nrec.p,
                                            (const double2 *)fd.rec, fd.shift, c->invV.p, (double2 *)fd.contrib);
    }
    if (fd.code)
        fd_gather<C, true><<<blocks(N, fd.rows), kFdThreads, 4 * sizeof(C) * (size_t)fd.max_visits, s>>>(N, fd);
    else
        fd_gather<C, false><<<blocks(N, fd.rows), kFdThreads, 0, s>>>(N, fd);
    if (c->ndir)
        fd_dirichlet<<<blocks(c->ndir, 256), 256, 0, s>>>(c->ndir, c->dnode.p, c->dval.p, fd.psi, fd.shift, fd.ia,
                                                          fd.dpos, fd.J);
}

int fd_jacobian_elem(fvp_ctx *c, const FdJacobian &fd, bool fp32) {
    if (fp32) fd_launch<float>(c, fd);
    else fd_launch<double>(c, fd);
    FVP_HIP(hipGetLastError());
    return 0;
}

int residual_impl(fvp_ctx *c, double t, const double *psi, const double *psip, double *F, int averaging,
                  const JvArgs *jv) {
    (void)t;
    hipStream_t s = c->stream;
    const int N = c->N, T = c->T;
    if (jv && averaging) {
        set_error("internal: fused J v needs the upwinded residual");
        return -1;
    }
    ++c->nres;
    prof_mark(c, 1, 0);
    const bool fused = c->owner_win && c->owner_vg && !averaging;  // the element kernel does the van Genuchten pass
    double *const nrec = c->rvariant == FVP_RESIDUAL_OWNER && !c->owner_win ? c->nrec.p : nullptr;
    if (jv && !fused)
        launch_vg<true>(c, psi, *jv, nrec);
    else if (!fused)
        launch_vg<false>(c, psi, JvArgs(), nrec);
    if (!averaging) {
        // tiled paths (element fluxes with the boundary fluxes, then the finalisation)
        const JvArgs none;
        if (c->dim == 3) {
            if (jv) launch_tile<3, true>(c, psi, psip, F, *jv);
            else launch_tile<3, false>(c, psi, psip, F, none);
        } else {
            if (jv) launch_tile<2, true>(c, psi, psip, F, *jv);
            else launch_tile<2, false>(c, psi, psip, F, none);
        }
    } else {
        FVP_HIP(hipMemsetAsync(c->acc.p, 0, sizeof(double) * N, s));
        if (c->dim == 3)
            elem_kernel<3><<<blocks(T, 256), 256, 0, s>>>(T, N, c->zt, c->rho0, c->conn.p, c->ezone.p, c->kmul.p,
                                                           c->emask.p, c->eorient.p, c->xyz.p, psi, c->kr.p,
                                                           c->acc.p);
        else
            elem_kernel<2><<<blocks(T, 256), 256, 0, s>>>(T, N, c->zt, c->rho0, c->conn.p, c->ezone.p, c->kmul.p,
                                                           c->emask.p, c->eorient.p, c->xyz.p, psi, c->kr.p,
                                                           c->acc.p);
        if (c->nb) boundary_kernel<<<blocks(c->nb, 256), 256, 0, s>>>(c->nb, c->bnode.p, c->bval.p, c->acc.p);
        finalize_kernel<<<blocks(N, 256), 256, 0, s>>>(N, c->acc.p, c->invV.p, psip, c->cap.p, F);
        if (c->ndir) dirichlet_kernel<<<blocks(c->ndir, 256), 256, 0, s>>>(c->ndir, c->dnode.p, c->dval.p, psi, F);
    }
    prof_mark(c, 1, 1);
    FVP_HIP(hipGetLastError());
    return 0;
}

// Set-up: summed CV face area of every edge (geometry only)
int edge_areas(fvp_ctx *c) {
    DevBuf<double> aface;
    if (aface.alloc((size_t)c->T * c->ned)) return -1;
    if (c->dim == 3) face_area_kernel<3><<<blocks(c->T, 256), 256, 0, c->stream>>>(c->T, c->conn.p, c->xyz.p, aface.p);
    else face_area_kernel<2><<<blocks(c->T, 256), 256, 0, c->stream>>>(c->T, c->conn.p, c->xyz.p, aface.p);
    edge_area_kernel<<<blocks(c->NE, 256), 256, 0, c->stream>>>(c->NE, c->slot_ptr.p, c->slot.p, aface.p, c->ea.p);
    FVP_HIP(hipGetLastError());
    FVP_HIP(hipStreamSynchronize(c->stream));
    aface.release();
    return 0;
}

// Event pairs are pooled per kind and folded into running totals every 4096 pairs.
static void prof_fold(fvp_ctx *c, int k) {
    if (!c->prof_used[k]) return;
    (void)hipStreamSynchronize(c->stream);
    for (size_t i = 0; i < c->prof_used[k]; ++i) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, c->prof_ev[k][i].first, c->prof_ev[k][i].second) == hipSuccess) {
            c->prof_ms[k] += ms;
            c->prof_n[k] += 1;
        }
    }
    c->prof_used[k] = 0;
}

void prof_mark(fvp_ctx *c, int k, int stop) {
    if (!c->prof) return;
    if (!stop) {
        if (c->prof_used[k] == 4096) prof_fold(c, k);
        if (c->prof_used[k] == c->prof_ev[k].size()) {
            hipEvent_t a, b;
            if (hipEventCreateWithFlags(&a, hipEventDisableSystemFence) != hipSuccess) return;
            if (hipEventCreateWithFlags(&b, hipEventDisableSystemFence) != hipSuccess) { (void)hipEventDestroy(a); return; }
            c->prof_ev[k].push_back({a, b});
        }
        (void)hipEventRecord(c->prof_ev[k][c->prof_used[k]].first, c->stream);
    } else {
        (void)hipEventRecord(c->prof_ev[k][c->prof_used[k]].second, c->stream);
        ++c->prof_used[k];
    }
}

// a start / stop event pair of kind k for one launch (both null when not profiling)
void prof_pair(fvp_ctx *c, int k, hipEvent_t *a, hipEvent_t *b) {
    *a = *b = nullptr;
    if (!c->prof) return;
    if (c->prof_used[k] == 4096) prof_fold(c, k);
    if (c->prof_used[k] == c->prof_ev[k].size()) {
        hipEvent_t e0, e1;
        if (hipEventCreateWithFlags(&e0, hipEventDisableSystemFence) != hipSuccess) return;
        if (hipEventCreateWithFlags(&e1, hipEventDisableSystemFence) != hipSuccess) { (void)hipEventDestroy(e0); return; }
        c->prof_ev[k].push_back({e0, e1});
    }
    *a = c->prof_ev[k][c->prof_used[k]].first;
    *b = c->prof_ev[k][c->prof_used[k]].second;
    ++c->prof_used[k];
}

void prof_release(fvp_ctx *c) {
    for (int k = 0; k < kProfKinds; ++k) {
        for (auto &e : c->prof_ev[k]) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
        c->prof_ev[k].clear();
        c->prof_used[k] = 0;
    }
}

}  // namespace fvp

using namespace fvp;

extern "C" int fvp_residual(fvp_ctx *c, double t, const double *psi, const double *psip, double *F) {
    if (!c || !psi || !psip || !F) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    return residual_impl(c, t, psi, psip, F, c->averaging);
}

static void launch_mask(fvp_ctx *c) {
    const auto mask = c->dim == 3 ? mask_kernel<3> : mask_kernel<2>;
    mask<<<blocks(c->T, 256), 256, 0, c->stream>>>(c->T, c->eedge.p, c->eorient.p, c->front.p, c->emask.p);
}

extern "C" int fvp_begin_step(fvp_ctx *c, double t, const double *psi, const double *psip) {
    if (!c || !psi || !psip) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    (void)t; (void)psip;
    const int N = c->N, T = c->T;
    // k_r at the state, then the averaged-weight face fluxes summed per edge
    launch_vg<false>(c, psi, JvArgs(), c->nrec.p);
    const auto faces = c->dim == 3 ? face_flux_kernel<3> : face_flux_kernel<2>;
    faces<<<blocks(T, 256), 256, 0, s>>>(T, N, c->zt, c->conn.p, c->ezone.p, c->kmul.p, c->eorient.p, c->nrec.p,
                                         c->kr.p, c->qface.p);
    edge_flux_kernel<<<blocks(c->NE, 256), 256, 0, s>>>(c->NE, c->slot_ptr.p, c->slot.p, c->qface.p, c->ea.p,
                                                        c->eflux.p, c->front.p);
    launch_mask(c);
    FVP_HIP(hipGetLastError());
    c->averaging = 0;
    return 0;
}

extern "C" int fvp_get_upwind(fvp_ctx *c, double *w_front, double *edge_flux) {
    if (!c) { set_error("null context"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    FVP_HIP(hipStreamSynchronize(c->stream));
    if (w_front && c->averaging) {
        std::fill(w_front, w_front + c->NE, 0.5);
    } else if (w_front) {
        std::vector<uint8_t> front(c->NE);
        FVP_HIP(hipMemcpy(front.data(), c->front.p, c->NE, hipMemcpyDeviceToHost));
        std::copy(front.begin(), front.end(), w_front);
    }
    if (edge_flux) FVP_HIP(hipMemcpy(edge_flux, c->eflux.p, sizeof(double) * c->NE, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int fvp_set_upwind(fvp_ctx *c, const double *w_front) {
    if (!c || !w_front) { set_error("null argument"); return -1; }
    int halves = 0;
    for (int i = 0; i < c->NE; ++i) {
        double w = w_front[i];
        if (w == 0.5) ++halves;
        else if (w != 0.0 && w != 1.0) { set_error("edge weights must be 0, 0.5 or 1"); return -1; }
    }
    if (halves && halves != c->NE) { set_error("averaged and upwind edge weights cannot be mixed"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    FVP_HIP(hipStreamSynchronize(c->stream));
    if (halves) { c->averaging = 1; return 0; }
    std::vector<uint8_t> front(c->NE);
    for (int i = 0; i < c->NE; ++i) front[i] = w_front[i] == 1.0;
    FVP_HIP(hipMemcpy(c->front.p, front.data(), c->NE, hipMemcpyHostToDevice));
    launch_mask(c);
    FVP_HIP(hipGetLastError());
    c->averaging = 0;
    return 0;
}

extern "C" int fvp_capacity(fvp_ctx *c, double *ahh) {
    if (!c || !ahh) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    FVP_HIP(hipMemcpyAsync(ahh, c->cap.p, sizeof(double) * c->N, hipMemcpyDeviceToDevice, c->stream));
    return 0;
}

extern "C" int fvp_profile(fvp_ctx *c, int enable) {
    if (!c) { set_error("null context"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    FVP_HIP(hipStreamSynchronize(c->stream));
    for (int k = 0; k < kProfKinds; ++k) { c->prof_used[k] = 0; c->prof_ms[k] = 0.; c->prof_n[k] = 0; }
    c->prof = enable ? 1 : 0;
    return 0;
}

extern "C" int fvp_profile_get(fvp_ctx *c, int kind, double *total_ms, long *count) {
    if (!c || kind < 0 || kind >= kProfKinds) { set_error("invalid argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    prof_fold(c, kind);
    if (total_ms) *total_ms = c->prof_ms[kind];
    if (count) *count = c->prof_n[kind];
    return 0;
}

extern "C" int fvp_default_tile_nodes(const fvp_ctx *c) {
    if (!c) { set_error("null context"); return -1; }
    return c->made_tile;
}

extern "C" int fvp_set_residual_launch(fvp_ctx *c, int variant, int tile_nodes, int xcd_map) {
    if (!c) { set_error("null context"); return -1; }
    if (variant != FVP_RESIDUAL_OWNER && variant != FVP_RESIDUAL_WINDOW) { set_error("unknown residual variant"); return -1; }
    if (tile_nodes < 64 || tile_nodes > 4096 || (tile_nodes & (tile_nodes - 1))) {
        set_error("tile_nodes must be a power of two in [64, 4096]");
        return -1;
    }
    FVP_HIP(hipSetDevice(c->device));
    FVP_HIP(hipStreamSynchronize(c->stream));
    const int old = c->tile_nodes, old_v = c->rvariant;
    c->rvariant = variant;  // the window variant's LDS check depends on it
    if ((tile_nodes != old || variant != old_v) && build_tiles(c, tile_nodes)) {
        const std::string why = fvp_last_error();
        c->rvariant = old_v;
        if (build_tiles(c, old)) return -1;  // keep the context usable
        set_error(why);
        return -1;
    }
    c->xcd_map = xcd_map ? 1 : 0;
    return 0;
}

// Launch-shape autotuner for the residual: every (tile size, XCD grouping)
// candidate that fits the LDS is built and timed with HIP events over a few
// upwinded residual evaluations at the given state; the fastest is kept.  The
// tile sizes that the context was made with and has now are candidates too.
extern "C" int fvp_autotune(fvp_ctx *c, double t, const double *psi, const double *psip, int *variant,
                            int *tile_nodes, int *xcd_map, double *best_us) {
    if (!c || !psi || !psip) { set_error("null argument"); return -1; }
    FVP_HIP(hipSetDevice(c->device));
    hipStream_t s = c->stream;
    if (fvp_begin_step(c, t, psi, psip)) return -1;
    hipEvent_t e0, e1;
    FVP_HIP(hipEventCreate(&e0));
    FVP_HIP(hipEventCreate(&e1));
    std::vector<int> tiles = {256, 512, 1024, 2048};
    for (int tn : {c->made_tile, c->tile_nodes})
        if (std::find(tiles.begin(), tiles.end(), tn) == tiles.end()) tiles.push_back(tn);
    int best_t = c->tile_nodes, best_x = c->xcd_map, best_v = c->rvariant;
    double best = 1e300;
    const int reps = 10;
    for (int v : {FVP_RESIDUAL_OWNER, FVP_RESIDUAL_WINDOW})
    for (int tn : tiles) {
        if (fvp_set_residual_launch(c, v, tn, 1)) continue;  // window does not fit the LDS
        for (int x = 0; x <= 1; ++x) {
            c->xcd_map = x;
            for (int w = 0; w < 3; ++w)
                if (residual_impl(c, t, psi, psip, c->tmp3.p, 0)) return -1;
            FVP_HIP(hipEventRecord(e0, s));
            for (int r = 0; r < reps; ++r)
                if (residual_impl(c, t, psi, psip, c->tmp3.p, 0)) return -1;
            FVP_HIP(hipEventRecord(e1, s));
            FVP_HIP(hipEventSynchronize(e1));
            float ms = 0.f;
            FVP_HIP(hipEventElapsedTime(&ms, e0, e1));
            const double us = 1e3 * ms / reps;
            if (us < best) { best = us; best_t = tn; best_x = x; best_v = v; }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (fvp_set_residual_launch(c, best_v, best_t, best_x)) return -1;
    if (variant) *variant = best_v;
    if (tile_nodes) *tile_nodes = best_t;
    if (xcd_map) *xcd_map = best_x;
    if (best_us) *best_us = best;
    return 0;
}
