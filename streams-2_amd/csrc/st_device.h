// st_device.h -- device helpers shared by the kernel files: wave and block
// reductions, the isothermal-wall ghost of a point and the ghost images of an
// interior value.
#pragma once

#include "st_internal.h"

namespace st {

constexpr int H = 3;           // stencil half width of the flux windows
constexpr int RED_THREADS = 256;

// -------------------------------------------------------------- utilities
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    return v;
}
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_down(v, off, 64));
    return v;
}

// Sum over the wave in lane 63, by DPP moves (shifts within the rows of 16
// lanes, then row broadcasts): no LDS round trips.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// Block sum of NV values in a fixed order; result valid in thread 0.
__device__ __forceinline__ int flat_block() { return blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z); }
__device__ __forceinline__ int flat_thread() { return threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z); }

template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double (*lds)[NV]) {
    const int ft = flat_thread();
    const int lane = ft & 63;
    const int wid = ft >> 6;
    const int nw = (blockDim.x * blockDim.y * blockDim.z + 63) >> 6;
#pragma unroll
    for (int q = 0; q < NV; q++) v[q] = wave_sum(v[q]);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; q++) lds[wid][q] = v[q];
    }
    __syncthreads();
    if (ft == 0) {
#pragma unroll
        for (int q = 0; q < NV; q++) {
            double a = lds[0][q];
            for (int w = 1; w < nw; w++) a += lds[w][q];
            v[q] = a;
        }
    }
}

// The viscosity of a conserved state, by the operations of k_aux: whether the
// aux pass or the kernel that last wrote w formed it must not show in a result.
__device__ __forceinline__ double mu_of(const KPar &P, const double (&c)[5]) {
    const double ri = 1.0 / c[0];
    const double uu = c[1] * ri, vv = c[2] * ri, ww = c[3] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = c[4] / c[0] - qq;
    return viscosity_of(P, temperature_from_e(P, ee, P.t0));
}

// The largest spectral radius of compute_dt_subroutine (kernels_cpu.F90:
// 6814-6880) at a point of viscosity mu with the Euler metrics a and the
// viscous ones s, by the operations of k_aux as mu_of.
__device__ __forceinline__ double cfl_radius(const KPar &P, const double (&c)[5], double mu, const double (&a)[3],
                                             const double (&s)[3]) {
    const double ri = 1.0 / c[0];
    const double uu = c[1] * ri, vv = c[2] * ri, ww = c[3] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = c[4] / c[0] - qq;
    const double tt = temperature_from_e(P, ee, P.t0);
    const double nu = ri * mu, kor = nu / P.prandtl;
    const double cs = sqrt(gamloc_of(P, tt) * P.rgas0 * tt);
    double mx = fmax(fmax((fabs(uu) + cs) * a[0], (fabs(vv) + cs) * a[1]), (fabs(ww) + cs) * a[2]);
    mx = fmax(mx, fmax(nu * s[0], fmax(nu * s[1], nu * s[2])));
    return fmax(mx, fmax(kor * s[0], fmax(kor * s[1], kor * s[2])));
}

// bcwall_staggered_subroutine (kernels_cpu.F90:6612-6678): the ghost state d
// that mirrors the state c about an isothermal wall (t_start as in
// temperature_from_e).
__device__ __forceinline__ void wall_ghost_of(const KPar &P, const double (&c)[5], double t_start, double (&d)[5]) {
    double rho = c[0];
    const double uu = c[1] / rho, vv = c[2] / rho, ww = c[3] / rho;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    double ee = c[4] / rho - qq;
    double tt = temperature_from_e(P, ee, t_start);
    const double pp = rho * tt * P.rgas0;
    tt = 2.0 * P.t_wall - tt;
    ee = e_from_temperature(P, tt);
    rho = pp / tt / P.rgas0;
    d[0] = rho;
    d[1] = -rho * uu;
    d[2] = -rho * vv;
    d[3] = -rho * ww;
    d[4] = rho * (ee + qq);
}
// for one ghost point: the mirror of interior point js, written at jg
template <typename R>
__device__ __forceinline__ void wall_ghost(const Geo &g, const KPar &P, double *__restrict__ w, const R *__restrict__ wa,
                                           int i, int js, int jg, int k) {
    const int s = gidx(g, i, js, k), d = gidx(g, i, jg, k);
    const size_t nv = g.nvol;
    double c[5], x[5];
#pragma unroll
    for (int m = 0; m < 5; m++) c[m] = w[m * nv + s];
    wall_ghost_of(P, c, double(wa[5 * nv + s]), x);
#pragma unroll
    for (int m = 0; m < 5; m++) w[m * nv + d] = x[m];
}

// exclusive prefix over the block's 256 threads of v; *total receives the sum
template <typename T>
__device__ __forceinline__ T block_excl_scan256(T v, T *wsum, T *total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const T y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    T before = 0, tot = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (q < wv) before += wsum[q];
        tot += wsum[q];
    }
    __syncthreads();
    *total = tot;
    return before + x - v;
}

// Ghost images of an interior value: periodic copy for periodic directions
// (bcswap_var), zero-gradient copy otherwise (bcextr_var).
template <typename R>
__device__ __forceinline__ void write_images(const Geo &g, const KPar &P, R *__restrict__ a, int i, int j, int k,
                                             R v, bool extrapolate) {
    const int ng = g.ng;
    if (P.periodic[0]) {
        if (i <= ng) a[gidx(g, i + g.nx, j, k)] = v;
        if (i > g.nx - ng) a[gidx(g, i - g.nx, j, k)] = v;
    } else if (extrapolate) {
        if (i == 1) for (int l = 1; l <= ng; l++) a[gidx(g, 1 - l, j, k)] = v;
        if (i == g.nx) for (int l = 1; l <= ng; l++) a[gidx(g, g.nx + l, j, k)] = v;
    }
    if (P.periodic[1]) {
        if (j <= ng) a[gidx(g, i, j + g.ny, k)] = v;
        if (j > g.ny - ng) a[gidx(g, i, j - g.ny, k)] = v;
    } else if (extrapolate) {
        if (j == 1) for (int l = 1; l <= ng; l++) a[gidx(g, i, 1 - l, k)] = v;
        if (j == g.ny) for (int l = 1; l <= ng; l++) a[gidx(g, i, g.ny + l, k)] = v;
    }
    if (P.periodic[2] && P.ndim == 3) {
        if (k <= ng) a[gidx(g, i, j, k + g.nz)] = v;
        if (k > g.nz - ng) a[gidx(g, i, j, k - g.nz)] = v;
    } else if (extrapolate) {
        if (k == 1) for (int l = 1; l <= ng; l++) a[gidx(g, i, j, 1 - l)] = v;
        if (k == g.nz) for (int l = 1; l <= ng; l++) a[gidx(g, i, j, g.nz + l)] = v;
    }
}

}  // namespace st
