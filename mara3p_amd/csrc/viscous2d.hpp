// Isothermal 2D stages with a kinematic viscosity: the viscous stress of
// godunov_and_viscous_fluxes (src/module_locally_isothermal.cpp:106-174,
// problems/minidisk_scheme.cpp:220-287) added to the HLLE flux of every face.
//
// The stress at a face needs the PLM slopes of its two cells along both
// axes, i.e. a 3 x 3 block of primitives plus the cross of radius 2 around
// each zone, corners included.  A face shared by two tiles is computed from
// the same operands in the same order by both, so the update stays
// conservative and the FP64 kernel reproduces the reference's arithmetic:
//   mu    = nu * 0.5 * (sigma_upper_state + sigma_lower_state)
//   x face: tau_xx = mu (dx vx - dy vy), tau_xy = mu (dx vy + dy vx),
//           F += (0, -tau_xx, -tau_xy)
//   y face: tau_yx = mu (dx vy + dy vx), tau_yy = -mu (dx vx - dy vy),
//           F += (0, -tau_yx, -tau_yy)
// with each derivative the mean of the two cells' full PLM slopes over dl
// (adjacent_mean, src/core_ndarray_ops.hpp:84-90).  This path is used only
// when nu != 0; the inviscid stages run the tile-march kernel.
#pragma once
#include "stage2d.hpp"

namespace m3p {

template<typename R>
struct ViscousTerms {
    // derivative from two full slopes: 0.5 (a + b) / dl (FP32: times 1 / dl)
    __device__ static __forceinline__ R mean_over(R a, R b, const Divisor<double>& by_dl, R idl)
    {
        if constexpr (is_fp64<R>::value) return by_dl(R(0.5) * (a + b));
        else return R(0.5) * (a + b) * idl;
    }
    // Adds the stress of a face of axis AXIS to f.  pl, pr: the face states
    // (lower cell + g/2, upper cell - g/2); gl*, gu*: full slopes of the lower
    // and upper cells, along (L) and across (T) the face normal.
    template<int AXIS>
    __device__ static __forceinline__ void add(R* f, const R* pl, const R* pr, const R* glL, const R* guL,
                                               const R* glT, const R* guT, double nu, const Divisor<double>& by_dl, R idl)
    {
        R mu = R(nu) * R(0.5) * (pr[0] + pl[0]);
        R dL_vx = mean_over(glL[1], guL[1], by_dl, idl);
        R dT_vx = mean_over(glT[1], guT[1], by_dl, idl);
        R dL_vy = mean_over(glL[2], guL[2], by_dl, idl);
        R dT_vy = mean_over(glT[2], guT[2], by_dl, idl);
        if constexpr (AXIS == 1) {          // L = x, T = y
            R tauxx = mu * (dL_vx - dT_vy);
            R tauxy = mu * (dL_vy + dT_vx);
            f[0] = f[0] + R(0);
            f[1] = f[1] + -tauxx;
            f[2] = f[2] + -tauxy;
        } else {                            // L = y, T = x
            R tauyx = mu * (dT_vy + dL_vx);
            R tauyy = -mu * (dT_vx - dL_vy);
            f[0] = f[0] + R(0);
            f[1] = f[1] + -tauyx;
            f[2] = f[2] + -tauyy;
        }
    }
};

// A workgroup owns a T x T tile of zones.  Primitives of the tile and two zones
// around it go to LDS, then the full slopes along both axes of the tile and
// one zone around it, then every face flux of the tile, each computed once
// (lane (j, k) the faces below its zone on both axes, 2 T lanes also the
// tile's upper faces), then each lane updates its zone.  One lane per zone
// with all its operands in registers recovered 13 zones, took ten slopes and
// computed every face twice, at two waves per SIMD: FP64 151 us a step at
// 1024^2 (83 by tiles), mixed 94 (61), FP64 512^2 43 (28).  Tiles that reach
// past the block clamp their loads and store nothing there.  The isothermal
// recoveries report no error (as the reference's), so nothing here does.
constexpr int kViscTile = 16;

template<class S, class Ld, int T>
__global__ void __launch_bounds__(T * T)
iso_visc_stage_kernel(typename S::Params prm, Ld ld_arg, StageArgs a, double nu)
{
    using R = typename S::Real;
    constexpr int NC = 3;
    constexpr int EP = T + 4, EG = T + 2;
    resolve_params(prm);
    const int n = a.n;
    const int tiles = (n + T - 1) / T;
    TileCtx tc;
    tc.b = blockIdx.x / (tiles * tiles);
    const int rem = blockIdx.x % (tiles * tiles);
    tc.k0 = rem / tiles * T;
    tc.c0 = rem % tiles * T;
    tc.n = n;
    const int b = tc.b;
    if (a.bcoord) { tc.bi = a.bcoord[2 * b]; tc.bj = a.bcoord[2 * b + 1]; }
    else          { tc.bi = a.bi0; tc.bj = a.bj0; }
    Ld ld = ld_arg;
    ld.bind(b);
    const int t = threadIdx.x, kl = t / T, cl = t % T;
    const int k = tc.k0 + kl, c = tc.c0 + cl;
    const bool inside = k < n && c < n;

    __shared__ typename S::template TileData<T, T> td;
    __shared__ R P[NC][EP][EP];             // [2 + r][2 + q]: zone (k0 + r, c0 + q)
    __shared__ R Gx[NC][EG][EG];            // [1 + r][1 + q]: full slopes of zone (k0 + r, c0 + q) along rows
    __shared__ R Gy[NC][EG][EG];            // and along columns
    __shared__ R Fx[NC][T + 1][T];          // x flux at face k0 + r of column c0 + q
    __shared__ R Fy[NC][T][T + 1];          // y flux at face c0 + q of row k0 + r

    S::setup(td, prm, tc);
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const double dl = a.dl_blk ? a.dl_blk[b] : a.dl;
    const Divisor<double> by_dl(dl);
    const R idl = R(1.0 / dl);
    const R theta = R(S::theta(prm));

    for (int i = t; i < EP * EP; i += T * T) {
        const int r = i / EP, q = i % EP;
        R p[NC];
        (void)ld.prim(b, min(tc.k0 + r - 2, n + 1), min(tc.c0 + q - 2, n + 1), prm, p);
#pragma unroll
        for (int m = 0; m < NC; ++m) P[m][r][q] = p[m];
    }
    double uu[NC], u0[NC] = {};
    if (inside) {
        ld.cons_row(b, k, c, uu);
        if (a.u0) {
            const double* z0 = a.u0 + ((size_t)b * NC * n + k) * n + c;
#pragma unroll
            for (int m = 0; m < NC; ++m) u0[m] = z0[(size_t)m * n * n];
        }
    }
    __syncthreads();
    for (int i = t; i < EG * EG; i += T * T) {
        const int r = i / EG, q = i % EG;
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            Gx[m][r][q] = plm(P[m][r][q + 1], P[m][r + 1][q + 1], P[m][r + 2][q + 1], theta);
            Gy[m][r][q] = plm(P[m][r + 1][q], P[m][r + 1][q + 1], P[m][r + 1][q + 2], theta);
        }
    }
    __syncthreads();

    // faces between zones (r - 1, q) and (r, q), and (r, q - 1) and (r, q):
    // states p_lo + 0.5 g_lo and p_up - 0.5 g_up
    auto xface = [&] (int r, int q) {
        R pl[NC], pr[NC], gl[NC], gu[NC], hl[NC], hu[NC], f[NC];
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            gl[m] = Gx[m][r][q + 1]; gu[m] = Gx[m][r + 1][q + 1];
            hl[m] = Gy[m][r][q + 1]; hu[m] = Gy[m][r + 1][q + 1];
            pl[m] = P[m][r + 1][q + 2] + R(0.5) * gl[m];
            pr[m] = P[m][r + 2][q + 2] - R(0.5) * gu[m];
        }
        S::template face<1>(pl, pr, prm, td, tc, min(tc.k0 + r, n), min(tc.c0 + q, n - 1), f);
        ViscousTerms<R>::template add<1>(f, pl, pr, gl, gu, hl, hu, nu, by_dl, idl);
#pragma unroll
        for (int m = 0; m < NC; ++m) Fx[m][r][q] = f[m];
    };
    auto yface = [&] (int r, int q) {
        R pl[NC], pr[NC], gl[NC], gu[NC], hl[NC], hu[NC], f[NC];
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            gl[m] = Gy[m][r + 1][q]; gu[m] = Gy[m][r + 1][q + 1];
            hl[m] = Gx[m][r + 1][q]; hu[m] = Gx[m][r + 1][q + 1];
            pl[m] = P[m][r + 2][q + 1] + R(0.5) * gl[m];
            pr[m] = P[m][r + 2][q + 2] - R(0.5) * gu[m];
        }
        S::template face<2>(pl, pr, prm, td, tc, min(tc.k0 + r, n - 1), min(tc.c0 + q, n), f);
        ViscousTerms<R>::template add<2>(f, pl, pr, gl, gu, hl, hu, nu, by_dl, idl);
#pragma unroll
        for (int m = 0; m < NC; ++m) Fy[m][r][q] = f[m];
    };
    xface(kl, cl);
    yface(kl, cl);
    if (t < T) xface(T, t);
    else if (t >= 64 && t < 64 + T) yface(t - 64, T);       // in another wave
    __syncthreads();

    if (inside) {
        double dfx[NC], dfy[NC], res[NC];
        R pc[NC];
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            dfx[m] = double(Fx[m][kl + 1][cl]) - double(Fx[m][kl][cl]);
            dfy[m] = double(Fy[m][kl][cl + 1]) - double(Fy[m][kl][cl]);
            pc[m] = P[m][kl + 2][cl + 2];
        }
        S::update(prm, td, tc, k, c, uu, pc, dfx, dfy, dt, dl, res);
        double* o = a.out + ((size_t)b * NC * n + k) * n + c;
#pragma unroll
        for (int m = 0; m < NC; ++m)
            o[(size_t)m * n * n] = a.u0 ? u0[m] * a.rk_b + res[m] * (1.0 - a.rk_b) : res[m];
    }
}

} // namespace m3p
