// The fused 1D Euler stage kernel: guard fill (periodic or outflow) +
// recover + PLM + HLLE + update (+ RK combine), one pass per stage.
//   modules::euler1d::updated_conserved, src/module_euler.cpp:107-135
//   outflow boundary condition,           src/mara.cpp:123-143
//
// A wave owns 60 zones, consecutive in storage, and holds them in its lanes 2 ..
// 61 with the two zones before and after: each lane recovers its zone and takes
// one half slope, one face flux (the left face of its zone) and one update, with
// its neighbours' values by wave shifts.  Every face flux is computed once in a
// window; nothing passes through LDS and nothing waits at a barrier.
//
// A workgroup per block with LDS rows took both slopes of every face, met two
// barriers and needed a pass of its own for the left faces; it was bound by its
// arithmetic.  512 problems of 512 to 8192 zones in blocks of 64, both stages,
// FP64: 149 to 100 us (445 MB, 4.5 TB/s: bound by memory); 64 problems in blocks
// of 128, 22.6 to 18.1; 1688 blocks of 32, 17.9 to 10.2; 1024 zones, a launch
// 4.5 to 4.1.
//
// A window is one chain where every block boundary in it joins blocks that are
// linked both ways and consecutive in storage; lanes before the list and past it
// hold the guard zones of its first and last block.  At any other boundary (an
// end of a chain, a neighbour stored elsewhere, links that do not lead back) the
// lanes on its two sides load the two guard zones of their own block's link
// themselves: blocks are at least 16 zones, so a lane has one such side at
// most, and one more pass of the left face's arithmetic gives the right faces
// of all chains that end in the window.  Links are read for blocks of the list
// only; a neighbour may be stored behind the list, with no row of its own.  Both
// stages, mixed: the 512 problems above in shuffled order 91 us (76 in order),
// blocks of 16 of 512 problems of 64 to 1024 zones 21 (17), 4096 problems of one
// block of 64 zones 19.6; done in pieces, each from its first zone along the
// links, they took 141, 60 and 24.
#pragma once
#include "physics.hpp"

namespace m3p {

struct Stage1DArgs {
    const double* u;       // [nblk][5][n]
    const double* u0;      // RK base or nullptr
    double* out;
    const int* nbr;        // [nblk][2] = {prev, next}; -1 = outflow boundary
    double dt, dl, rk_b;
    const double* dt_dev;  // device-resident dt or nullptr
    const double* dl_blk;  // per-block cell spacing or nullptr
    int n, nblk;
    int* err;
    // extended-array mode (per-block compatibility): pe [5][n+4] primitives
    const double* pe;
    int outflow_lower, outflow_upper;
    // fused CFL reduction: atomic max of (max(|v1|, |v2|) + c_s) / dl of the
    // values written, or nullptr
    unsigned long long* rate_slot;
};

constexpr int kWindowStage1D = 60;     // zones a wave updates
constexpr int kWindowGroup = 4;        // waves of a workgroup

// FP64 at four waves per SIMD (124 VGPRs): left to itself the compiler takes 132
// and three waves (512 problems in order 102 us, 90 at four).
template<typename R>
__global__ void __launch_bounds__(64 * kWindowGroup) __attribute__((amdgpu_waves_per_eu(is_fp64<R>::value ? 4 : 6, 8)))
stage1d_kernel(EulerParams prm, Stage1DArgs a)
{
    constexpr int NC = 5;
    const int n = a.n;
    const int i = threadIdx.x & 63;
    const long total = (long)a.nblk * n;
    // The second RK stage (u0 given) walks the list backwards: its first reads
    // are what the first stage wrote last (likeliest to be cached).
    const long group = a.u0 ? (long)gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const long lo = (group * kWindowGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kWindowStage1D;
    const long end = lo + kWindowStage1D < total ? lo + kWindowStage1D : total;
    const R theta = R(prm.theta);
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    double rate = 0.0;                      // fused CFL reduction

    if (lo < end) {
        // block and zone of lo, then of each lane along the storage order
        const int b0 = total < (1l << 31) ? (int)((unsigned)lo / (unsigned)n) : (int)(lo / n);
        const int p0 = (int)(lo - (long)b0 * n) + i - 2;      // the lane's zone counted from block b0's first
        int b = b0, z = p0;
        while (z >= n) { ++b; z -= n; }
        if (z < 0) { --b; z += n; }
        const bool there = b >= 0 && b < a.nblk;
        const bool edge = !a.pe && i > 0 && z == 0 && b > 0 && there;       // a block boundary before the lane's zone
        int prev = -1, next = -1;                             // the links across it
        if (edge) { prev = a.nbr[2 * b]; next = a.nbr[2 * (b - 1) + 1]; }
        const bool cut = edge && !(prev == b - 1 && next == b);
        // lanes before the list and past it hold the guard zones of its first
        // and its last block
        size_t at = (size_t)b * NC * n + z, from = at;
        bool behind = false;                                  // of a block with no row in the list
        if (!there) {
            const int eb = b < 0 ? 0 : a.nblk - 1, ez = b < 0 ? 0 : n - 1;
            const int link = a.pe ? -1 : a.nbr[b < 0 ? 0 : 2 * a.nblk - 1];
            const int gz = link < 0 ? ez : b < 0 ? z : min((b - a.nblk) * n + z, n - 1);
            from = (size_t)(link < 0 ? eb : link) * NC * n + gz;
            behind = link >= a.nblk && (b < 0 || gz < 2);
            b = eb;
            z = ez;
            at = (size_t)b * NC * n + z;
        }
        double u[NC], u0[NC] = {};
        double dl = a.dl;
#pragma unroll
        for (int q = 0; q < NC; ++q) u[q] = a.u[from + (size_t)q * n];
        if (a.u0) {
#pragma unroll
            for (int q = 0; q < NC; ++q) u0[q] = a.u0[at + (size_t)q * n];
        }
        if (a.dl_blk) dl = a.dl_blk[b];
        const bool mine = i >= 2 && i < 2 + (int)(end - lo);

        bool ok = true;
        R p[NC];
        // dF of the lane's zone.  CUT: with first and last, the lanes on the two
        // sides of a boundary that joins nothing, and their blocks' link there.
        double dfx[NC];
        auto fluxes = [&] (auto cut_c, bool first, bool last, int link) {
            constexpr bool CUT = decltype(cut_c)::value;
            // the two guard zones, fetched before the zone's own values arrive
            // (copies of the edge zone at an outflow end)
            double g1[NC] = {}, g2[NC] = {};
            const bool away = CUT && (first || last) && link >= 0;
            if constexpr (CUT) {
                if (away) {
                    const double* src = a.u + (size_t)link * NC * n + (last ? 0 : n - 1);
                    const int step = last ? 1 : -1;
#pragma unroll
                    for (int q = 0; q < NC; ++q) { g1[q] = src[(size_t)q * n]; g2[q] = src[(size_t)q * n + step]; }
                }
            }
            if (a.pe) {
                // extended-array mode (per-block compatibility): zones -2 .. n + 1 of
                // the caller's primitive array
                int e = min(p0, n + 1);
                if (a.outflow_lower && e < 0) e = 0;
                else if (!a.outflow_lower && a.outflow_upper && e >= n) e = n - 1;
#pragma unroll
                for (int q = 0; q < NC; ++q) p[q] = R(a.pe[(size_t)q * (n + 4) + e + 2]);
            } else {
                ok = Euler<R>::recover(u, prm, p);
            }
            // the nearest guard zone's primitives, and its face state
            R gp[NC] = {}, gs[NC] = {};
            if constexpr (CUT) {
                if (first || last) {
                    R gq[NC];
#pragma unroll
                    for (int q = 0; q < NC; ++q) gp[q] = gq[q] = p[q];
                    if (away) {
                        bool gok = Euler<R>::recover(g1, prm, gp);
                        gok &= Euler<R>::recover(g2, prm, gq);
                        if (link >= a.nblk) ok &= gok;        // no lane of the list reports it
                    }
#pragma unroll
                    for (int q = 0; q < NC; ++q) {
                        const R h = plm_half(first ? gq[q] : p[q], gp[q], first ? p[q] : gq[q], theta);
                        gs[q] = first ? gp[q] + h : gp[q] - h;
                    }
                }
            }
            // the left face of the lane's zone, from the half slopes of this
            // zone and the one before
            R pl[NC], pr[NC], up[NC], f[NC];
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                R below = lane_before(p[q]), above = lane_after(p[q]);
                if constexpr (CUT) { below = first ? gp[q] : below; above = last ? gp[q] : above; }
                const R g = plm_half(below, p[q], above, theta);
                up[q] = p[q] + g;
                pl[q] = lane_before(up[q]);
                if constexpr (CUT) pl[q] = first ? gs[q] : pl[q];
                pr[q] = p[q] - g;
            }
            Euler<R>::template riemann<1>(pl, pr, prm, f);
            R fr[NC];
            if constexpr (CUT) {
                if (last) Euler<R>::template riemann<1>(up, gs, prm, fr);
            }
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                R upper = lane_after(f[q]);
                if constexpr (CUT) upper = last ? fr[q] : upper;
                dfx[q] = double(upper) - double(f[q]);
            }
        };
        const unsigned long long cuts = __ballot(cut);
        if (__builtin_expect(cuts != 0, 0)) {
            const int above = lane_after(next);               // the next link of a last lane's block
            fluxes(std::true_type{}, there && cut, there && (cuts >> i) >> 1 & 1, cut ? prev : above);
        } else {
            fluxes(std::false_type{}, false, false, -1);
        }

        double wv[NC];
        const Divisor<double> by_dl(dl);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            if constexpr (is_fp64<R>::value) wv[q] = u[q] - by_dl(dfx[q] * dt);
            else wv[q] = u[q] - dfx[q] * (dt / dl);
            if (a.u0) wv[q] = u0[q] * a.rk_b + wv[q] * (1.0 - a.rk_b);
        }
        if (!ok && (mine || behind)) report_error(a.err, 1, b, z);
        if (mine) {
            double* o = a.out + at;
#pragma unroll
            for (int q = 0; q < NC; ++q) o[(size_t)q * n] = wv[q];
            if (a.rate_slot) rate = fmax(rate, Euler<double>::max_speed(wv, prm) * (1.0 / dl));
        }
    }
    if (a.rate_slot) workgroup_atomic_max<64 * kWindowGroup>(rate, a.rate_slot);
}

} // namespace m3p
