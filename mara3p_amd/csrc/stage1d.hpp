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
// Zones of a window are one chain where every block boundary in it joins blocks
// that are linked and consecutive in storage (nearly always).  Else the window is
// done in pieces, each piece's lanes finding their zones from the piece's first
// zone along the prev/next links: a neighbour stored elsewhere, or a copy of the
// edge zone past an outflow end.  A piece ends where the next block's own prev
// link does not lead back (its guard zones are not this chain's).
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

template<typename R>
__global__ void __launch_bounds__(64 * kWindowGroup)
stage1d_kernel(EulerParams prm, Stage1DArgs a)
{
    constexpr int NC = 5;
    const int n = a.n;
    const int i = threadIdx.x & 63;
    const long total = (long)a.nblk * n;
    // The second RK stage (u0 given) walks the list backwards: its first reads
    // are what the first stage wrote last (likeliest to be cached).
    const long group = a.u0 ? (long)gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const long first = (group * kWindowGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kWindowStage1D;
    const long end = first + kWindowStage1D < total ? first + kWindowStage1D : total;
    const R theta = R(prm.theta);
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    double rate = 0.0;                      // fused CFL reduction

    for (long lo = first; lo < end;) {
        // block and zone of lo, then of each lane along the storage order
        const int b0 = total < (1l << 31) ? (int)((unsigned)lo / (unsigned)n) : (int)(lo / n);
        const int p0 = (int)(lo - (long)b0 * n) + i - 2;      // the lane's zone counted from block b0's first
        int b = b0, z = p0;
        while (z >= n) { ++b; z -= n; }
        if (z < 0) { --b; z += n; }
        const bool inside = !a.pe && lo >= 2 && lo + 62 <= total;
        int prev = b - 1, next = b;                           // the links across the boundary before the lane's zone
        if (inside && i > 0 && z == 0) { prev = a.nbr[2 * b]; next = a.nbr[2 * (b - 1) + 1]; }
        // the state is fetched before the links are known (the latencies
        // overlap), and again by the pieces that do not follow the storage
        double u[NC], u0[NC] = {};
        double dl = a.dl;
        auto fetch = [&] () {
            const size_t at = (size_t)b * NC * n + z;
#pragma unroll
            for (int q = 0; q < NC; ++q) u[q] = a.u[at + (size_t)q * n];
            if (a.u0) {
#pragma unroll
                for (int q = 0; q < NC; ++q) u0[q] = a.u0[at + (size_t)q * n];
            }
            if (a.dl_blk) dl = a.dl_blk[b];
        };
        if (inside) fetch();
        int count = (int)(end - lo);                          // zones this piece updates
        if (__builtin_expect(__ballot(inside && prev == b - 1 && next == b) != ~0ull, 0)) {
            b = b0;
            z = p0;
            bool cut = false;                                 // past an end of the piece's chain
            if (a.pe) {
                cut = z >= n;
                z = min(max(z, 0), n - 1);
            } else if (z < 0) {
                const int pb = a.nbr[2 * b];
                if (pb >= 0) { b = pb; z += n; }
                else z = 0;
            } else {
                while (z >= n) {
                    const int nb = a.nbr[2 * b + 1];
                    cut |= nb < 0 || a.nbr[2 * nb] != b;
                    if (nb >= 0) { b = nb; z -= n; }
                    else z = n - 1;
                }
            }
            const unsigned long long other = __ballot(i >= 2 && (cut || (long)b * n + z != lo + (i - 2)));
            if (other) count = min(count, __builtin_ctzll(other) - 2);
            fetch();
        }
        const bool mine = i >= 2 && i < 2 + min(count, kWindowStage1D);

        bool ok = true;
        R p[NC], pl[NC], pr[NC], f[NC];
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
        // the left face of the lane's zone, from the half slopes of this zone
        // and the one before
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const R g = plm_half(lane_before(p[q]), p[q], lane_after(p[q]), theta);
            pl[q] = lane_before(p[q] + g);
            pr[q] = p[q] - g;
        }
        Euler<R>::template riemann<1>(pl, pr, prm, f);
        double wv[NC];
        const Divisor<double> by_dl(dl);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const double dfx = double(lane_after(f[q])) - double(f[q]);
            if constexpr (is_fp64<R>::value) wv[q] = u[q] - by_dl(dfx * dt);
            else wv[q] = u[q] - dfx * (dt / dl);
            if (a.u0) wv[q] = u0[q] * a.rk_b + wv[q] * (1.0 - a.rk_b);
        }
        if (mine) {
            double* o = a.out + (size_t)b * NC * n + z;
#pragma unroll
            for (int q = 0; q < NC; ++q) o[(size_t)q * n] = wv[q];
            if (!ok) report_error(a.err, 1, b, z);
            if (a.rate_slot) rate = fmax(rate, Euler<double>::max_speed(wv, prm) * (1.0 / dl));
        }
        lo += count;
    }
    if (a.rate_slot) workgroup_atomic_max<64 * kWindowGroup>(rate, a.rate_slot);
}

} // namespace m3p
