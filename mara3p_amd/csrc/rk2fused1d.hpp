// Fused RK2 step of the 1D work-list stage (mixed precision): both stages of
// one RK2 step in one launch, the first stage's state never stored.
//
// The two-stage form (stage1d_kernel twice) writes U1 = L(U0) for every block
// and reads it back, with its guard zones, for U = b U0 + (1 - b) L(U1)
// (modules::euler1d::updated_conserved, src/module_euler.cpp:107-135, per
// stage; outflow ends, src/mara.cpp:123-143).  Here a wave owns 56 zones,
// consecutive in storage, and holds them in its lanes 4 .. 59 with the four
// zones before and after: each lane takes one half slope and one face flux
// (the left face of its zone) and one update per stage, and gets its
// neighbours' values by wave shifts.  Each stage leaves two lanes less at each
// end with the right values, so after two stages lanes 4 .. 59 have theirs.
// Nothing passes through LDS and nothing waits at a barrier.
//
// A workgroup per 64-zone block, a lane per zone, needed 69 and 65 faces of 64
// lanes in the two stages, two nearly empty passes out of four, took two
// slopes per face and met four barriers.  512 problems of 512 to 8192 zones in
// blocks of 64: 55 to 45 us a step (some 530 VALU instructions per 56 zones, 965
// per 64 before; 201 MB, 4.5 TB/s), with the CFL reduction at half that size 52 to
// 36, 300 problems in blocks of 16 16.7 to 8.9.  One-wave workgroups: 48 us,
// with the CFL reduction 48.
//
// Zones of a window are one chain where every block boundary in it joins
// blocks that are linked and consecutive in storage (nearly always).  Else the
// window is done in pieces, each piece's lanes finding their zones along the
// prev/next links from the piece's first zone: a neighbour stored elsewhere,
// or, past an outflow end, a copy of the edge zone, whose lanes take the edge
// zone's U1 in the second stage as the two-stage guard fill does.
//
// Every U1 value is the one the two-stage path computes: a zone of another
// block is updated with that block's cell spacing from the same operands (its
// guard zones are this chain's zones, which needs the prev/next links to be
// mutual: block pb = prev(b) has next(pb) = b, and likewise for next, as in
// every chain and ring; a table where they are not is reported through the
// error latch with code M3P_ERR_BAD_SHAPE, and such an end is treated as
// outflow).  So the step equals two stage1d launches value for value; HBM sees
// U0 and U once, instead of U0, U1, U1, U0 and U.
#pragma once
#include "stage1d.hpp"

namespace m3p {

constexpr int kWindow1D = 56;          // zones a wave updates

static __global__ void __launch_bounds__(64 * kWindowGroup)
rk2_fused_1d_kernel(EulerParams prm, Stage1DArgs a)
{
    using R = float;
    constexpr int NC = 5;
    const int n = a.n;
    const int i = threadIdx.x & 63;
    const long total = (long)a.nblk * n;
    const long first = ((long)blockIdx.x * kWindowGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kWindow1D;
    const long end = first + kWindow1D < total ? first + kWindow1D : total;
    const R theta = R(prm.theta);
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    double rate = 0.0;                      // fused CFL reduction

    for (long lo = first; lo < end;) {
        // block and zone of lo, then of each lane along the storage order
        const int b0 = total < (1l << 31) ? (int)((unsigned)lo / (unsigned)n) : (int)(lo / n);
        const int p0 = (int)(lo - (long)b0 * n) + i - 4;      // the lane's zone counted from block b0's first
        int b = b0, z = p0;
        while (z >= n) { ++b; z -= n; }
        if (z < 0) { --b; z += n; }
        const bool inside = lo >= 4 && lo + 60 <= total;
        int prev = b - 1, next = b;                           // the links across the boundary before the lane's zone
        if (inside && i > 0 && z == 0) { prev = a.nbr[2 * b]; next = a.nbr[2 * (b - 1) + 1]; }
        // the state is fetched before the links are known (the latencies
        // overlap), and again by the pieces that do not follow the storage
        double u0[NC];
        auto fetch = [&] () {
            const double* src = a.u + (size_t)b * NC * n + z;
#pragma unroll
            for (int q = 0; q < NC; ++q) u0[q] = src[(size_t)q * n];
        };
        double dl = a.dl;
        if (inside) {
            fetch();
            if (a.dl_blk) dl = a.dl_blk[b];
        }
        int count = (int)(end - lo);                          // zones this piece updates
        unsigned long long low = 0, high = 0;                 // lanes past an outflow end
        if (__builtin_expect(__ballot(inside && prev == b - 1 && next == b) != ~0ull, 0)) {
            b = b0;
            z = p0;
            bool out_lo = false, out_hi = false;
            if (z < 0) {
                const int pb = a.nbr[2 * b];
                const bool mutual = pb < 0 || a.nbr[2 * pb + 1] == b;
                if (!mutual) report_error(a.err, 4, b, -1);
                if (pb >= 0 && mutual) { b = pb; z += n; }
                else { z = 0; out_lo = true; }
            }
            while (z >= n) {
                const int nb = a.nbr[2 * b + 1];
                const bool mutual = nb < 0 || a.nbr[2 * nb] == b;
                if (!mutual) report_error(a.err, 4, b, n);
                if (nb >= 0 && mutual) { b = nb; z -= n; }
                else { z = n - 1; out_hi = true; }
            }
            low = __ballot(out_lo);
            high = __ballot(out_hi);
            // the piece ends at the first lane whose zone is not the storage's
            const unsigned long long other = __ballot(i >= 4 && (out_hi || (long)b * n + z != lo + (i - 4)));
            if (other) count = min(count, __builtin_ctzll(other) - 4);
            fetch();
            if (a.dl_blk) dl = a.dl_blk[b];
        }
        const bool mine = i >= 4 && i < 4 + min(count, kWindow1D);
        const double dtdl = dt / dl;
        double u1[NC];
        R p[NC], f[NC];

        // the left face of the lane's zone, from the half slopes of this zone
        // and the one before, with the operands and order of stage1d_kernel
        auto face = [&] () {
            R pl[NC], pr[NC];
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const R g = plm_half(lane_before(p[q]), p[q], lane_after(p[q]), theta);
                pl[q] = lane_before(p[q] + g);
                pr[q] = p[q] - g;
            }
            Euler<R>::template riemann<1>(pl, pr, prm, f);
        };
        auto flux_difference = [&] (int q) { return double(lane_after(f[q])) - double(f[q]); };

        bool ok = Euler<R>::recover(u0, prm, p);
        face();
#pragma unroll
        for (int q = 0; q < NC; ++q) u1[q] = u0[q] - flux_difference(q) * dtdl;
        ok &= Euler<R>::recover(u1, prm, p);
        if (low) {          // the lanes below take the edge zone's, the first lane of the chain
            const int e = 64 - __builtin_clzll(low);
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const R v = __shfl(p[q], e, 64);
                if (i < e) p[q] = v;
            }
        }
        if (high) {         // and those above the last lane's
            const int e = __builtin_ctzll(high) - 1;
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const R v = __shfl(p[q], e, 64);
                if (i > e) p[q] = v;
            }
        }
        face();
        double wv[NC];
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const double res = u1[q] - flux_difference(q) * dtdl;
            wv[q] = u0[q] * a.rk_b + res * (1.0 - a.rk_b);
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
