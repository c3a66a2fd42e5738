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
// blocks of 64: 55 to 41 us a step (513 VALU instructions per 56 zones, 965 per 64
// before; 193 MB, 4.8 TB/s), with the CFL reduction at half that size 52 to
// 36, 300 problems in blocks of 16 16.7 to 8.9.  One-wave workgroups: 48 us,
// with the CFL reduction 48.
//
// Zones of a window are one chain where every block boundary in it joins
// blocks that are linked both ways and consecutive in storage (nearly always);
// lanes before the list and past it hold the guard zones of its first and last
// block.  Else the window is cut there, and each part takes the two stages in turn
// with its zones in their lanes; the lanes beside it hold its guard zones for
// the while, found once for the whole window: blocks are at least 16 zones,
// so a lane stands beside one cut at most.  The guard zones lie across the
// part's own prev/next link or, past an outflow end, copy the edge zone, whose
// lanes take the edge zone's U1 in the second stage as the two-stage guard fill
// does.  The list above in shuffled order (two parts a window) takes 63 us, in
// order 39.6; blocks of 16 of 512 problems of 64 to 1024 zones 20 and 9.8.  Parts
// that found their zones along the links one after the other took 71 and 27; a
// workgroup per block 50 and 25, whatever the order.
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
    const long lo = ((long)blockIdx.x * kWindowGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kWindow1D;
    const long end = lo + kWindow1D < total ? lo + kWindow1D : total;
    const R theta = R(prm.theta);
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    double rate = 0.0;                      // fused CFL reduction

    if (lo < end) {
        // block and zone of lo, then of each lane along the storage order
        const int b0 = total < (1l << 31) ? (int)((unsigned)lo / (unsigned)n) : (int)(lo / n);
        const int p0 = (int)(lo - (long)b0 * n) + i - 4;      // the lane's zone counted from block b0's first
        int b = b0, z = p0;
        while (z >= n) { ++b; z -= n; }
        if (z < 0) { --b; z += n; }
        const bool there = b >= 0 && b < a.nblk;
        const bool edge = i > 0 && z == 0 && b > 0 && there;  // a block boundary before the lane's zone
        int prev = -1, next = -1;                             // the links across it
        if (edge) { prev = a.nbr[2 * b]; next = a.nbr[2 * (b - 1) + 1]; }
        const bool cut = edge && !(prev == b - 1 && next == b);
        const int stop = 4 + (int)(end - lo);                 // lanes 4 .. stop - 1 are the window's own

        // the link of block eb past its lower or upper end; -1 where it leads
        // nowhere or not back
        auto link_of = [&] (int link, int eb, bool upper) {
            if (link >= 0 && a.nbr[2 * link + (upper ? 0 : 1)] != eb) {
                report_error(a.err, 4, eb, upper ? n : -1);
                return -1;
            }
            return link;
        };
        // lanes before the list and past it hold the guard zones of its first
        // and its last block
        bool ends = false;                                    // at an outflow there
        bool g4 = false, g2 = false;                          // one of four, two next to a block, of a block behind the list
        if (!there) {
            const bool upper = b > 0;
            const int eb = upper ? a.nblk - 1 : 0, over = (b - a.nblk) * n + z;
            const int link = link_of(a.nbr[upper ? 2 * eb + 1 : 0], eb, upper);
            ends = link < 0;
            g4 = link >= a.nblk && (upper ? over : n - 1 - z) < 4;
            g2 = g4 && (upper ? over : n - 1 - z) < 2;
            z = ends ? (upper ? n - 1 : 0) : upper ? min(over, n - 1) : z;
            b = ends ? eb : link;
        }
        // the state is fetched before the links are known (the latencies overlap)
        const size_t at = (size_t)b * NC * n + z;
        double u0[NC], dl = a.dl;
#pragma unroll
        for (int q = 0; q < NC; ++q) u0[q] = a.u[at + (size_t)q * n];
        if (a.dl_blk) dl = a.dl_blk[b];

        const unsigned long long cuts = __ballot(cut), past = __ballot(ends), behind = __ballot(g4);
        int gb = b;                                           // the guard zone that the lane holds for a part
        size_t gat = at;                                      // beside it
        unsigned long long outflow = 0;
        if (__builtin_expect(cuts != 0, 0)) {
            // the cut at or below the lane and the next one above it: within four
            // lanes of one, the lane is beside the part on its other side
            const unsigned long long upto = (2ull << i) - 1, below = cuts & upto, above = cuts & ~upto;
            const int kd = below ? 63 - __builtin_clzll(below) : 0, ku = above ? __builtin_ctzll(above) : 64;
            const bool up = below && i - kd < 4;              // past the end of the part below
            const bool dn = above && ku - 1 - i < 4;
            const int eb = __shfl(b, up ? kd - 1 : ku & 63, 64);      // that part's block
            const int from_below = __shfl(next, kd, 64), from_above = __shfl(prev, ku & 63, 64);
            int link = -1;
            if (up || dn) {
                link = link_of(up ? from_below : from_above, eb, up);
                gb = link < 0 ? eb : link;
                const int gz = link < 0 ? (up ? n - 1 : 0) : (up ? i - kd : n - ku + i);
                gat = (size_t)gb * NC * n + gz;
                if (gb >= a.nblk) { g4 = true; g2 = (up ? i - kd : ku - 1 - i) < 2; }
            }
            outflow = __ballot((up || dn) && link < 0);
        }

        // The two stages of the zones in lanes ka .. kb - 1 (one part, all of
        // them, where nothing is cut), the window's own among them stored.
        for (int ka = 0; ka < stop;) {
            const unsigned long long rest = cuts & ~((2ull << ka) - 1);
            const int kb = rest ? __builtin_ctzll(rest) : 64;
            const int la = ka;
            ka = kb;
            if (kb <= 4) continue;
            const bool in = i >= la && i < kb;
            // the first and the last lane of the part's chain where an outflow is past it
            const int low = la > 0 ? (outflow >> (la - 1) & 1 ? la : 0) : past & 1 ? __builtin_ctzll(~past) : 0;
            const int high = kb < 64 ? (outflow >> kb & 1 ? kb - 1 : 63) : past >> 63 ? 63 - __builtin_clzll(~past) : 63;
            if (cuts) {
                const double* src = a.u + (in ? at : gat);
#pragma unroll
                for (int q = 0; q < NC; ++q) u0[q] = src[(size_t)q * n];
                if (a.dl_blk) dl = a.dl_blk[in ? b : gb];
            }
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

            const bool ok0 = Euler<R>::recover(u0, prm, p);
            face();
#pragma unroll
            for (int q = 0; q < NC; ++q) u1[q] = u0[q] - flux_difference(q) * dtdl;
            const bool ok1 = Euler<R>::recover(u1, prm, p);
            if (cuts || past || behind) {
                // a guard zone behind the list has no lane of its own to report it
                const int near = __shfl(b, in ? (i < 4 ? 4 : stop - 1) : i < la ? la : kb - 1, 64);
                if (g4 && (in ? i < 4 || i >= stop : i >= la - 4 && i < kb + 4) && (!ok0 || (g2 && !ok1)))
                    report_error(a.err, 1, near, i < stop - 1 && i < kb ? 0 : n - 1);
                if (low > 0) {                                // the lanes below take the edge zone's
#pragma unroll
                    for (int q = 0; q < NC; ++q) {
                        const R v = __shfl(p[q], low, 64);
                        if (i < low) p[q] = v;
                    }
                }
                if (high < 63) {                              // and those above the last one's
#pragma unroll
                    for (int q = 0; q < NC; ++q) {
                        const R v = __shfl(p[q], high, 64);
                        if (i > high) p[q] = v;
                    }
                }
            }
            face();
            double wv[NC];
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const double res = u1[q] - flux_difference(q) * dtdl;
                wv[q] = u0[q] * a.rk_b + res * (1.0 - a.rk_b);
            }
            if (in && i >= 4 && i < stop) {
                double* o = a.out + at;
#pragma unroll
                for (int q = 0; q < NC; ++q) o[(size_t)q * n] = wv[q];
                if (!ok0 || !ok1) report_error(a.err, 1, b, z);
                if (a.rate_slot) rate = fmax(rate, Euler<double>::max_speed(wv, prm) * (1.0 / dl));
            }
        }
    }
    if (a.rate_slot) workgroup_atomic_max<64 * kWindowGroup>(rate, a.rate_slot);
}

} // namespace m3p
