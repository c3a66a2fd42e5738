// Launcher of the fused RK2 step (rk2fused.hpp), included by the units that
// instantiate it (one scheme each: large kernels).
#pragma once
#include "launch.hpp"
#include "rk2fused.hpp"

namespace m3p {

// The rows of a workgroup by the size of the mesh.  A workgroup marches
// H + 5 steps in series, so a mesh that does not fill the device is bound by
// them: 512^2 zones and less take 4 rows (minidisk 20 us a step, 75 with 32;
// euler2d 27 to 30, 120), 1024^2 take 8 (34 to 41 us against 42 to 46 with 4
// and 73 to 79 with 32; euler2d 52 to 61, 67 to 73, 111 to 129).  Meshes that
// fill it want the fewest extra rows (four of the first stage per workgroup):
// 32 (4096^2 in 256^2 blocks: minidisk 323 us, 346 with 16; 64 rows need
// about 55 KB of LDS and run 14 % slower), but 16 in blocks of 64, whose
// one-wave workgroups then share the work more evenly (2048^2: euler2d 190 us
// against 302 with 32, minidisk 116 with either; 4096^2: 738 against 799, 419
// against 448).
template<class S>
int launch_rk2_fused(const typename S::Params& p1, const typename S::Params& p2, const MeshLoader<S>& ld,
                     const StageArgs& a, hipStream_t s)
{
    const double zones = (double)a.nblk * a.n * a.n;
    const int rows = zones / (64 * 8) < 2048 ? 4 : zones / (64 * 16) < 4096 ? 8 : a.n == 64 ? 16 : 32;
    auto go = [&] (auto kern) {
        hipLaunchKernelGGL(kern, dim3(a.nblk * (a.n / rows)), dim3(a.n), 0, s, p1, p2, ld, a);
        return launch_status("rk2_fused_kernel");
    };
    switch (a.n) {
        case 64:
            if (rows == 4) return go(rk2_fused_kernel<S, 4, 64>);
            if (rows == 8) return go(rk2_fused_kernel<S, 8, 64>);
            return go(rk2_fused_kernel<S, 16, 64>);
        case 128:
            if (rows == 4) return go(rk2_fused_kernel<S, 4, 128>);
            if (rows == 8) return go(rk2_fused_kernel<S, 8, 128>);
            return go(rk2_fused_kernel<S, 32, 128>);
        case 256:
            if (rows == 4) return go(rk2_fused_kernel<S, 4, 256>);
            if (rows == 8) return go(rk2_fused_kernel<S, 8, 256>);
            return go(rk2_fused_kernel<S, 32, 256>);
    }
    return fail(M3P_ERR_BAD_SHAPE, "m3p: the fused RK2 step takes blocks of 64, 128 or 256 zones a side (got " +
                                   std::to_string(a.n) + ")");
}

} // namespace m3p
