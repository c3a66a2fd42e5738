// Definitions of the stage launchers declared in launch.hpp, included only by
// the k_*.hip units that instantiate them (M3P_INSTANTIATE_* below).
#pragma once
#include <climits>
#include "launch.hpp"
#include "viscous2d.hpp"

namespace m3p {

template<class S, class Ld, bool FIRST>
int launch_stage2d_variant(TileShape ts, const typename S::Params& prm, const Ld& ld, const StageArgs& a, hipStream_t s)
{
    // The mixed kernels keep the conserved state in registers between its load
    // and its update; the FP64 kernels (register-bound) re-load it.
    constexpr bool K = !is_fp64<typename S::Real>::value;
    const int n = a.n;
    auto go = [&] (auto kern, int strips) {
        const int grid = a.nblk * (n / ts.h) * (n / ts.tj);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(ts.tj * strips), 0, s, prm, ld, a);
        return launch_status("stage2d_kernel");
    };
    if (ts.tj == 256 && ts.h == 128) return go(stage2d_kernel<S, Ld, 128, 256, 1, K, FIRST>, 1);
    if (ts.tj == 256 && ts.h == 64) return go(stage2d_kernel<S, Ld, 64, 256, 1, K, FIRST>, 1);
    if (ts.tj == 256 && ts.h == 32) return go(stage2d_kernel<S, Ld, 32, 256, 1, K, FIRST>, 1);
    if (ts.tj == 256 && ts.h == 16) return go(stage2d_kernel<S, Ld, 16, 256, 1, K, FIRST>, 1);
    if (ts.tj == 128 && ts.h == 64) return go(stage2d_kernel<S, Ld, 64, 128, 1, K, FIRST>, 1);
    if (ts.tj == 128 && ts.h == 32) return go(stage2d_kernel<S, Ld, 32, 128, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 64)  return go(stage2d_kernel<S, Ld, 64, 64, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 32)  return go(stage2d_kernel<S, Ld, 32, 64, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 16)  return go(stage2d_kernel<S, Ld, 16, 64, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 8)   return go(stage2d_kernel<S, Ld, 8, 64, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 4)   return go(stage2d_kernel<S, Ld, 4, 64, 1, K, FIRST>, 1);
    if (ts.tj == 64 && ts.h == 2)   return go(stage2d_kernel<S, Ld, 2, 64, 1, K, FIRST>, 1);
    if (ts.tj == 32 && ts.h == 32)  return go(stage2d_kernel<S, Ld, 32, 32, 2, K, FIRST>, 2);
    if (ts.tj == 32 && ts.h == 16)  return go(stage2d_kernel<S, Ld, 16, 32, 2, K, FIRST>, 2);
    if (ts.tj == 32 && ts.h == 8)   return go(stage2d_kernel<S, Ld, 8, 32, 2, K, FIRST>, 2);
    if (ts.tj == 32 && ts.h == 4)   return go(stage2d_kernel<S, Ld, 4, 32, 2, K, FIRST>, 2);
    if (ts.tj == 16 && ts.h == 16)  return go(stage2d_kernel<S, Ld, 16, 16, 4, K, FIRST>, 4);
    if (ts.tj == 16 && ts.h == 8)   return go(stage2d_kernel<S, Ld, 8, 16, 4, K, FIRST>, 4);
    return fail(M3P_ERR_BAD_SHAPE, "m3p: 2D block size must be 16, 32 or a multiple of 64 (got " + std::to_string(n) + ")");
}

template<class S, class Ld>
int launch_stage2d_shape(TileShape ts, const typename S::Params& prm, const Ld& ld, const StageArgs& a, hipStream_t s)
{
    // A stage without a base state has its own kernels only where the scheme
    // fetches more rows ahead there (and the loader pipelines its rows).
    if constexpr (S::kFirstStage && Ld::kPrefetch)
        if (!a.u0) return launch_stage2d_variant<S, Ld, true>(ts, prm, ld, a, s);
    return launch_stage2d_variant<S, Ld, false>(ts, prm, ld, a, s);
}

template<class S, class Ld>
int launch_visc(const typename S::Params& prm, const Ld& ld, const StageArgs& a, double nu, hipStream_t s)
{
    if (a.n < 1) return fail(M3P_ERR_BAD_SHAPE, "m3p: 2D block size must be positive (got " + std::to_string(a.n) + ")");
    const int tiles = (a.n + kViscTile - 1) / kViscTile;
    hipLaunchKernelGGL((iso_visc_stage_kernel<S, Ld, kViscTile>), dim3(a.nblk * tiles * tiles),
                       dim3(kViscTile * kViscTile), 0, s, prm, ld, a, nu);
    return launch_status("iso_visc_stage_kernel");
}

template<typename R>
int launch_stage1d(const EulerParams& prm, const Stage1DArgs& a, hipStream_t s)
{
    const int n = a.n;
    if (n != 16 && n != 32 && n != 64 && n != 128 && (n < 256 || n % 256 != 0))
        return fail(M3P_ERR_BAD_SHAPE, "m3p: 1D block size must be 16, 32, 64, 128 or a multiple of 256 (got " + std::to_string(n) + ")");
    constexpr long zones = (long)kWindowStage1D * kWindowGroup;
    const long groups = ((long)a.nblk * n + zones - 1) / zones;
    if (groups > INT_MAX) return fail(M3P_ERR_BAD_SHAPE, "m3p: too many 1D blocks for one launch");
    hipLaunchKernelGGL(stage1d_kernel<R>, dim3((unsigned)groups), dim3(64 * kWindowGroup), 0, s, prm, a);
    return launch_status("stage1d_kernel");
}

} // namespace m3p

#define M3P_INSTANTIATE_STAGE2D(S, LD) \
    template int m3p::launch_stage2d_shape<S, LD<S>>(m3p::TileShape, const typename S::Params&, const LD<S>&, \
                                                    const m3p::StageArgs&, hipStream_t);
#define M3P_INSTANTIATE_VISC(S, LD) \
    template int m3p::launch_visc<S, LD<S>>(const typename S::Params&, const LD<S>&, const m3p::StageArgs&, \
                                           double, hipStream_t);
