// Fused RK2 step of the 1D work-list stage (mixed precision).
#include <climits>
#include "launch.hpp"
#include "rk2fused1d.hpp"

namespace m3p {

int launch_rk2_fused_1d(const EulerParams& prm, const Stage1DArgs& a, hipStream_t s)
{
    const int n = a.n;
    if (n != 16 && n != 32 && n != 64 && n != 128 && (n < 256 || n % 256 != 0))
        return fail(M3P_ERR_BAD_SHAPE, "m3p: 1D block size must be 16, 32, 64, 128 or a multiple of 256 (got " +
                                       std::to_string(n) + ")");
    constexpr long zones = (long)kWindow1D * kWindowGroup;
    const long groups = ((long)a.nblk * n + zones - 1) / zones;
    if (groups > INT_MAX) return fail(M3P_ERR_BAD_SHAPE, "m3p: too many 1D blocks for one launch");
    hipLaunchKernelGGL(rk2_fused_1d_kernel, dim3((unsigned)groups), dim3(64 * kWindowGroup), 0, s, prm, a);
    return launch_status("rk2_fused_1d_kernel");
}

} // namespace m3p
