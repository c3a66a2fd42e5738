// Fused RK2 step of the mixed minidisk scheme.
#include "rk2fused_launch.hpp"

namespace m3p {

template int launch_rk2_fused<MinidiskScheme<float>>(const MinidiskScheme<float>::Params&,
                                                      const MinidiskScheme<float>::Params&,
                                                      const MeshLoader<MinidiskScheme<float>>&, const StageArgs&,
                                                      hipStream_t);

} // namespace m3p
