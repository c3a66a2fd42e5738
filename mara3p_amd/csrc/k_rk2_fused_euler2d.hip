// Fused RK2 step of the mixed euler2d scheme.
#include "rk2fused_launch.hpp"

namespace m3p {

template int launch_rk2_fused<EulerScheme<float>>(const EulerScheme<float>::Params&,
                                                   const EulerScheme<float>::Params&,
                                                   const MeshLoader<EulerScheme<float>>&, const StageArgs&,
                                                   hipStream_t);

} // namespace m3p
