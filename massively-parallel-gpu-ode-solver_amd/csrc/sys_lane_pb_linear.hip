// Lane-per-pair kernel instantiations of the per-block system pb_linear.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_KERNELS(::mpgos::systems::PBLinear)
} // namespace pb
} // namespace mpgos
