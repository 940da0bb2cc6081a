// Solver and dense-contraction kernel instantiations of the per-block system pb_linear.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_EXTERN(::mpgos::systems::PBLinear)
MPGOS_PB_FACTORY(pb_linear, ::mpgos::systems::PBLinear)
} // namespace pb
} // namespace mpgos
