// Solver and dense-contraction kernel instantiations of the per-block system ring_dw.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_EXTERN(::mpgos::systems::RingDW)
MPGOS_PB_FACTORY(ring_dw, ::mpgos::systems::RingDW)
} // namespace pb
} // namespace mpgos
