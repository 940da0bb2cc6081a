// Solver and dense-contraction kernel instantiations of the per-block system ring_duffing.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_EXTERN(::mpgos::systems::RingDuffing)
MPGOS_PB_FACTORY(ring_duffing, ::mpgos::systems::RingDuffing)
} // namespace pb
} // namespace mpgos
