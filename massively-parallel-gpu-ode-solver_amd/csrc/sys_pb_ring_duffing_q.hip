// Solver and dense-contraction kernel instantiations of the per-block system ring_duffing_q.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_EXTERN(::mpgos::systems::RingDuffingQ)
MPGOS_PB_FACTORY(ring_duffing_q, ::mpgos::systems::RingDuffingQ)
} // namespace pb
} // namespace mpgos
