// Lane-per-pair kernel instantiations of the per-block system ring_duffing.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_KERNELS(::mpgos::systems::RingDuffing)
} // namespace pb
} // namespace mpgos
