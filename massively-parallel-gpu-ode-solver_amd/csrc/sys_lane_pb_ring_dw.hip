// Lane-per-pair kernel instantiations of the per-block system ring_dw.
#include "registry.h"
#include "systems/pb_ring.h"

namespace mpgos {
namespace pb {
MPGOS_PB_LANE_KERNELS(::mpgos::systems::RingDW)
} // namespace pb
} // namespace mpgos
