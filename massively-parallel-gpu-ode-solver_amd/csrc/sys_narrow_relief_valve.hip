// Kernels of the per-thread system relief_valve that are held to few registers.
#include "registry.h"
#include "systems/relief_valve.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::ReliefValve)
} // namespace pt
} // namespace mpgos
