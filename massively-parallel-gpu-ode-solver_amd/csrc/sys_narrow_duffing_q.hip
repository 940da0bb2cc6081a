// Kernels of the per-thread system duffing_q that are held to few registers.
#include "registry.h"
#include "systems/duffing.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::DuffingQ)
} // namespace pt
} // namespace mpgos
