// Kernels of the per-thread system duffing_dw that are held to few registers.
#include "registry.h"
#include "systems/duffing_dw.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::DuffingDW)
} // namespace pt
} // namespace mpgos
