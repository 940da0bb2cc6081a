// Kernels of the per-thread system keller_miksis that are held to few registers.
#include "registry.h"
#include "systems/keller_miksis.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::KellerMiksis)
} // namespace pt
} // namespace mpgos
