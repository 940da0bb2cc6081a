// Kernels of the per-thread system lorenz that are held to few registers.
#include "registry.h"
#include "systems/lorenz.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::Lorenz)
} // namespace pt
} // namespace mpgos
