// Kernels of the per-thread system affine2 that are held to few registers.
#include "registry.h"
#include "systems/affine2.h"

namespace mpgos {
namespace pt {
MPGOS_PT_NARROW_KERNELS(::mpgos::systems::Affine2)
} // namespace pt
} // namespace mpgos
