// The batched emission kernels of 1 to 8 stencil slots
#include "batch_emission.h"

namespace bear_amd {

bool launchEmissionSlots1To8(size_t slots, const SpectrumBatch& a) {
  return withSlots<1, 8>(slots, [&](auto ns) { launchEmission<ns>(a); });
}

}  // namespace bear_amd
