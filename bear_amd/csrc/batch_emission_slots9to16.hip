// The batched emission kernels of 9 to 16 stencil slots
#include "batch_emission.h"

namespace bear_amd {

bool launchEmissionSlots9To16(size_t slots, const SpectrumBatch& a) {
  return withSlots<9, 16>(slots, [&](auto ns) { launchEmission<ns>(a); });
}

}  // namespace bear_amd
