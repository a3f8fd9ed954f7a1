// The batched transmission kernels of 1 to 8 stencil slots
#include "batch_transmission.h"

namespace bear_amd {

bool launchTransmissionSlots1To8(size_t slots, const SpectrumBatch& a) {
  return withSlots<1, 8>(slots, [&](auto ns) { launchTransmission<ns>(a); });
}

}  // namespace bear_amd
