// The batched transmission kernels of 9 to 16 stencil slots
#include "batch_transmission.h"

namespace bear_amd {

bool launchTransmissionSlots9To16(size_t slots, const SpectrumBatch& a) {
  return withSlots<9, 16>(slots, [&](auto ns) { launchTransmission<ns>(a); });
}

}  // namespace bear_amd
