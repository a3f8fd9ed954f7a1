// Launches of the batched spectrum kernels by stencil-slot count: the kernels
// of each half of the counts are compiled in a file of their own, so that
// they build in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include "device_math.h"
#include "engine.h"
#include "tile_window.h"

namespace bear_amd {

constexpr int kBatchBlock = 256;
constexpr int kSplitBlock = 512;                 // at most 8 wavefronts share one tile's levels
constexpr int kTransmissionBlock = 512;          // 8 wavefronts share one tile's extinction in LDS

// What a batched spectrum launch takes: the tables and rows of its precision,
// the points' records, the launch shape and the outputs
struct SpectrumBatch {
  TablePrecision precision;
  BatchLaunch shape;
  hipStream_t stream;
  const double* wavenumber;
  const double* wavelength;
  const double* rayleigh;
  const void* tab64;
  const void* tab_low;
  const float* base;
  size_t stride;
  Extras ex;
  bool isothermal;               // DeviceEngine::setIsothermalStencils
  bool extras;                   // the H- rows or the points' cloud models are in use
  dev::Records rec;
  const double* chord;
  const float* chord32;
  int levels, n, batch;
  size_t lds_limit;              // bytes per workgroup
  dev::TileWindow win;
  double* flux;
  bool adjoint;                  // the forward of a gradient call
  float* keep;                   // kept forward quantities (FP64 tables), or none
  int* reach;                    // transmission with keep
};

// false: no such slot count in the range
bool launchEmissionSlots1To8(size_t slots, const SpectrumBatch& a);
bool launchEmissionSlots9To16(size_t slots, const SpectrumBatch& a);
bool launchTransmissionSlots1To8(size_t slots, const SpectrumBatch& a);
bool launchTransmissionSlots9To16(size_t slots, const SpectrumBatch& a);

size_t transmissionBatchLds(int levels, int tile, bool wide, int threads = kTransmissionBlock);

}  // namespace bear_amd
