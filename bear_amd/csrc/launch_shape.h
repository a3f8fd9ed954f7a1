// Launch shapes that follow from sizes alone, apart from the kernels, so that
// every size can be checked without a device.
#pragma once

#include <cstddef>

#include "engine.h"

namespace bear_amd {

// LDS of a transit workgroup: the segment extinction sums of its tile
// (S[segment][tile], rows padded to chordSegments) and the partial effective
// heights [threads / tile][tile], FP64
constexpr size_t transitLds(int levels, int tile, int threads) {
  return (size_t(chordSegments(levels)) + size_t(threads / tile)) * size_t(tile) * sizeof(double);
}

// the exponential table in LDS (exp_table.h)
constexpr size_t kExpTableBytes = 128 * 16 * sizeof(double);

// Threads of a workgroup over general stencils: 8 wavefronts share one tile;
// over isothermal ones 16 up to 12 slots (128 registers: beyond that the
// slots' values spill), 8 above.
constexpr int kTransitThreads = 512;
constexpr int isothermalThreads(size_t slots) { return slots <= 12 ? 1024 : kTransitThreads; }

// The single-point transit kernel's form and shape for `levels` levels and
// `slots` stencil slots, within `lds_limit` bytes of LDS.
struct TransitShape {
  bool isothermal;               // two-value stencils: they have no other exponential than the table's
  int threads, tile;             // tile: wavenumbers per workgroup
  int exp_offset;                // of the exponential table in the LDS doubles; 0: no room, no table
  size_t lds;                    // bytes
};

// Isothermal stencils where the model has them and the table fits beside the
// sums of the tile that is launched: tiles of 128 wavenumbers, else of 64;
// otherwise the general stencils, on the wider tile that fits and with the
// table only where there is room beside it.  One transit of 7 slots and 46,935
// wavenumbers, general -> isothermal, per likelihood: 136 levels (tile 128)
// 252 -> 149 us, 150 levels (tile 64) 286 -> 157 us, 200 levels 342 -> 201 us.
constexpr TransitShape transitShape(int levels, size_t slots, bool isothermal, size_t lds_limit) {
  if (isothermal) {
    const int threads = isothermalThreads(slots);
    for (int tile : {128, 64}) {
      const size_t sums = transitLds(levels, tile, threads);
      if (sums + kExpTableBytes <= lds_limit)
        return {true, threads, tile, int(sums / sizeof(double)), sums + kExpTableBytes};
    }
  }
  const int tile = transitLds(levels, 128, kTransitThreads) <= lds_limit ? 128 : 64;
  const size_t sums = transitLds(levels, tile, kTransitThreads);
  if (sums + kExpTableBytes <= lds_limit)
    return {false, kTransitThreads, tile, int(sums / sizeof(double)), sums + kExpTableBytes};
  return {false, kTransitThreads, tile, 0, sums};
}

// Emission: wavefronts that share one tile's levels, by the tiles of a launch:
// 8 up to 8 tiles per CU, 4 up to 16, so that it has 8 to 64 wavefronts per CU,
// else 1, whole columns, which stop where they are opaque.  One point of 100
// levels and 8 slots, us per likelihood in 1 / 2 / 4 / 8 wavefronts per tile:
//    0.7 tiles per CU  187 / 120 /  86 /  72     17.8  321 / 382 / 256 / 270
//    5.9               193 / 205 / 132 / 127     29.7  431 / 562 / 388 / 415
//   11.9               241 / 290 / 191 / 198     47.4  608 / 828 / 586 / 642
// (above 16 per CU 4 wavefronts would still gain 4 to 20 % there; with 14 slots
// 23.7 per CU take 657 / 706 / 663 / 751, with 17.8 634 / 531 / 512 / 583).
constexpr int levelSplit(size_t tiles, int cus) {
  return tiles <= size_t(cus) * 8 ? 8 : tiles <= size_t(cus) * 16 ? 4 : 1;
}

// A launch takes fewer than 2^32 threads in x.  Workgroups at most, in whole
// rounds of the 8 XCDs (device_math.h, workItem).
constexpr size_t maxWorkgroups(int threads) { return ((size_t(1) << 32) - 1) / size_t(threads) / 8 * 8; }

// Live points per launch of a kernel with one workgroup of `threads` per
// (tile, point): larger batches take several launches.
constexpr size_t pointsPerLaunch(int tiles, int threads) {
  const size_t points = maxWorkgroups(threads) / (size_t((tiles + 7) / 8) * 8);
  return points > 0 ? points : 1;
}

}  // namespace bear_amd
