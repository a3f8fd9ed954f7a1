// The FP64 opacity of a level as an object of the forward kernels: load a
// level's rows, form its kappa from the rows held.
#pragma once

#include "exp_table.h"

namespace bear_amd {
namespace dev {

// NS register-cached slots, the powers of two from the LDS table; kTable
// false: the table only where there is one, else the octave polynomial.
template <int NS, bool kTable = true>
struct Opacity64 {
  static constexpr int kNS = NS;
  static constexpr bool kScaled = false;
  using Species = LevelSpecies;
  using K = double;
  const double* tab;
  unsigned i;
  const double* copy;                                   // this lane's copy of the exponential table
  double v[NS][4];
  __device__ __forceinline__ void init(const void* tables, const float*, size_t, int at, const double* exp_copy) {
    tab = static_cast<const double*>(tables);
    i = unsigned(at);
    copy = exp_copy;
  }
  __device__ __forceinline__ int slots() const { return NS; }
  __device__ __forceinline__ void load(const LevelSpecies* d, const LevelState&, StencilGroups) {
    loadRows<NS>(tab, i, d, v);
  }
  __device__ __forceinline__ double form(const LevelSpecies* d, const LevelState& lev, StencilGroups groups) const {
    if (!kTable && !copy) return kappaFrom<NS>(v, d, lev, groups);
    double k = 0.0;
    if (groups.grouped) {
      double a[4], b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[q] = lev.table_w[0][q];
        b[q] = lev.table_w[1][q];
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        double x = lev.table_n[s];
#pragma unroll
        for (int q = 0; q < 4; ++q) x = fma(groupWeight<NS>(a, b, groups, s, q), v[s][q], x);
        k = addPow2(k, copy, x);
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        double x = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) x = fma(d[s].w[q], v[s][q], x);
        k = addPow2(k, copy, fma(x, double(kExpSteps), lev.table_n[s]));
      }
    }
    return k;
  }
};

// The same for isothermal stencils (grouped; DeviceEngine::
// setIsothermalStencils): the fraction between the temperature rows is the
// same at every level, so a row pair is interpolated in T once, when it is
// loaded, and a slot keeps its value at the lower pressure row and the step
// to the upper one, in the table's units.  Half the registers, which lets 16
// wavefronts share a tile of 200 levels where 8 could, and two operations per
// slot and level fewer.  The launch has to bring the table (exp_copy not
// null): transitShape and launchTransmission take this form only where it fits.
template <int NS>
struct Opacity64Isothermal {
  static constexpr int kNS = NS;
  static constexpr bool kScaled = false;
  using Species = LevelSpecies;
  using K = double;
  const double* tab;
  unsigned i;
  const double* copy;
  double u[NS], du[NS];
  __device__ __forceinline__ void init(const void* tables, const float*, size_t, int at, const double* exp_copy) {
    tab = static_cast<const double*>(tables);
    i = unsigned(at);
    copy = exp_copy;
  }
  __device__ __forceinline__ void load(const LevelSpecies* d, const LevelState& lev, StencilGroups groups) {
    constexpr double kUnit = kLog2Ten * kExpSteps;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = (tab + (size_t(d[s].block[q]) << 6))[i];
      const double ft = groupValue<NS>(lev.fraction_t[0], lev.fraction_t[1], groups, s);
      const double lo = fma(ft, v[2] - v[0], v[0]), hi = fma(ft, v[3] - v[1], v[1]);
      u[s] = lo * kUnit;
      du[s] = (hi - lo) * kUnit;
    }
  }
  __device__ __forceinline__ double form(const LevelSpecies*, const LevelState& lev, StencilGroups groups) const {
    double k = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double fp = groupValue<NS>(lev.fraction_p[0], lev.fraction_p[1], groups, s);
      k = addPow2(k, copy, fma(fp, du[s], u[s] + lev.table_n[s]));
    }
    return k;
  }
};

// any number of species in chunks, nothing held between levels
struct OpacityChunked {
  using Species = LevelSpecies;
  using K = double;
  const double* tab;
  unsigned i;
  int nb_chunks;
  __device__ __forceinline__ int slots() const { return nb_chunks * kChunk; }
  __device__ __forceinline__ void load(const LevelSpecies*, const LevelState&, StencilGroups) {}
  __device__ __forceinline__ double form(const LevelSpecies* d, const LevelState& lev, StencilGroups) const {
    return chunkedKappa(tab, i, d, lev, nb_chunks);
  }
};

}  // namespace dev
}  // namespace bear_amd
