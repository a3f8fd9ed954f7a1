// Emission radiative transfer of one column (one wavenumber of one live
// point), shared by the single-point and the batched kernels.
//
// Bound: FP64 vector instructions (batches, about 80 % of their issue time),
// latency of the level records and row reloads (small launches, single
// points).  Hence columns from the top down, so that the levels below the
// photosphere are never evaluated; D = I - B, which needs two operations per
// angle and layer; and levels split over wavefronts when the tiles alone do
// not fill the chip.  Measured before -> after, all of it together: one point
// of 20,000 wavenumbers, 60 levels, 2 species 114 -> 47 us; 64 points of
// 99,777, 100 levels, 8 species 6.6 -> 4.3 ms; 192 points of 300,000, 14
// species on FP16 tables 62 -> 29 ms.
#pragma once

#include "opacity64.h"

namespace bear_amd {
namespace dev {

// Two-angle short characteristics (short_characteristics.cpp:88-114),
//   I_l = a I_{l-1} + (1 + q) B_l + (-a - q) B_{l-1},
//   a = e^(-tau / mu), q = (a - 1) mu / tau,
// written for D = I - B, for which a layer is D_l = a D_{l-1} + q (B_l -
// B_{l-1}): two operations per angle after q instead of eight.  A run of
// layers is then the map D -> A D + S with A = prod a and, from its top
// down, S = sum over its layers of (prod of a above) q (B_l - B_{l-1}).
struct LayerRun {
  double a1 = 1.0, s1 = 0.0, a2 = 1.0, s2 = 0.0;
};

// The attenuation factor and q of one angle; r = 1 / tau
__device__ __forceinline__ void attenuation(const double* __restrict__ copy, double tau, double r, double mu, double& a,
                                            double& q) {
  a = tablePow2(copy, tau * (-kLog2E * kExpSteps / mu));
  q = (a - 1.0) * (mu * r);
}

__device__ __forceinline__ void addLayerBelow(const double* __restrict__ copy, double tau, double db, LayerRun& c) {
  if (tau != 0) {
    const double r = recip(tau);
    double a, q;
    attenuation(copy, tau, r, kMu1, a, q);
    c.s1 = fma(c.a1, q * db, c.s1);
    c.a1 *= a;
    attenuation(copy, tau, r, kMu2, a, q);
    c.s2 = fma(c.a2, q * db, c.s2);
    c.a2 *= a;
  } else {                                             // the intensity passes unchanged: a = 1, q = -1
    c.s1 = fma(c.a1, -db, c.s1);
    c.s2 = fma(c.a2, -db, c.s2);
  }
}

// the same layer from below, for the kernels that keep every level's D
__device__ __forceinline__ void addLayerAbove(const double* __restrict__ copy, double tau, double db, double& d1,
                                              double& d2) {
  if (tau != 0) {
    const double r = recip(tau);
    double a, q;
    attenuation(copy, tau, r, kMu1, a, q);
    d1 = fma(a, d1, q * db);
    attenuation(copy, tau, r, kMu2, a, q);
    d2 = fma(a, d2, q * db);
  } else {
    d1 -= db;
    d2 -= db;
  }
}

// The layers are taken in kRuns runs fixed by the number of levels alone, and
// the runs' maps joined from the top down, whichever wavefronts computed
// them: so a column's flux has the same bits in every launch shape.
constexpr int kRuns = 16;
__device__ __forceinline__ int runTop(int nb_levels, int run) { return nb_levels - 1 - run * (nb_levels - 1) / kRuns; }

// Below a level with attenuation a above it, nothing reaches the top but
// a (I_l - B_l) with 0 <= I_l, B_l <= B of the column's hottest level.  Once
// that is under 2^-60 of both angles' sums so far, no layer below can change
// a bit of them: the column is done.  kExitScale = 2^60.
constexpr double kExitScale = 1152921504606846976.0;

struct Column {
  const double* copy;          // this lane's copy of the exponential table
  double b_num, x_nu;          // Planck function: numerator and exponent per 1 / T
  double b_exit;               // kExitScale B of the hottest level

  __device__ __forceinline__ double planck(const LevelState& lev) const {
    return planckTable(copy, b_num, x_nu, lev.inv_temperature);
  }
};

__device__ __forceinline__ Column columnAt(const double* copy, double nu, double min_inv_t) {
  Column c;
  c.copy = copy;
  c.b_num = kPlanckC1 * nu * nu * nu;
  c.x_nu = -(6.62606896e-27 * nu * 2.99792458e10 / 1.3806504e-16) * kLog2E;
  c.b_exit = planckAt(c.b_num, c.x_nu, min_inv_t) * kExitScale;
  return c;
}

// The runs [first, end) of a column from the top down: fused opacity (Op: load
// the stencil rows of a level, form its kappa from them) and transfer, kappa
// and the run in registers; emit(run index, run) after each, false to stop.
// The rows are loaded only where they change from one level to the next.
// Returns the Planck function of the top level.
template <class Op, bool EX, class Emit>
__device__ __forceinline__ double sweepDown(Op& op, const typename Op::Species* __restrict__ species,
                                            const LevelState* __restrict__ levels, StencilGroups groups, int nb_levels,
                                            int first, int end, const Column& col, const Extras& e,
                                            const double (&hm)[7], const double (&cf)[kMaxClouds], int i, int n,
                                            Emit&& emit) {
  const int ns = op.slots();
  auto level = [&](int l) { return species + size_t(l) * ns; };
  auto form = [&](int l) {
    const double k = double(op.form(level(l), levels[l], groups));
    return EX && e.hminus ? withHminus(k, hm, levels[l]) : k;
  };
  int l = runTop(nb_levels, first);
  op.load(level(l), levels[l], groups);
  double k_hi = form(l);
  const double b_top = col.planck(levels[l]);
  double b_hi = b_top;
  for (int r = first; r < end; ++r) {
    const int bottom = runTop(nb_levels, r + 1);
    LayerRun run;
    for (; l > bottom; --l) {
      if (levels[l].reload) op.load(level(l - 1), levels[l - 1], groups);
      const double k_lo = form(l - 1);
      const double b_lo = col.planck(levels[l - 1]);
      double tau = levels[l].half_dz * (k_hi + k_lo);
      if (EX) tau += cloudLayer(e, cf, levels[l], l, i, n);
      addLayerBelow(col.copy, tau, b_hi - b_lo, run);
      k_hi = k_lo;
      b_hi = b_lo;
    }
    if (!emit(r, run)) break;
  }
  return b_top;
}

// both angles' attenuation and sums of the runs above and of the next below
__device__ __forceinline__ void joinBelow(LayerRun& all, const LayerRun& run) {
  all.s1 = fma(all.a1, run.s1, all.s1);
  all.a1 *= run.a1;
  all.s2 = fma(all.a2, run.s2, all.s2);
  all.a2 *= run.a2;
}

// A whole column by its own lane, from the top down to where it is opaque for
// the whole wavefront.  Of 100 levels between 1e2 and 1e-6 bar, 10 to 25 % are
// never evaluated that way; from the bottom up all of them would be.
template <class Op, bool EX>
__device__ __forceinline__ LayerRun sweepColumn(Op& op, const typename Op::Species* __restrict__ species,
                                                const LevelState* __restrict__ levels, StencilGroups groups,
                                                int nb_levels, const Column& col, const Extras& e,
                                                const double (&hm)[7], const double (&cf)[kMaxClouds], int i, int n,
                                                double& b_top) {
  LayerRun all;
  b_top = sweepDown<Op, EX>(op, species, levels, groups, nb_levels, 0, kRuns, col, e, hm, cf, i, n,
                                    [&](int, const LayerRun& run) {
                                      joinBelow(all, run);
                                      const bool done =
                                          all.a1 * col.b_exit <= fabs(all.s1) && all.a2 * col.b_exit <= fabs(all.s2);
                                      return __builtin_amdgcn_ballot_w64(!done) != 0;
                                    });
  return all;
}

// Wavefronts per SIMD to compile for: what the cached rows (and the extras'
// per-column values) leave of the 512 vector registers.  Left to itself the
// compiler overlaps more slots and drops a wavefront.
template <class Op, bool EX>
constexpr int sweepWaves() {
  const int cached = Op::kNS * (sizeof(typename Op::K) == 8 ? 8 : Op::kScaled ? 6 : 5) + (EX ? 22 : 0);
  return cached + 58 <= 128 ? 4 : cached + 58 <= 168 ? 3 : 2;
}

// F = 2 pi (mu1 w I1 + mu2 w I2) 1e-3 scaling (short_characteristics.cpp:117-122)
__device__ __forceinline__ double columnFlux(double i1, double i2, double scaling) {
  return 2.0 * kPi * (i1 * kMu1 * kW + i2 * kMu2 * kW) * 1e-3 * scaling;
}

// One tile of 64 wavenumbers with its levels split over the workgroup's
// wavefronts (2, 4 or 8), for launches of too few tiles to fill the chip (20,000
// wavenumbers are 313 wavefronts for 1,024 SIMDs, each a chain of levels): each
// sweeps its share of the runs (the boundary levels' opacity is formed on both
// sides); the first joins its own as it goes and then the others' from LDS
// (part [runs of the others][4][64]).  The joined column in wavefront 0.
template <class Op, bool EX>
__device__ __forceinline__ LayerRun sweepSplit(Op& op, const typename Op::Species* __restrict__ species,
                                               const LevelState* __restrict__ levels, StencilGroups groups,
                                               int nb_levels, const Column& col, const Extras& e,
                                               const double (&hm)[7], const double (&cf)[kMaxClouds], int i, int n,
                                               double* __restrict__ part, double& b_top) {
  const int share = kRuns * 64 / int(blockDim.x);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 64), lane = int(threadIdx.x) & 63;
  LayerRun all;
  b_top = sweepDown<Op, EX>(op, species, levels, groups, nb_levels, wave * share, (wave + 1) * share, col, e,
                                    hm, cf, i, n, [&](int r, const LayerRun& run) {
                                      if (wave == 0) {
                                        joinBelow(all, run);
                                      } else {
                                        double* p = part + size_t(r - share) * 4 * 64 + lane;
                                        p[0] = run.a1;
                                        p[64] = run.s1;
                                        p[128] = run.a2;
                                        p[192] = run.s2;
                                      }
                                      return true;
                                    });
  __syncthreads();
  if (wave == 0)
    for (int r = share; r < kRuns; ++r) {
      const double* p = part + size_t(r - share) * 4 * 64 + lane;
      joinBelow(all, LayerRun{p[0], p[64], p[128], p[192]});
    }
  return all;
}
// LDS doubles of part for `split` wavefronts
constexpr int splitPart(int split) { return (kRuns - kRuns / split) * 4 * 64; }

}  // namespace dev
}  // namespace bear_amd
