// Batched emission and eclipse spectra: the kernels and their launch by
// precision.
#pragma once

#include "batch_launch.h"
#include "emission_sweep.h"
#include "reduced_opacity.h"

namespace bear_amd {

using namespace dev;

namespace {

// Fused opacity + two-angle short characteristics per (wavenumber, point)
// (emission_sweep.h): the flux F = 2 pi sum mu w I 1e-3 scaling goes to
// flux[point][i].  A workgroup is blockDim wavenumbers of one point, each
// wavefront sweeping its columns from the top down to where they are opaque,
// one item per workgroup: the items' costs differ with their opacity, and the
// dispatcher levels them (a persistent grid that walked the items held more
// registers, spilled, and was 1.17x slower at 64 points of 8 species, 1.48x at
// 192 of 14 on FP16 tables);
// kSplit: 64 wavenumbers of one point with the levels split over the
// workgroup's wavefronts.
// EX (FP64 tables): the H- continuum joins each level's opacity and the
// point's cloud models (BatchModel::clouds, weights in its LevelState) each
// layer's optical depth, as in the single-point kernel.
template <class Op, bool EX, bool kSplit>
__global__ __launch_bounds__((kSplit ? kSplitBlock : kBatchBlock), (sweepWaves<Op, EX>())) void emissionBatchKernel(
    const double* __restrict__ wavenumber, const double* __restrict__ wavelength, const void* __restrict__ tables,
    const float* __restrict__ base, size_t stride, Extras ex, Records rec, int nb_levels, int n, int tiles, int batch,
    double* __restrict__ flux) {
  using Species = typename Op::Species;
  extern __shared__ double part[];                      // kSplit: splitPart
  __shared__ double exp_table[kExpTable];
  int m, tile;
  if (!workItem(blockIdx.x, batch, tiles, m, tile)) return;       // uniform over the workgroup
  fillExpTable(exp_table);
  const int at = kSplit ? tile * 64 + int(threadIdx.x & 63) : tile * int(blockDim.x) + int(threadIdx.x);
  if (!kSplit && at >= n) return;
  const int i = kSplit ? min(at, n - 1) : at;         // idle lanes of a split tile follow its last column
  const unsigned char* r = rec.at(m);
  const BatchModel* bm = reinterpret_cast<const BatchModel*>(r);
  const LevelState* levels = reinterpret_cast<const LevelState*>(r + rec.levels);
  const Species* species = reinterpret_cast<const Species*>(r + rec.species);
  Op op;
  op.init(tables, base, stride, i, expCopy(exp_table));
  const Column col = columnAt(expCopy(exp_table), wavenumber[i], bm->min_inv_temperature);
  Extras e = ex;
  double hm[7], cf[kMaxClouds];
  if constexpr (EX) {
    e.clouds = bm->clouds;
    loadExtras(e, i, n, wavelength[i], hm, cf);
  }
  LayerRun run;
  double b_top;
  if constexpr (kSplit) {
    run = sweepSplit<Op, EX>(op, species, levels, rec.groups, nb_levels, col, e, hm, cf, i, n, part, b_top);
    if (threadIdx.x < 64 && at < n)
      flux[size_t(m) * stride + i] = columnFlux(b_top + run.s1, b_top + run.s2, bm->scaling);
  } else {
    run = sweepColumn<Op, EX>(op, species, levels, rec.groups, nb_levels, col, e, hm, cf, i, n, b_top);
    flux[size_t(m) * stride + i] = columnFlux(b_top + run.s1, b_top + run.s2, bm->scaling);
  }
}

// The same from the bottom up for the gradient calls, with every level's
// forward quantities kept for the adjoint's backward sweep (unless it
// recomputes them: keep null, the same flux to the last bit): both angles' intensity less the level's
// Planck function, D = I - B, and the opacity go to keep (keptColumn layout)
// in FP32 (the backward sweep recomputes B in FP64: the difference it needs
// keeps its own relative precision, and the gradient's bar is 1e-4).
template <class Op, bool EX>
__global__ __launch_bounds__((kBatchBlock), (sweepWaves<Op, EX>())) void emissionKeptKernel(
    const double* __restrict__ wavenumber, const double* __restrict__ wavelength, const void* __restrict__ tables,
    size_t stride, Extras ex, Records rec, int nb_levels, int n, int tiles, int batch, double* __restrict__ flux,
    float* __restrict__ keep) {
  using Species = typename Op::Species;
  __shared__ double exp_table[kExpTable];
  int m, tile;
  if (!workItem(blockIdx.x, batch, tiles, m, tile)) return;
  fillExpTable(exp_table);
  const int i = tile * int(blockDim.x) + int(threadIdx.x);
  if (i >= n) return;
  const unsigned char* r = rec.at(m);
  const BatchModel* bm = reinterpret_cast<const BatchModel*>(r);
  const LevelState* levels = reinterpret_cast<const LevelState*>(r + rec.levels);
  const Species* species = reinterpret_cast<const Species*>(r + rec.species);
  Op op;
  op.init(tables, nullptr, stride, i, expCopy(exp_table));
  const Column col = columnAt(expCopy(exp_table), wavenumber[i], 1.0);
  Extras e = ex;
  double hm[7], cf[kMaxClouds];
  if constexpr (EX) {
    e.clouds = bm->clouds;
    loadExtras(e, i, n, wavelength[i], hm, cf);
  }
  op.load(species, levels[0], rec.groups);
  double k_prev = op.form(species, levels[0], rec.groups);
  if (EX && e.hminus) k_prev = withHminus(k_prev, hm, levels[0]);
  double b_prev = col.planck(levels[0]), d1 = 0.0, d2 = 0.0;       // I = B at the bottom
  float* kept = keep + keptColumn(m, stride, nb_levels, i);
  if (keep) {
    kept[0] = 0.0f;
    kept[kKeptValue] = 0.0f;
    kept[2 * kKeptValue] = float(k_prev);
  }
  for (int l = 1; l < nb_levels; ++l) {
    const Species* d = species + size_t(l) * Op::kNS;
    if (levels[l].reload) op.load(d, levels[l], rec.groups);
    double k_next = op.form(d, levels[l], rec.groups);
    if (EX && e.hminus) k_next = withHminus(k_next, hm, levels[l]);
    const double b_next = col.planck(levels[l]);
    double tau = levels[l].half_dz * (k_next + k_prev);
    if (EX) tau += cloudLayer(e, cf, levels[l], l, i, n);
    addLayerAbove(col.copy, tau, b_next - b_prev, d1, d2);
    if (keep) {
      float* out = kept + size_t(l) * kKeptLevel;
      out[0] = float(d1);
      out[kKeptValue] = float(d2);
      out[2 * kKeptValue] = float(k_next);
    }
    k_prev = k_next;
    b_prev = b_next;
  }
  flux[size_t(m) * stride + i] = columnFlux(b_prev + d1, b_prev + d2, bm->scaling);
}

template <class Op, bool EX>
void launchEmissionSweep(const SpectrumBatch& a, const void* tab) {
  const BatchLaunch& lc = a.shape;
  const int tiles = (a.n + lc.tile - 1) / lc.tile;
  const dim3 grid{unsigned(nbItems(tiles, a.batch))}, block{unsigned(lc.block)};
  if (lc.split > 1)
    hipLaunchKernelGGL((emissionBatchKernel<Op, EX, true>), grid, block, splitPart(lc.split) * sizeof(double),
                       a.stream, a.wavenumber, a.wavelength, tab, a.base, a.stride, a.ex, a.rec, a.levels, a.n, tiles,
                       a.batch, a.flux);
  else
    hipLaunchKernelGGL((emissionBatchKernel<Op, EX, false>), grid, block, 0, a.stream, a.wavenumber, a.wavelength, tab,
                       a.base, a.stride, a.ex, a.rec, a.levels, a.n, tiles, a.batch, a.flux);
}

template <class Op, bool EX>
void launchEmissionKept(const SpectrumBatch& a) {        // FP64 tables, tiles of whole workgroups
  const int tiles = (a.n + a.shape.block - 1) / a.shape.block;
  hipLaunchKernelGGL((emissionKeptKernel<Op, EX>), dim3(unsigned(nbItems(tiles, a.batch))), dim3(unsigned(a.shape.block)), 0,
                     a.stream, a.wavenumber, a.wavelength, a.tab64, a.stride, a.ex, a.rec, a.levels, a.n, tiles,
                     a.batch, a.flux, a.keep);
}

template <int NS>
void launchEmission(const SpectrumBatch& a) {
  if (a.adjoint && a.extras) return launchEmissionKept<Opacity64<NS>, true>(a);
  if (a.adjoint) return launchEmissionKept<Opacity64<NS>, false>(a);
  switch (a.precision) {
    case TablePrecision::fp64:
      return a.extras ? launchEmissionSweep<Opacity64<NS>, true>(a, a.tab64)
                      : launchEmissionSweep<Opacity64<NS>, false>(a, a.tab64);
    case TablePrecision::fp32:
      return launchEmissionSweep<Opacity32<NS, TabF32>, false>(a, a.tab_low);
    case TablePrecision::fp16:
      return launchEmissionSweep<Opacity32<NS, TabF16>, false>(a, a.tab_low);
    case TablePrecision::bf16:
      return launchEmissionSweep<Opacity32<NS, TabBF16>, false>(a, a.tab_low);
    case TablePrecision::int16:
      return launchEmissionSweep<Opacity32<NS, TabS16>, false>(a, a.tab_low);
  }
}

}  // namespace
}  // namespace bear_amd
