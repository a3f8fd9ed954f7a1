// Batched transit spectra: the kernel and its launch by precision.
#pragma once

#include <algorithm>

#include "batch_launch.h"
#include "launch_shape.h"
#include "opacity64.h"
#include "reduced_opacity.h"

namespace bear_amd {

using namespace dev;

namespace {

__device__ __forceinline__ double transmittance(double tau) { return pow2(-tau * kLog2E); }
__device__ __forceinline__ double transmittance(float tau) {
  return double(__builtin_amdgcn_exp2f(-tau * 1.44269504088896340736f));
}

// Transit depth per (wavenumber, point) (transmission_spectrum.cpp:32-154).
// One work item = `tile` wavenumbers of one point:
//  1. extinction k_l (Op::K: FP64 or FP32), threads split over level ranges
//     with register-cached stencils, stored as the segment sums
//     S[q] = k_q + k_{q+1} in LDS (across a group boundary after the first
//     barrier, from the next group's first level);
//  2. blocks of eight tangent levels per thread group (tangentBlock: tau
//     summed outward in the reference's order, stopping at the first sum
//     above 10); each path adds c_t (1 - e^-tau) to its thread's FP64
//     partial, where c_t = (R+z_t)(z_{t+1} - z_{t-1}) is the coefficient of
//     (1 - T_t) in the reference's trapezoid (one-sided at t = 0; T = 1 at
//     the top level);
//  3. per wavenumber, the partials in a fixed order, h = sqrt(H + R^2) - R
//     and depth (R + h)^2 / R_*^2 1e6 in FP64.
// kKeep (FP64 tables, for the adjoint): also, in the keptColumn layout,
// {k_l, tau_t, last segment summed by path t} per level in FP32.
// EX (FP64 tables): the H- continuum and the point's cloud extinction
// (BatchModel::clouds, the layer below each level over its thickness) join
// each level's extinction, as in the single-point kernel.
template <class Op, int kThreads, bool kKeep = false, bool EX = false>
__global__ __launch_bounds__(kThreads) void transmissionBatchKernel(
    const void* __restrict__ tables, const float* __restrict__ base, size_t stride, const double* __restrict__ rayleigh,
    const double* __restrict__ wavelength, Extras ex, Records rec, const double* __restrict__ chord64,
    const float* __restrict__ chord32, int nb_levels, int n, TileWindow win, int tile, int batch, int point_group,
    double* __restrict__ depth, float* __restrict__ keep, int* __restrict__ reach, int exp_offset) {
  using K = typename Op::K;
  using Species = typename Op::Species;
  extern __shared__ double lds[];
  // the exponential table where the levels leave room for it (FP64 tables)
  const double* exp_copy = nullptr;
  if constexpr (sizeof(typename Op::K) == 8)
    if (exp_offset > 0) {
      fillExpTable(lds + exp_offset);
      exp_copy = expCopy(lds + exp_offset);
    }
  const int L = nb_levels;
  const int segments = chordSegments(L), tangents = chordTangents(L);
  K* S = reinterpret_cast<K*>(lds);
  double* part = lds + (size_t(segments) * tile * sizeof(K) + 7) / 8;   // also the group-boundary levels
  const int groups = kThreads / tile;
  const int j = int(threadIdx.x) % tile;
  const int g = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / tile);   // tile: a multiple of 64
  const int chunk = (L + groups - 1) / groups;
  const int l0 = g * chunk;
  const int l1 = min(L, l0 + chunk);
  const size_t total = nbItems(win.count, batch);
  for (size_t item = blockIdx.x; item < total; item += gridDim.x) {
    int m, tl;
    if (!windowItem(item, batch, win, m, tl, point_group)) continue;      // uniform over the workgroup
    const unsigned char* r = rec.at(m);
    const BatchModel* bm = reinterpret_cast<const BatchModel*>(r);
    const LevelState* levels = reinterpret_cast<const LevelState*>(r + rec.levels);
    const Species* species = reinterpret_cast<const Species*>(r + rec.species);
    const int i = tl * tile + j;
    K last = K(0);
    if (i < n) {
      Op op;
      op.init(tables, base, stride, i, exp_copy);
      const double sigma_r = rayleigh ? rayleigh[i] : 0.0;
      Extras e = ex;
      double hm[7], cf[kMaxClouds];
      if constexpr (EX) {
        e.clouds = bm->clouds;
        loadExtras(e, i, n, wavelength[i], hm, cf);
      }
      for (int l = l0; l < l1; ++l) {
        const Species* d = species + size_t(l) * Op::kNS;
        if (l == l0 || levels[l].reload != 0) op.load(d, levels[l], rec.groups);
        const double kd = double(op.form(d, levels[l], rec.groups));
        double ke = kd + sigma_r * levels[l].rayleigh_density;
        if constexpr (EX) {
          if (e.hminus) ke += hminusKappa(hm, levels[l]);
          if (l > 0) ke += cloudLayer(e, cf, levels[l], l, i, n) * levels[l].cloud_scale;
        }
        const K k = K(ke);
        if constexpr (kKeep) keep[keptAt(win, m, stride, L, i) + size_t(l) * kKeptLevel] = float(k);
        if (l == l0) part[g * tile + j] = double(k);
        else S[(l - 1) * tile + j] = last + k;
        last = k;
      }
    } else {
      for (int l = l0; l < l1; ++l) {
        if (l == l0) part[g * tile + j] = 0.0;
        else S[(l - 1) * tile + j] = K(0);
      }
    }
    __syncthreads();
    if (l0 < l1 && l1 < L) S[(l1 - 1) * tile + j] = last + K(part[(g + 1) * tile + j]);
    if (g == 0)
      for (int q = L - 1; q < segments; ++q) S[q * tile + j] = K(0);
    __syncthreads();
    const double r0 = bm->bottom_radius;
    const K* chords;
    if constexpr (sizeof(K) == 8) chords = chord64;
    else chords = chord32;
    chords += size_t(m) * segments * tangents;
    double h = 0.0;
    for (int t0 = kTangentBlock * g; t0 < tangents; t0 += kTangentBlock * groups) {
      K tau[kTangentBlock];
      if constexpr (kKeep) {
        int stop[kTangentBlock];
        tangentBlock<K, true>(S + j, tile, chords, tangents, t0, L - 1, tau, stop);
        // per tile of 64 wavenumbers (a wavefront) and path: the largest
        // last segment, with which the adjoint passes over paths and steps
        // that end below its segments
        const int first64 = tl * tile + (j & ~63);
        int* rl = reach + (size_t(m) * ((n + 63) / 64) + first64 / 64) * (L - 1);
#pragma unroll
        for (int k = 0; k < kTangentBlock; ++k) {
          const int t = t0 + k;
          if (t < L - 1) {                                                 // uniform
            const int mx = waveMaxInt(i < n ? stop[k] : -1);
            if ((j & 63) == 0 && first64 < n) rl[t] = mx;
          }
        }
        if (i < n)
#pragma unroll
          for (int k = 0; k < kTangentBlock; ++k) {
            const int t = t0 + k;
            if (t < L - 1) {
              float* kt = keep + keptAt(win, m, stride, L, i) + size_t(t) * kKeptLevel;
              kt[kKeptValue] = float(tau[k]);
              kt[2 * kKeptValue] = float(stop[k]);
            }
          }
      } else {
        tangentBlock<K>(S + j, tile, chords, tangents, t0, L - 1, tau);
      }
#pragma unroll
      for (int k = 0; k < kTangentBlock; ++k) {
        const int t = t0 + k;
        if (t < L - 1) {
          const double zl = levels[t > 0 ? t - 1 : 0].altitude;
          const double zu = levels[t + 1].altitude;
          h += (r0 + levels[t].altitude) * (zu - zl) * (1.0 - transmittance(tau[k]));
        }
      }
    }
    part[g * tile + j] = h;
    __syncthreads();
    if (int(threadIdx.x) < tile && i < n) {
      double hs = 0.0;
      for (int q = 0; q < groups; ++q) hs += part[q * tile + j];
      const double hh = sqrt(hs + r0 * r0) - r0;
      const double rr = hh + r0;
      depth[size_t(m) * stride + i] = rr * rr / bm->star_radius / bm->star_radius * 1e6;
    }
    __syncthreads();
  }
}

template <class Op, int kThreads, bool kKeep, bool EX>
void launchTransmissionKernel(const SpectrumBatch& a, const void* tab) {
  constexpr bool wide = sizeof(typename Op::K) == 8;
  size_t lds = transmissionBatchLds(a.levels, a.shape.tile, wide, kThreads);
  int exp_offset = 0;
  if (wide && lds + kExpTable * sizeof(double) <= a.lds_limit) {
    exp_offset = int(lds / sizeof(double));
    lds += kExpTable * sizeof(double);
  }
  // FP64: a persistent grid, whose workgroups fill their exponential table
  // once; reduced precision: one item per workgroup, levelled by the
  // dispatcher (100 transits of 100 levels on INT16 tables 4.4 -> 4.0 ms), as
  // far as a launch goes
  const unsigned grid = wide ? unsigned(a.shape.grid)
                             : unsigned(std::min(nbItems(a.win.count, a.batch), maxWorkgroups(kThreads)));
  hipLaunchKernelGGL((transmissionBatchKernel<Op, kThreads, kKeep, EX>), dim3(grid), dim3(kThreads), lds,
                     a.stream, tab, a.base, a.stride, a.rayleigh, a.wavelength, a.ex, a.rec, a.chord, a.chord32,
                     a.levels, a.n, a.win, a.shape.tile, a.batch, a.shape.group, a.flux, a.keep, a.reach, exp_offset);
}

template <int NS>
void launchTransmission(const SpectrumBatch& a) {
  switch (a.precision) {
    case TablePrecision::fp64: {
      // Isothermal stencils where the wavefronts' partials and the exponential
      // table fit beside the tile's segment sums; 16 wavefronts per CU up to
      // 12 slots (128 registers: beyond that the slots' values spill), 8 above.
      // 200 transits, 12 slots, 200 levels: 11.35 -> 8.96 ms against the
      // general stencils.  Both go through the same tangent sums, 4 ms of it.
      constexpr int kWide = isothermalThreads(NS);
      if (a.isothermal && !a.extras &&
          transmissionBatchLds(a.levels, a.shape.tile, true, kWide) + kExpTable * sizeof(double) <= a.lds_limit)
        return a.keep ? launchTransmissionKernel<Opacity64Isothermal<NS>, kWide, true, false>(a, a.tab64)
                      : launchTransmissionKernel<Opacity64Isothermal<NS>, kWide, false, false>(a, a.tab64);
      if (a.keep)
        return a.extras ? launchTransmissionKernel<Opacity64<NS, false>, 512, true, true>(a, a.tab64)
                        : launchTransmissionKernel<Opacity64<NS, false>, 512, true, false>(a, a.tab64);
      return a.extras ? launchTransmissionKernel<Opacity64<NS, false>, 512, false, true>(a, a.tab64)
                      : launchTransmissionKernel<Opacity64<NS, false>, 512, false, false>(a, a.tab64);
    }
    case TablePrecision::fp32:
      return launchTransmissionKernel<Opacity32<NS, TabF32>, 512, false, false>(a, a.tab_low);
    case TablePrecision::fp16:
      return launchTransmissionKernel<Opacity32<NS, TabF16>, 512, false, false>(a, a.tab_low);
    case TablePrecision::bf16:
      return launchTransmissionKernel<Opacity32<NS, TabBF16>, 512, false, false>(a, a.tab_low);
    case TablePrecision::int16:
      return launchTransmissionKernel<Opacity32<NS, TabS16>, 512, false, false>(a, a.tab_low);
  }
}

}  // namespace
}  // namespace bear_amd
