// Reduced-precision cross-section tables: the stored types and the opacity of
// a level formed from them.
#pragma once

#include <hip/hip_runtime.h>

#include "device_math.h"
#include "engine.h"

namespace bear_amd {
namespace dev {

constexpr float kLog2TenF = 3.32192809488736234787f;

// ---------------------------------------------------------------- storage types
// raw(): the stored value as loaded; value(): its FP32 value
struct TabF32 {
  using T = float;
  using R = float;
  static __device__ __forceinline__ R raw(const T* p) { return *p; }
  static __device__ __forceinline__ float value(R r) { return r; }
  static __device__ __forceinline__ T store(double v) { return float(v); }
  static constexpr bool kScaled = false;
};
struct TabF16 {
  using T = _Float16;
  using R = _Float16;
  static __device__ __forceinline__ R raw(const T* p) { return *p; }
  static __device__ __forceinline__ float value(R r) { return float(r); }
  static __device__ __forceinline__ T store(double v) { return _Float16(float(v)); }
  static constexpr bool kScaled = false;
};
struct TabBF16 {
  using T = uint16_t;
  using R = float;                                 // widened when a row is read
  static __device__ __forceinline__ R raw(const T* p) { return __uint_as_float(uint32_t(*p) << 16); }
  static __device__ __forceinline__ float value(R r) { return r; }
  static __device__ __forceinline__ T store(double v) {   // round to nearest even
    const uint32_t u = __float_as_uint(float(v));
    return uint16_t((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
  }
  static constexpr bool kScaled = false;
};
// 16-bit integers q in [-32767, 32767] with value = base + scale q, base and
// scale per (species, wavenumber): the 16 bits cover each wavenumber's own
// range uniformly (an absolute error of at most range / 131068), where FP16
// residuals spend bits on exponents.  The base array then holds per species
// slot the base row and the scale row.
struct TabS16 {
  using T = int16_t;
  using R = float;                                 // scale q, formed when a row is read
  static __device__ __forceinline__ float value(R r) { return r; }
  static constexpr bool kScaled = true;
  static constexpr int kMax = 32767;
};

// Reduced-precision tables: x = log2(10) base + log2 n + sum_k w_k v_k in
// FP32 and sigma n = 2^x with the hardware exponential.
template <int NS, class Tab>
struct Opacity32 {
  static constexpr int kNS = NS;
  static constexpr bool kScaled = Tab::kScaled;
  using Species = LevelSpecies32;
  using K = float;
  const typename Tab::T* tab;
  unsigned i;
  float bz[NS];
  float sc[Tab::kScaled ? NS : 1];                 // scales of TabS16
  typename Tab::R v[NS][4];       // as stored; converted where used (FP16 folds into v_fma_mix_f32)
  __device__ __forceinline__ void init(const void* tables, const float* base, size_t s, int at, const double*) {
    tab = static_cast<const typename Tab::T*>(tables);
    i = unsigned(at);
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      if constexpr (Tab::kScaled) {
        bz[q] = base[size_t(2 * q) * s + i] * kLog2TenF;
        sc[q] = base[size_t(2 * q + 1) * s + i];
      } else {
        bz[q] = base[size_t(q) * s + i] * kLog2TenF;
      }
    }
  }
  __device__ __forceinline__ int slots() const { return NS; }
  // x = bz + log2 n + sum_k w_k v_k (TabS16: v = scale q, formed at the row's read)
  __device__ __forceinline__ float exponent(int s, float start, const float* w) const {
    float x = fmaf(w[0], Tab::value(v[s][0]), start);
    x = fmaf(w[1], Tab::value(v[s][1]), x);
    x = fmaf(w[2], Tab::value(v[s][2]), x);
    return fmaf(w[3], Tab::value(v[s][3]), x);
  }
  __device__ __forceinline__ typename Tab::R value(const typename Tab::T* p, int s) const {
    if constexpr (Tab::kScaled) return sc[s] * float(*p);
    else return Tab::raw(p);
  }
  __device__ __forceinline__ void load(const LevelSpecies32* d, const LevelState&, StencilGroups) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[s][q] = value(tab + (size_t(d[s].block[q]) << 6) + i, s);
  }
  // grouped stencils: the level's shared weights and contiguous densities
  // (FP32 copies), as kappaFrom does for the FP64 tables
  __device__ __forceinline__ float form(const LevelSpecies32* d, const LevelState& lev, StencilGroups groups) const {
    float k = 0.0f;
    if (groups.grouped) {
      // as bits: a uniform choice of words stays in the scalar unit, one of
      // floats is made per lane (14 slots: 56 selects per level, 224 of some
      // 1,000 cycles; 100 transits of 100 levels on INT16 tables 7.2 -> 4.4 ms)
      int a[4], b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[q] = __float_as_int(lev.group_w32[0][q]);
        b[q] = __float_as_int(lev.group_w32[1][q]);
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        float w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          w[q] = __int_as_float(s >= NS - NS / 2 && ((groups.group1 >> s) & 1u) ? b[q] : a[q]);
        k += __builtin_amdgcn_exp2f(exponent(s, bz[s] + lev.log2_n32[s], w));
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) k += __builtin_amdgcn_exp2f(exponent(s, bz[s] + d[s].log2_n, d[s].w));
    }
    return k;
  }
};

}  // namespace dev
}  // namespace bear_amd
