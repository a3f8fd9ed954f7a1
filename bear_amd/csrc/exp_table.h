// FP64 powers of two from a table in LDS: a table of the octave's steps and a
// short polynomial within a step (P. T. P. Tang, Table-driven implementation of
// the exponential function, ACM TOMS 15, 1989).
//
// 2^(i / 128 + f / 128) = 2^(i / 128) P(f): the table holds 2^(j / 128) for j
// in [0, 128), and P is a polynomial of degree 3 or 4 in f, so that a power
// of ten costs 10 FP64 instructions and 3 integer ones (about 52 cycles of a
// wavefront) instead of 17 with the degree-8 polynomial of a whole octave
// (68), and an attenuation factor 9 + 3 instead of 15.  FP64 instructions
// issue at 4 cycles each whatever they do, so their count is what bounds the
// opacity and transfer kernels.  The table is held 16 times over, copy c in
// bank pair c: the 16 lanes that LDS serves together never meet in a bank
// (random entries of a single copy cost 12 cycles per read instead of 4).
// Measured with 64 points of 100 levels, 8 species and 99,777 wavenumbers:
// 6.2 -> 5.6 ms per batch.
#pragma once

#include "device_math.h"

namespace bear_amd {
namespace dev {

constexpr int kExpSteps = 128, kExpCopies = 16;
constexpr int kExpTable = kExpSteps * kExpCopies;      // doubles
// Arguments are taken in steps of 1 / 128 with this bias, so that their
// integer part is positive: 1024 octaves
constexpr double kExpBias = kTableBias;
static_assert(kTableSteps == kExpSteps, "levels staged for another table");

__device__ const double kPow2Steps[kExpSteps] = {
    0x1.0000000000000p+0, 0x1.0163da9fb3335p+0, 0x1.02c9a3e778061p+0, 0x1.04315e86e7f85p+0,
    0x1.059b0d3158574p+0, 0x1.0706b29ddf6dep+0, 0x1.0874518759bc8p+0, 0x1.09e3ecac6f383p+0,
    0x1.0b5586cf9890fp+0, 0x1.0cc922b7247f7p+0, 0x1.0e3ec32d3d1a2p+0, 0x1.0fb66affed31bp+0,
    0x1.11301d0125b51p+0, 0x1.12abdc06c31ccp+0, 0x1.1429aaea92de0p+0, 0x1.15a98c8a58e51p+0,
    0x1.172b83c7d517bp+0, 0x1.18af9388c8deap+0, 0x1.1a35beb6fcb75p+0, 0x1.1bbe084045cd4p+0,
    0x1.1d4873168b9aap+0, 0x1.1ed5022fcd91dp+0, 0x1.2063b88628cd6p+0, 0x1.21f49917ddc96p+0,
    0x1.2387a6e756238p+0, 0x1.251ce4fb2a63fp+0, 0x1.26b4565e27cddp+0, 0x1.284dfe1f56381p+0,
    0x1.29e9df51fdee1p+0, 0x1.2b87fd0dad990p+0, 0x1.2d285a6e4030bp+0, 0x1.2ecafa93e2f56p+0,
    0x1.306fe0a31b715p+0, 0x1.32170fc4cd831p+0, 0x1.33c08b26416ffp+0, 0x1.356c55f929ff1p+0,
    0x1.371a7373aa9cbp+0, 0x1.38cae6d05d866p+0, 0x1.3a7db34e59ff7p+0, 0x1.3c32dc313a8e5p+0,
    0x1.3dea64c123422p+0, 0x1.3fa4504ac801cp+0, 0x1.4160a21f72e2ap+0, 0x1.431f5d950a897p+0,
    0x1.44e086061892dp+0, 0x1.46a41ed1d0057p+0, 0x1.486a2b5c13cd0p+0, 0x1.4a32af0d7d3dep+0,
    0x1.4bfdad5362a27p+0, 0x1.4dcb299fddd0dp+0, 0x1.4f9b2769d2ca7p+0, 0x1.516daa2cf6642p+0,
    0x1.5342b569d4f82p+0, 0x1.551a4ca5d920fp+0, 0x1.56f4736b527dap+0, 0x1.58d12d497c7fdp+0,
    0x1.5ab07dd485429p+0, 0x1.5c9268a5946b7p+0, 0x1.5e76f15ad2148p+0, 0x1.605e1b976dc09p+0,
    0x1.6247eb03a5585p+0, 0x1.6434634ccc320p+0, 0x1.6623882552225p+0, 0x1.68155d44ca973p+0,
    0x1.6a09e667f3bcdp+0, 0x1.6c012750bdabfp+0, 0x1.6dfb23c651a2fp+0, 0x1.6ff7df9519484p+0,
    0x1.71f75e8ec5f74p+0, 0x1.73f9a48a58174p+0, 0x1.75feb564267c9p+0, 0x1.780694fde5d3fp+0,
    0x1.7a11473eb0187p+0, 0x1.7c1ed0130c132p+0, 0x1.7e2f336cf4e62p+0, 0x1.80427543e1a12p+0,
    0x1.82589994cce13p+0, 0x1.8471a4623c7adp+0, 0x1.868d99b4492edp+0, 0x1.88ac7d98a6699p+0,
    0x1.8ace5422aa0dbp+0, 0x1.8cf3216b5448cp+0, 0x1.8f1ae99157736p+0, 0x1.9145b0b91ffc6p+0,
    0x1.93737b0cdc5e5p+0, 0x1.95a44cbc8520fp+0, 0x1.97d829fde4e50p+0, 0x1.9a0f170ca07bap+0,
    0x1.9c49182a3f090p+0, 0x1.9e86319e32323p+0, 0x1.a0c667b5de565p+0, 0x1.a309bec4a2d33p+0,
    0x1.a5503b23e255dp+0, 0x1.a799e1330b358p+0, 0x1.a9e6b5579fdbfp+0, 0x1.ac36bbfd3f37ap+0,
    0x1.ae89f995ad3adp+0, 0x1.b0e07298db666p+0, 0x1.b33a2b84f15fbp+0, 0x1.b59728de5593ap+0,
    0x1.b7f76f2fb5e47p+0, 0x1.ba5b030a1064ap+0, 0x1.bcc1e904bc1d2p+0, 0x1.bf2c25bd71e09p+0,
    0x1.c199bdd85529cp+0, 0x1.c40ab5fffd07ap+0, 0x1.c67f12e57d14bp+0, 0x1.c8f6d9406e7b5p+0,
    0x1.cb720dcef9069p+0, 0x1.cdf0b555dc3fap+0, 0x1.d072d4a07897cp+0, 0x1.d2f87080d89f2p+0,
    0x1.d5818dcfba487p+0, 0x1.d80e316c98398p+0, 0x1.da9e603db3285p+0, 0x1.dd321f301b460p+0,
    0x1.dfc97337b9b5fp+0, 0x1.e264614f5a129p+0, 0x1.e502ee78b3ff6p+0, 0x1.e7a51fbc74c83p+0,
    0x1.ea4afa2a490dap+0, 0x1.ecf482d8e67f1p+0, 0x1.efa1bee615a27p+0, 0x1.f252b376bba97p+0,
    0x1.f50765b6e4540p+0, 0x1.f7bfdad9cbe14p+0, 0x1.fa7c1819e90d8p+0, 0x1.fd3c22b8f71f1p+0};

// The workgroup fills its table: entry j holds the bits of 2^(j / 128) with
// (j << 13) + (1024 << 20) taken off the high word, so that adding i << 13 for
// the biased integer i = 128 (n + 1024) + j leaves the exponent of 2^n alone.
__device__ __forceinline__ void fillExpTable(double* __restrict__ table) {
  for (int k = int(threadIdx.x); k < kExpTable; k += int(blockDim.x)) {
    const int j = k / kExpCopies;
    const double v = kPow2Steps[j];
    table[k] = __hiloint2double(__double2hiint(v) - (j << 13) - (1024 << 20), __double2loint(v));
  }
  __syncthreads();
}

// 2^(i / 128 - 1024) for the biased integer i; copy: this lane's column of
// the table (table + lane % 16)
__device__ __forceinline__ double expStep(const double* __restrict__ copy, int i) {
  const double v = copy[(i & (kExpSteps - 1)) * kExpCopies];
  return __hiloint2double(__double2hiint(v) + (i << 13), __double2loint(v));
}

__device__ __forceinline__ const double* expCopy(const double* table) { return table + (threadIdx.x & (kExpCopies - 1)); }

// acc + 2^(x / 128 - 1024) for 0 < x < 2^18: relative error of the power
// 2.8e-13 from the polynomial (2^(f / 128) on [0, 1)) plus the rounding of x,
// 1e-13 (the degree-8 octave polynomial it replaces: 1.1e-12).  For the
// opacity terms, which add and where nothing cancels.
__device__ __forceinline__ double addPow2(double acc, const double* __restrict__ copy, double x) {
  const double f = __builtin_amdgcn_fract(x);
  const int i = int(x);
  double p = 2.6538188920206277e-08;
  p = fma(p, f, 1.4662217512320395e-05);
  p = fma(p, f, 0.0054152123571012765);
  p = fma(p, f, 0.9999999999997194);
  return fma(expStep(copy, i), p, acc);
}

// 2^(x / 128) with relative error below 4e-16 (pow2: 3.1e-15), and near x = 0
// the correctly rounded 1 + x ln2 / 128 of pow2; results beyond 2^-1021 and
// 2^1022 stay there.  For the attenuation factors and the Planck function.
constexpr double kExpLowest = -1021.0 * kExpSteps, kExpHighest = 1022.0 * kExpSteps;

__device__ __forceinline__ double tablePow2(const double* __restrict__ copy, double x) {
  x = fmin(fmax(x, kExpLowest), kExpHighest);
  // round to the nearest integer by its place in the sum, which also leaves
  // the biased integer in the low word
  constexpr double kRound = 6755399441055744.0 + kExpBias;       // 1.5 2^52 + bias
  const double m = x + kRound;
  const double f = x - (m - kRound);
  double p = 3.5830329620923136e-11;
  p = fma(p, f, 2.6466428720412216e-08);
  p = fma(p, f, 1.4662262387640425e-05);
  p = fma(p, f, 0.0054152123481245725);
  return expStep(copy, __double2loint(m)) * fma(p, f, 1.0);
}

// planckAt from the table
__device__ __forceinline__ double planckTable(const double* __restrict__ copy, double b_num, double x_nu,
                                              double inv_t) {
  const double q = tablePow2(copy, x_nu * double(kExpSteps) * inv_t);
  return b_num * q * recip(1.0 - q);
}

}  // namespace dev
}  // namespace bear_amd
