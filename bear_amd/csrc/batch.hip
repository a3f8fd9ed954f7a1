// Batched likelihood evaluation on gfx950: many live points of one retrieval
// per launch sequence.
//
// One work item is (wavenumber tile, live point), ordered so that every live
// point of one tile runs on the same XCD (workgroups go to XCDs round-robin by
// id, and the grid is a multiple of 8), where the tile's table rows stay in
// that XCD's L2 while the points reuse them.  A workgroup takes one item, and
// the dispatcher levels them; only the FP64 transits walk the items with a
// persistent grid, sized by the autotuner.
//
// Per batch, in one hipGraph when enabled: the pinned per-point records go to
// the device in one copy; (transmission) the chord lengths of every point are
// computed; the spectrum kernel writes [point][wavenumber] FP64; one
// workgroup per (bin, point) folds the observation operator and the Gaussian
// term; one workgroup per point sums its terms; the log-likelihoods come back
// in one copy.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <string>

#include "batch_launch.h"
#include "device_math.h"
#include "engine.h"
#include "launch_shape.h"
#include "reduced_opacity.h"
#include "tile_window.h"

namespace bear_amd {

using namespace dev;

namespace {

void check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  const int code = (e == hipErrorOutOfMemory) ? kOutOfMemory : kDevice;
  raise(code, std::string(what) + ": " + hipGetErrorString(e));
}

template <class T>
T* deviceAlloc(size_t count, const char* what) {
  void* p = nullptr;
  if (count == 0) count = 1;
  check(hipMalloc(&p, count * sizeof(T)), what);
  return static_cast<T*>(p);
}

void deviceFree(void* p) {
  if (p) (void)hipFree(p);
}

// One species' FP64 rows [0, count) (row-major, `stride` apart) at
// wavenumber i: base = FP32 midrange of the values, residual = value - base
// into the species' rows of `low` (same layout).  Nothing is floored:
// log-linear interpolation between a row at the reference's 1e-200 floor and
// a row far above it yields values in between that can dominate a level's
// opacity.
template <class Tab>
__global__ __launch_bounds__(kBatchBlock) void splitTableKernel(const double* __restrict__ rows, size_t stride, int n,
                                                                uint32_t count, int slot, float* __restrict__ base,
                                                                typename Tab::T* __restrict__ low) {
  const int i = blockIdx.x * kBatchBlock + threadIdx.x;
  if (i >= n) return;
  double hi = -INFINITY, lo = INFINITY;
  for (uint32_t r = 0; r < count; ++r) {
    const double v = rows[size_t(r) * stride + i];
    hi = fmax(hi, v);
    lo = fmin(lo, v);
  }
  const float b = float(0.5 * (hi + lo));
  if constexpr (Tab::kScaled) {
    // scale: the smallest FP32 value with kMax scale >= the largest residual
    const double reach = fmax(hi - double(b), double(b) - lo);
    float sc = reach > 0.0 ? float(reach / Tab::kMax) : 1.0f;
    if (double(sc) * Tab::kMax < reach) sc = __uint_as_float(__float_as_uint(sc) + 1u);   // next FP32 up
    base[size_t(2 * slot) * stride + i] = b;
    base[size_t(2 * slot + 1) * stride + i] = sc;
    for (uint32_t r = 0; r < count; ++r) {
      const double q = rint((rows[size_t(r) * stride + i] - double(b)) / double(sc));
      low[size_t(r) * stride + i] = typename Tab::T(fmin(fmax(q, -double(Tab::kMax)), double(Tab::kMax)));
    }
  } else {
    base[size_t(slot) * stride + i] = b;
    for (uint32_t r = 0; r < count; ++r)
      low[size_t(r) * stride + i] = Tab::store(rows[size_t(r) * stride + i] - double(b));
  }
}

// Chord lengths of every point, transposed (chord[point][q][t], chordLength);
// one workgroup per (segment q, point), FP64 and/or FP32.
__global__ __launch_bounds__(kBatchBlock) void chordKernel(Records rec, int nb_levels, double* __restrict__ chord,
                                                           float* __restrict__ chord32) {
  const int q = blockIdx.x, m = blockIdx.y;
  const int tangents = chordTangents(nb_levels);
  const unsigned char* r = rec.at(m);
  const double r0 = reinterpret_cast<const BatchModel*>(r)->bottom_radius;
  const LevelState* levels = reinterpret_cast<const LevelState*>(r + rec.levels);
  const size_t row = (size_t(m) * gridDim.x + q) * tangents;
  for (int t = int(threadIdx.x); t < tangents; t += kBatchBlock) {
    const double c = chordLength(levels, r0, nb_levels, q, t);
    if (chord) chord[row + t] = c;
    if (chord32) chord32[row + t] = float(c);
  }
}

// ---------------------------------------------------------------- bins and likelihood
// One workgroup per (piece of a bin's segment, point) (binChunkBody); mode 1
// (eclipse) also sums the folded blackbody star of that point.
__global__ __launch_bounds__(kBlockBins) void binBatchKernel(
    const double* __restrict__ flux, size_t stride, const double* __restrict__ wavenumber,
    const double* __restrict__ weights, const BinChunk* __restrict__ chunks, int nb_chunks, Records rec, int mode,
    double* __restrict__ chunk_sums) {
  const int m = blockIdx.y;
  const BatchModel* bm = reinterpret_cast<const BatchModel*>(rec.at(m));
  binChunkBody(flux + size_t(m) * stride, wavenumber, weights, chunks[blockIdx.x], mode, bm->star_inv_temperature,
               chunk_sums + (size_t(m) * nb_chunks + blockIdx.x) * 2);
}

// Bins and log-likelihood of one point per workgroup (binFinalizeBody)
__global__ __launch_bounds__(1024) void sumBatchKernel(const double* __restrict__ chunk_sums, int nb_chunks,
                                                       const BinDesc* __restrict__ bins, int nb_bins, Records rec,
                                                       int mode, double* __restrict__ out, double* __restrict__ ll) {
  const int m = blockIdx.x;
  const unsigned char* r = rec.at(m);
  const BatchModel* bm = reinterpret_cast<const BatchModel*>(r);
  const double* shifts = reinterpret_cast<const double*>(r + rec.shifts);
  binFinalizeBody(chunk_sums + size_t(m) * nb_chunks * 2, bins, nb_bins, mode, bm->depth_scale, shifts,
                  bm->inflation, out + size_t(m) * nb_bins, ll + m, nullptr);
}

// high-resolution output per point: emission F per micron, eclipse depth
// F / F_* (Rp/Rs)^2 1e6, transmission depth; elements [first, first + count)
// of the [point][n] output to out (pinned host memory)
__global__ __launch_bounds__(kBatchBlock) void batchSpectrumKernel(
    const double* __restrict__ flux, size_t stride, const double* __restrict__ wavenumber,
    const double* __restrict__ wavelength, Records rec, int mode, int n, size_t first, int count,
    double* __restrict__ out) {
  const int k = int(blockIdx.x) * kBatchBlock + int(threadIdx.x);
  if (k >= count) return;
  const size_t m = (first + size_t(k)) / size_t(n);
  const int i = int((first + size_t(k)) - m * size_t(n));
  const BatchModel* bm = reinterpret_cast<const BatchModel*>(rec.at(m));
  const double f = flux[size_t(m) * stride + i];
  double v = f;
  if (mode == 0) {
    const double lam = wavelength[i];
    v = f / lam / lam * 10000.0;
  } else if (mode == 1) {
    v = f * recip(starFlux(wavenumber[i], bm->star_inv_temperature)) * bm->depth_scale;
  }
  out[k] = v;
}

size_t align(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace

size_t transmissionBatchLds(int L, int tile, bool wide, int threads) {
  const size_t k = size_t(chordSegments(L)) * tile * (wide ? 8 : 4);
  return align(k, 8) + size_t(threads / tile) * tile * sizeof(double);
}

// ---------------------------------------------------------------- precision
// residual tables [rows][stride] and the base [slots][stride], zero base in
// the padding slots (their density is zero, their row is row 0)
void DeviceEngine::allocateReduced(TablePrecision p, size_t nb_rows, size_t slots) {
  void* low = nullptr;
  check(hipMalloc(&low, nb_rows * stride_ * tableElementBytes(p)), "reduced-precision tables");
  tables_low_ = low;
  check(hipMemsetAsync(low, 0, stride_ * tableElementBytes(p), static_cast<hipStream_t>(stream_)), "clear table row");
  base_rows_ = slots * (p == TablePrecision::int16 ? 2 : 1);          // int16: base and scale per slot
  table_base_ = deviceAlloc<float>(base_rows_ * stride_, "table base");
  check(hipMemsetAsync(table_base_, 0, base_rows_ * stride_ * sizeof(float), static_cast<hipStream_t>(stream_)),
        "clear table base");
}

// species `slot`'s FP64 rows (device, [count][stride]) split into the base and
// the residual rows [first, first + count)
void DeviceEngine::splitSpecies(const double* rows, size_t count, int slot, size_t first) {
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const int n = int(n_points_);
  const dim3 grid((n + kBatchBlock - 1) / kBatchBlock), block(kBatchBlock);
  const uint32_t c = uint32_t(count);
  switch (precision_) {
    case TablePrecision::fp32:
      hipLaunchKernelGGL(splitTableKernel<TabF32>, grid, block, 0, s, rows, stride_, n, c, slot, table_base_,
                         static_cast<float*>(tables_low_) + first * stride_);
      break;
    case TablePrecision::fp16:
      hipLaunchKernelGGL(splitTableKernel<TabF16>, grid, block, 0, s, rows, stride_, n, c, slot, table_base_,
                         static_cast<_Float16*>(tables_low_) + first * stride_);
      break;
    case TablePrecision::bf16:
      hipLaunchKernelGGL(splitTableKernel<TabBF16>, grid, block, 0, s, rows, stride_, n, c, slot, table_base_,
                         static_cast<uint16_t*>(tables_low_) + first * stride_);
      break;
    case TablePrecision::int16:
      hipLaunchKernelGGL(splitTableKernel<TabS16>, grid, block, 0, s, rows, stride_, n, c, slot, table_base_,
                         static_cast<int16_t*>(tables_low_) + first * stride_);
      break;
    default:
      raise(kInternal, "no split for FP64 tables");
  }
  check(hipGetLastError(), "table split kernel");
}

void DeviceEngine::setTablePrecision(TablePrecision p,
                                     const std::vector<std::pair<uint32_t, uint32_t>>& species_rows) {
  check(hipSetDevice(device_), "hipSetDevice");
  if (storage_ != TablePrecision::fp64) {
    if (p != storage_)
      raise(kInvalidInput, "the tables were loaded at reduced precision only; no other precision is available");
    return;
  }
  releaseGraph();
  deviceFree(tables_low_);
  deviceFree(table_base_);
  tables_low_ = nullptr;
  table_base_ = nullptr;
  precision_ = p;
  batch_capacity_ = 0;                                  // record layout depends on the precision
  tuned_.clear();
  if (p == TablePrecision::fp64) return;
  if (species_rows.size() > species_stride_) raise(kInvalidInput, "more species than stencil slots");
  allocateReduced(p, n_rows_, species_stride_);
  for (size_t q = 0; q < species_rows.size(); ++q) {
    const uint32_t r0 = species_rows[q].first, r1 = species_rows[q].second;
    if (r1 <= r0 || r1 > n_rows_) raise(kInternal, "species rows out of range");
    splitSpecies(tables_ + size_t(r0) * stride_, r1 - r0, int(q), r0);
  }
  check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "table split");
}

// ---------------------------------------------------------------- staging
LevelSpecies* DeviceEngine::batchSpecies(size_t b) {
  if (precision_ != TablePrecision::fp64) raise(kInternal, "FP64 stencils requested with reduced-precision tables");
  return reinterpret_cast<LevelSpecies*>(record(b) + rec_species_);
}

LevelSpeciesAdjoint* DeviceEngine::batchSpeciesAdjoint(size_t b) {
  if (precision_ != TablePrecision::fp64) raise(kInternal, "adjoint stencils requested with reduced-precision tables");
  return reinterpret_cast<LevelSpeciesAdjoint*>(record(b) + rec_adjoint_);
}

LevelSpecies32* DeviceEngine::batchSpecies32(size_t b) {
  if (precision_ == TablePrecision::fp64) raise(kInternal, "FP32 stencils requested with FP64 tables");
  return reinterpret_cast<LevelSpecies32*>(record(b) + rec_species_);
}

void DeviceEngine::reserveBatch(size_t batch) {
  if (batch == 0) raise(kInvalidInput, "empty batch");
  if (batch > 65535) raise(kInvalidInput, "at most 65535 live points per batch");
  if (batch <= batch_capacity_) return;
  check(hipSetDevice(device_), "hipSetDevice");
  check(hipStreamSynchronize(static_cast<hipStream_t>(stream_)), "batch");
  releaseGraph();
  const size_t L = nb_levels_, NS = species_stride_;
  const size_t spc = precision_ == TablePrecision::fp64 ? sizeof(LevelSpecies) : sizeof(LevelSpecies32);
  const bool wide = precision_ == TablePrecision::fp64;
  rec_levels_ = align(sizeof(BatchModel), 64);
  rec_species_ = align(rec_levels_ + L * sizeof(LevelState), 64);
  rec_adjoint_ = wide ? align(rec_species_ + L * NS * spc, 64) : 0;
  rec_shifts_ = align(wide ? rec_adjoint_ + L * NS * sizeof(LevelSpeciesAdjoint) : rec_species_ + L * NS * spc, 64);
  rec_bytes_ = align(rec_shifts_ + (n_obs_ + 1) * sizeof(double), 256);
  if (batch_host_) (void)hipHostFree(batch_host_);
  if (batch_ll_host_) (void)hipHostFree(batch_ll_host_);
  batch_host_ = nullptr;
  batch_ll_host_ = nullptr;
  for (void* p : {(void*)batch_dev_, (void*)batch_flux_, (void*)batch_bins_, (void*)batch_chunk_sums_, (void*)batch_ll_,
                  (void*)batch_chord_, (void*)batch_chord32_})
    deviceFree(p);
  batch_dev_ = nullptr;
  batch_flux_ = batch_bins_ = batch_chunk_sums_ = batch_ll_ = batch_chord_ = nullptr;
  batch_chord32_ = nullptr;
  batch_capacity_ = 0;
  void* h = nullptr;
  check(hipHostMalloc(&h, batch * rec_bytes_, hipHostMallocDefault), "pinned batch records");
  batch_host_ = static_cast<unsigned char*>(h);
  std::memset(batch_host_, 0, batch * rec_bytes_);
  check(hipHostMalloc(&h, batch * sizeof(double), hipHostMallocDefault), "pinned batch log-likelihoods");
  batch_ll_host_ = static_cast<double*>(h);
  batch_dev_ = deviceAlloc<unsigned char>(batch * rec_bytes_, "batch records");
  batch_flux_ = deviceAlloc<double>(batch * stride_, "batch spectra");
  batch_bins_ = deviceAlloc<double>(batch * std::max<size_t>(1, n_bins_), "batch bins");
  batch_chunk_sums_ = deviceAlloc<double>(batch * std::max<size_t>(1, n_chunks_) * 2, "batch bin piece sums");
  batch_ll_ = deviceAlloc<double>(batch, "batch log-likelihoods");
  if (transmission_) {
    const size_t chord_size = size_t(chordSegments(int(L))) * chordTangents(int(L));
    if (precision_ == TablePrecision::fp64) batch_chord_ = deviceAlloc<double>(batch * chord_size, "batch chord lengths");
    else batch_chord32_ = deviceAlloc<float>(batch * chord_size, "batch chord lengths");
  }
  batch_capacity_ = batch;
}

// ---------------------------------------------------------------- launches
void DeviceEngine::launchBatchSpectrum(ModelKind kind, size_t batch, const BatchLaunch& lc, size_t first,
                                       float* keep, size_t nu_first, size_t nu_count, int* reach, bool adjoint) {
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const Records rec{batch_dev_ + first * rec_bytes_, rec_bytes_, rec_levels_, rec_species_, rec_adjoint_,
                    rec_shifts_, groups_};
  double* flux = batch_flux_ + first * stride_;
  const int n = int(n_points_), L = int(nb_levels_), B = int(batch);
  const bool wide = precision_ == TablePrecision::fp64;
  SpectrumBatch a;
  a.precision = precision_;
  a.shape = lc;
  a.stream = s;
  a.wavenumber = wavenumber_;
  a.wavelength = wavelength_;
  a.rayleigh = rayleigh_;
  a.tab64 = tables_;
  a.tab_low = tables_low_;
  a.base = table_base_;
  a.stride = stride_;
  a.ex = Extras{hminus_, nullptr, CloudSpec{}};          // the clouds' parameters come with each point's record
  a.extras = hminus_ != nullptr || cloud_models_ > 0;
  a.isothermal = isothermal_;
  a.rec = rec;
  a.chord = batch_chord_;
  a.chord32 = batch_chord32_;
  a.levels = L;
  a.n = n;
  a.batch = B;
  a.lds_limit = lds_limit_;
  a.win = TileWindow{0, 0, 0};
  a.flux = flux;
  a.adjoint = adjoint;
  a.keep = keep;
  a.reach = reach;
  bool launched;
  if (kind == ModelKind::transmission) {
    hipLaunchKernelGGL(chordKernel, dim3(unsigned(chordSegments(L)), unsigned(B)), dim3(kBatchBlock), 0, s, rec, L,
                       wide ? batch_chord_ : nullptr, wide ? nullptr : batch_chord32_);
    check(hipGetLastError(), "chord kernel");
    a.win = wholeGrid((n + lc.tile - 1) / lc.tile);
    if (nu_count > 0) {                                   // wavenumbers [nu_first, nu_first + nu_count)
      if (nu_first % size_t(lc.tile) != 0 || nu_first >= size_t(n)) raise(kInternal, "misaligned wavenumber window");
      a.win.first = int(nu_first / size_t(lc.tile));
      a.win.count =
          int((std::min(size_t(n), nu_first + nu_count) + size_t(lc.tile) - 1) / size_t(lc.tile)) - a.win.first;
      a.win.kept_origin = nu_first / kKeptValue * size_t(L) * kKeptLevel;
    }
    launched = launchTransmissionSlots1To8(species_stride_, a) || launchTransmissionSlots9To16(species_stride_, a);
  } else {
    const size_t run = pointsPerLaunch((n + lc.tile - 1) / lc.tile, lc.block);
    launched = true;
    for (size_t m = 0; m < batch && launched; m += run) {
      a.batch = int(std::min(run, batch - m));
      a.rec.base = rec.base + m * rec_bytes_;
      a.flux = flux + m * stride_;
      a.keep = keep ? keep + m * (stride_ / kKeptValue) * size_t(L) * kKeptLevel : nullptr;   // keptColumn
      launched = launchEmissionSlots1To8(species_stride_, a) || launchEmissionSlots9To16(species_stride_, a);
    }
  }
  if (!launched) raise(kInvalidInput, "the batched kernels take at most 16 tabulated species");
  check(hipGetLastError(), "batched spectrum kernel");
}

void DeviceEngine::launchBatchRest(ModelKind kind, size_t batch, size_t first) {
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const Records rec{batch_dev_ + first * rec_bytes_, rec_bytes_, rec_levels_, rec_species_, rec_adjoint_,
                    rec_shifts_, groups_};
  if (n_bins_ > 0) {
    const int mode = kind == ModelKind::eclipse ? 1 : 0;
    double* sums = batch_chunk_sums_ + first * n_chunks_ * 2;
    hipLaunchKernelGGL(binBatchKernel, dim3(unsigned(n_chunks_), unsigned(batch)), dim3(kBlockBins), 0, s,
                       batch_flux_ + first * stride_, stride_, wavenumber_, weights_, bin_chunks_, int(n_chunks_), rec,
                       mode, sums);
    check(hipGetLastError(), "batch bin kernel");
    hipLaunchKernelGGL(sumBatchKernel, dim3(unsigned(batch)), dim3(1024), 0, s, sums, int(n_chunks_), bins_desc_,
                       int(n_bins_), rec, mode, batch_bins_ + first * n_bins_, batch_ll_ + first);
    check(hipGetLastError(), "batch likelihood kernel");
    check(hipMemcpyAsync(batch_ll_host_ + first, batch_ll_ + first, batch * sizeof(double), hipMemcpyDeviceToHost,
                         s),
          "read batch log-likelihoods");
  }
}

// Autotuner: times the spectrum kernel for each candidate launch shape and
// keeps the fastest, on the records that the host holds of the first
// min(batch, 64) points.  A batch staged on the device leaves those as they
// were, all zeros at first: the kernels then do their full work on values that
// mean nothing, without the early ends of opaque columns and paths.
//   emission / eclipse: workgroups of 128 or 256 wavenumbers; where that
//     leaves the chip under four rounds of wavefronts, also tiles of 64
//     wavenumbers with their levels split over 2, 4 or 8 wavefronts
//   transmission: tile of 64 or 128 wavenumbers within the device's LDS per
//     workgroup; FP64: grid of 1, 2 or 4 workgroups per CU; points taken in
//     groups of 1 or 4 (each point brings its own chord matrix)
BatchLaunch DeviceEngine::tune(ModelKind kind, size_t batch) {
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const size_t b = std::min<size_t>(batch, 64);
  std::vector<BatchLaunch> cand;
  if (kind == ModelKind::transmission) {
    const bool wide = precision_ == TablePrecision::fp64;
    for (int tile : {64, 128}) {
      if (transmissionBatchLds(int(nb_levels_), tile, wide) > lds_limit_) continue;
      for (int group : {1, 4})
        for (int per_cu : {1, 2, 4}) {
          if (!wide && per_cu > 1) continue;                // one item per workgroup: no grid to choose
          cand.push_back(BatchLaunch{kTransmissionBlock, tile, std::max(8, nb_cus_ * per_cu), group});
        }
    }
    if (cand.empty()) raise(kInvalidInput, "too many levels for the transmission batch kernel");
  } else {
    auto shape = [&](int block, int tile, int split) {
      const size_t items = nbItems(int((n_points_ + tile - 1) / tile), int(batch));
      return BatchLaunch{block, tile, int(std::min<size_t>(items, INT32_MAX)), kPointGroup, split};
    };
    const size_t tiles = (n_points_ + 63) / 64 * batch;
    const int split = levelSplit(tiles, nb_cus_);
    if (!autotune_) return split > 1 ? shape(64 * split, 64, split) : shape(256, 256, 1);
    for (int block : {256, 128}) cand.push_back(shape(block, block, 1));
    if (tiles < size_t(nb_cus_) * 64)
      for (int k : {2, 4, 8}) cand.push_back(shape(64 * k, 64, k));
  }
  if (kind == ModelKind::transmission)
    for (auto& c : cand) c.grid = int(align(size_t(c.grid), 8));
  if (!autotune_) return cand[cand.size() / 2];
  check(hipMemcpyAsync(batch_dev_, batch_host_, b * rec_bytes_, hipMemcpyHostToDevice, s), "upload batch");
  hipEvent_t e0, e1;
  check(hipEventCreate(&e0), "hipEventCreate");
  check(hipEventCreate(&e1), "hipEventCreate");
  BatchLaunch best = cand.front();
  float best_ms = std::numeric_limits<float>::max();
  try {
    for (const auto& c : cand) {
      launchBatchSpectrum(kind, b, c);                    // warm-up
      check(hipEventRecord(e0, s), "hipEventRecord");
      launchBatchSpectrum(kind, b, c);
      check(hipEventRecord(e1, s), "hipEventRecord");
      check(hipEventSynchronize(e1), "tuning");
      float ms = 0;
      check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
      if (ms < best_ms) { best_ms = ms; best = c; }
    }
  } catch (...) {
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    throw;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return best;
}

// The launch shape of (kind, table precision, batch size): tuned on first use
BatchLaunch DeviceEngine::tuned(ModelKind kind, size_t batch) {
  const TuneKey key{int(kind), int(precision_), batch};
  for (auto& t : tuned_)
    if (t.first.kind == key.kind && t.first.precision == key.precision && t.first.batch == key.batch) {
      last_launch_ = t.second;
      return t.second;
    }
  const BatchLaunch launch = tune(kind, batch);
  tuned_.push_back({key, launch});
  last_launch_ = launch;
  return launch;
}

void DeviceEngine::releaseGraph() {
  if (graph_exec_) (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph_exec_));
  graph_exec_ = nullptr;
  graph_key_ = TuneKey{-1, -1, 0};
}

void DeviceEngine::evaluateBatch(ModelKind kind, size_t batch) { evaluateBatch(kind, batch, false); }

void DeviceEngine::evaluateBatch(ModelKind kind, size_t batch, bool staged) {
  if (staged && (!stage_blob_ || batch > stage_capacity_)) raise(kInternal, "device staging not prepared");
  if (species_stride_ > kMaxSlots) raise(kInvalidInput, "the batched kernels take at most 16 tabulated species");
  if ((hminus_ || cloud_models_ > 0) && precision_ != TablePrecision::fp64)
    raise(kInvalidInput, "the H- continuum and cloud layers take FP64 tables");
  if (batch == 0 || batch > batch_capacity_) raise(kInternal, "batch larger than the staged records");
  if ((kind == ModelKind::transmission) != transmission_) raise(kInvalidInput, "model kind does not match the engine");
  check(hipSetDevice(device_), "hipSetDevice");
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const TuneKey key{int(kind), int(precision_), batch};
  auto same = [](const TuneKey& a, const TuneKey& b) {
    return a.kind == b.kind && a.precision == b.precision && a.batch == b.batch;
  };
  const BatchLaunch launch = tuned(kind, batch);
  auto sequence = [&] {
    if (staged) launchStage(batch);
    else check(hipMemcpyAsync(batch_dev_, batch_host_, batch * rec_bytes_, hipMemcpyHostToDevice, s), "upload batch");
    launchBatchSpectrum(kind, batch, launch);
    launchBatchRest(kind, batch);
    if (staged)
      check(hipMemcpyAsync(stage_neglect_host_, stage_neglect_, batch * sizeof(int), hipMemcpyDeviceToHost, s),
            "read neglect flags");
  };
  if (profiling_) check(hipEventRecord(static_cast<hipEvent_t>(event_start_), s), "hipEventRecord");
  if (use_graph_) {
    if (!graph_exec_ || !same(graph_key_, key) || graph_staged_ != staged) {
      releaseGraph();
      check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "begin graph capture");
      hipGraph_t graph = nullptr;
      try {
        sequence();
      } catch (...) {
        (void)hipStreamEndCapture(s, &graph);
        if (graph) (void)hipGraphDestroy(graph);
        throw;
      }
      check(hipStreamEndCapture(s, &graph), "end graph capture");
      hipGraphExec_t exec = nullptr;
      const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      check(e, "instantiate graph");
      graph_exec_ = exec;
      graph_key_ = key;
      graph_staged_ = staged;
    }
    check(hipGraphLaunch(static_cast<hipGraphExec_t>(graph_exec_), s), "launch graph");
  } else {
    sequence();
  }
  last_used_graph_ = use_graph_;
  if (profiling_) check(hipEventRecord(static_cast<hipEvent_t>(event_stop_), s), "hipEventRecord");
  check(hipStreamSynchronize(s), "batch evaluation");
  if (profiling_) {
    float ms = 0;
    check(hipEventElapsedTime(&ms, static_cast<hipEvent_t>(event_start_), static_cast<hipEvent_t>(event_stop_)),
          "hipEventElapsedTime");
    batch_ms_ += ms;
  }
  batch_evaluations_ += batch;
}

void DeviceEngine::copyBatchBins(size_t batch, std::vector<double>& out) {
  out.resize(batch * n_bins_);
  copyDoubles(out.data(), batch_bins_, out.size());
}

void DeviceEngine::copyBatchSpectrum(ModelKind kind, size_t batch, double* host) {
  hipStream_t s = static_cast<hipStream_t>(stream_);
  const Records rec{batch_dev_, rec_bytes_, rec_levels_, rec_species_, rec_adjoint_, rec_shifts_, groups_};
  const int n = int(n_points_), mode = kind == ModelKind::emission ? 0 : (kind == ModelKind::eclipse ? 1 : 2);
  streamOut(batch * n_points_, host, [&](size_t first, size_t count, double* out) {
    hipLaunchKernelGGL(batchSpectrumKernel, dim3(unsigned((count + kBatchBlock - 1) / kBatchBlock)),
                       dim3(kBatchBlock), 0, s, batch_flux_, stride_, wavenumber_, wavelength_, rec, mode, n, first,
                       int(count), out);
    check(hipGetLastError(), "batch spectrum kernel");
  });
}

void DeviceEngine::releaseBatch() {
  releaseGraph();
  if (batch_host_) (void)hipHostFree(batch_host_);
  if (batch_ll_host_) (void)hipHostFree(batch_ll_host_);
  for (void* p : {(void*)batch_dev_, (void*)batch_flux_, (void*)batch_bins_, (void*)batch_chunk_sums_, (void*)batch_ll_,
                  (void*)batch_chord_, (void*)batch_chord32_, tables_low_, (void*)table_base_})
    deviceFree(p);
}

}  // namespace bear_amd
