// Host-side launchers of the precompute and lookup kernels.
#ifndef ATMO_KERNELS_H_
#define ATMO_KERNELS_H_

#include <hip/hip_runtime.h>

#include "atmo_device.h"

namespace atmo {

// One launch of a pass over a set of jobs. Block b of the launch belongs to
// job i with first_block[i] <= b < first_block[i + 1] (device arrays).
struct PassLaunch {
  const Job* jobs;
  const int* first_block;
  int njobs;
  int total_blocks;
  int max_nnu;  // largest nu size among the jobs (LDS sizing)
  int max_ew;   // largest irradiance width among the jobs (LDS sizing)
  int max_w;    // largest packed row (nu x mu_s texels) among the jobs
  int min_w;    // smallest packed row among the jobs
  int max_lds_w;  // longest packed row of at most kMsMaxRow texels (0: none)
  int kinds;    // kJobsF32 | kJobsAcc64: which kinds of jobs the launch holds
  int tile;     // tile shape of the jobs (scattering density, multiple
                // scattering): every job of a launch has the same one
  int dj_kinds;  // dj_kind of the jobs, or-ed
  int ss_kinds;    // ss_kind of the jobs, or-ed
  size_t ss_lds;   // largest ss_lds of the jobs
  int sd_kinds;    // 1 << sd_split of the jobs, or-ed
  int arc_kinds;   // arc_kind of the jobs, or-ed
  size_t arc_lds;  // largest arc_lds of the jobs
};

constexpr int kDjF32 = 1;    // delta J as RGB float (FP32-storage jobs)
constexpr int kDjRgb21 = 2;  // delta J as 3 x 21-bit floats (FP16-storage jobs)
constexpr int kDjPairs = 4;  // the same, read two texels at a time (ms_pairs)

constexpr int kJobsF32 = 1;    // jobs accumulating S and SM in FP32
constexpr int kJobsAcc64 = 2;  // illuminance-mode jobs with FP64 accumulators

constexpr int kBlock = 256;

// Tile shapes of the two passes that dominate Init, picked per LUT size
// class by the autotuner (autotune.cpp). Every shape computes each texel
// with the same operations in the same order, so the LUTs do not depend on
// the choice.
//
// Scattering density direction by direction: nu outputs per thread (they share the phase
// function of the outgoing direction) and threads per block. A (r, mu_s) plane of
// MU x ceil(NU / chunk) threads is split into ceil(plane / block) blocks,
// each of which builds the plane's nu tables in LDS.
struct SdTile {
  int chunk, block;
};
constexpr int kSdTiles = 6;
constexpr SdTile kSdTile[kSdTiles] = {{4, 256}, {2, 256}, {1, 256},
                                      {4, 128}, {2, 128}, {4, 64}};
// Default shape: 4 nu per thread, in blocks of 128 threads when a plane has
// at most 256 threads (MU x ceil(NU / 4)), else 256. Measured on MI355X
// with the other shapes: at MU x NU = 128 x 8 (a 256-thread plane) the
// 128-thread blocks are 4% faster; at 256 x 16 (1024) the
// 256-thread blocks are, the blocks then rebuilding a plane's tables from
// a LUT beyond the caches 4 times instead of 8.
ATMO_HD int sd_default_tile(int nmu, int nnu) {
  return nmu * ((nnu + 3) / 4) <= 256 ? 3 : 0;
}

// FP16-storage models of up to kFixedTexels texels keep the bits of their tables
// (half_precision in include/atmo.h): the order in which their sums of float32 were
// always made. FP16 rounding turns a difference of 1e-7 of a sum into the last bit of
// 9e-5 of the texels (arc sums for the orders >= 3, 1.05M texels), and
// GetSkyRadianceToPoint, a difference of two lookups, that into up to 4e-3 of the rms
// radiance: within the format's error, but a model would shade differently from LUT
// files and models made before. The price, ms per Init by directions | arcs and split
// order 2, on MI355X:
//   texels    3 wavelengths, 4 orders   15, 4          15, 8
//   8192      .77 | .33                 .81 | .46      1.6 | .84
//   262144    .89 | .58                 2.0 | 1.6      3.7 | 2.6
//   1.05M     1.54 | 1.35               6.2 | 4.9      12.1 | 8.2
//   2.1M      2.7 | 2.4                 12.5 | 9.8     24.2 | 16.5
//   4.2M      5.2 | 4.7                 24.3 | 19.3    48.0 | 32.9
//   8.4M      9.8 | 8.9                 47.5 | 37.8    94.0 | 66.8
//   16.8M     20.1 | 19.5               96.6 | 78.9    193 | 140
// The share is much the same at every size, so the line is no crossover: it is where
// 8 orders cost 15 ms more, at four times the default sizes. A table beyond it takes
// the time, up to 53 ms, and its last bits are not promised.
constexpr int64_t kFixedTexels = int64_t{1} << 22;
ATMO_HD bool fixed_sums(const Job& j) {
  return j.half_luts != 0 &&
         static_cast<int64_t>(j.nr) * j.nmu * j.nmus * j.nnu <= kFixedTexels;
}

// Whether the density of the orders >= 3 is made of arc sums (density_arcs.h) or
// direction by direction. The arcs' terms serve all iterations of a model, and are
// 2 + 2/3 NU in number: with one iteration and many NU the directions are faster.
// Measured on MI355X, ms per order, 3 wavelengths, directions | arcs:
//   NU 16, 8.4M texels 1.43 | 1.32;  NU 20, 2.6M .55 | .54, 5.2M .99 | 1.07
//   NU 24, 1.6M .42 | .40, 2.0M .42 | .48, 3.1M .60 | .73, 12.6M 2.24 | 2.88
//   NU 32, 2.1M .45 | .49, 8.4M 1.66 | 1.89
// With 6 wavelengths the arcs are 1.4 times as fast at the least.
constexpr int kArcMaxNu = 20;
constexpr int64_t kArcTexels = 1900000;
ATMO_HD bool arc_sums(const Job& j) {
  const int64_t n = static_cast<int64_t>(j.nr) * j.nmu * j.nmus * j.nnu;
  return !fixed_sums(j) && !(j.niter == 1 && j.nnu >= kArcMaxNu && n >= kArcTexels);
}

// Grids too small to fill the GPU at 4 outputs per thread: several threads
// share an output, each summing some of the zenith angles, whatever the tile
// shape. A job takes the first of these whose 'texels' it does not exceed (of
// all its model's iterations), or none. Measured on MI355X (ms, 3 wavelengths
// unless given; the shape of sd_default_tile in the first column):
//   texels               1 part   4     8     16
//   8192                  .287    -     -    .021
//   32768                 .244  .096  .057   .032
//   65536                 .243    -     -    .058
//   131072                .268  .101  .078   .108
//   262144                .274  .134  .137   .204
//   524288                .334  .240  .248   .394
//   1048576               .491  .423  .484   .774
//   3 x 391230 (9 wl)     .63   .573  .664
//   5 x 262144 (15 wl)    .518  .543  .600   .973
struct SdSplit {
  int chunk, block, parts, texels;
};
constexpr int kSdSplits = 3;
constexpr SdSplit kSdSplit[kSdSplits] = {
    {1, 1024, 16, 1 << 16}, {4, 512, 8, 1 << 18}, {4, 256, 4, 1250000}};
// The job's index into kSdSplit, or kSdSplits.
ATMO_HD int sd_split(const Job& j) {
  const int64_t n = static_cast<int64_t>(j.nr) * j.nmu * j.nmus * j.nnu * j.niter;
  int i = fixed_sums(j) ? kSdSplits : 0;
  while (i < kSdSplits && n > kSdSplit[i].texels) ++i;
  return i;
}

// Whether the density of an order takes the job's tile shape (kSdTile): the directions
// with a thread per output.
ATMO_HD bool sd_uses_tile(const Job& j, int order) {
  return order == 2 ? sd_split(j) == kSdSplits : !arc_sums(j);
}

// Single scattering: blocks of 'block' texels of a packed row, for 'nit'
// iterations of a model. Where 'staged', the block blends the transmittance
// rows of each sample in LDS for ss_rows of them; otherwise every texel gathers
// its four transmittance texels.
//
// A staged block blends all TW columns for each sample, however few texels it
// has, and has a barrier per sample: 2 columns a thread are worth it, or 4 in
// blocks of 512 that serve several iterations. Rows of 513..768 texels, which
// leave a third of 512-thread blocks idle, take blocks of 256 while TW is 2 columns
// a thread. Gathering blocks of one iteration run three to a CU, so up to
// kSsGatherBlocks of them are a single round that staging does not shorten;
// from 3 iterations on it does, at 512. Measured on MI355X (ms; wl:
// wavelengths), gathered | staged:
//   row of 256, TW 256, 3 wl: 4096 rows .147 | .131, 512 rows .028 | .034
//   row of 512, TW 256, 3 wl: 384 rows .038 | .041, 400 rows .045 | .040; 15 wl:
//     192 rows .092 | .118, 256 rows .112 | .119, 496 rows .210 | .170
//   row of 297, TW 256, 15 wl: 192 rows .090 | .098, 256 rows .113 | .101
//   row of 600, TW 256, 432 rows, 15 wl: .240 | .229 (256 threads), .308 (512);
//     row of 768, TW 256, 512 rows, 6 wl: .161 | .117 (256), .141 (512)
//   row of 256, TW 1024, 9 wl: 800 rows .152 | .220; row of 512, TW 2048, 3 wl:
//     400 rows .060 | .075
//   row of 65, 16128 rows, TW 4096: .34 | 9.0 (3 wl), 1.8 | 50 (15 wl)
// Iterations share a block that gathers where three blocks per CU are left and
// the lines that the block reads per sample, in each iteration 2 rows of at most
// one line per texel, leave room in the 32 KB L1. Alone | shared: row of 65, 4032
// rows, TW 256, 15 wl .48 | .365; row of 96, 10880 rows, TW 1024, 6 wl .59 | .85;
// row of 32, TW 256, 15 wl: 2048 rows .126 | .117, 512 rows .046 | .069.
constexpr int kSsIters = 5;
constexpr int kSsRowBytes = 64 << 10;  // at most, if iterations share a block
constexpr int kSsStagedWidth = 160;    // shortest row
constexpr int kSsStagedBlocks = 512;   // of 256 texels, 3 iterations or more
constexpr int kSsGatherBlocks = 768;
constexpr int kSsGatherBytes = 24 << 10;
constexpr ATMO_HD int ss_rows(int nit, bool staged) { return !staged ? 0 : (nit < 3 ? 1 : 2); }
template <bool kF64>
constexpr int kSsBuffers = kF64 ? 1 : 2;
ATMO_HD size_t ss_row_bytes(const Job& j, int nit, bool staged) {
  const size_t texels = static_cast<size_t>(ss_rows(nit, staged)) * j.tw * 3;
  return texels * (j.acc64 ? kSsBuffers<true> * sizeof(double)
                           : kSsBuffers<false> * sizeof(float));
}
struct SsTiling {
  int block;
  bool staged;
  int nit;  // 0: the job is served by the blocks of an earlier iteration
  bool fixed;  // FP32 job of fixed_sums: k_single_scattering_fixed instead
  ATMO_HD explicit SsTiling(const Job& j) {
    const int w = j.nnu * j.nmus, most = j.niter < kSsIters ? j.niter : kSsIters;
    const bool thirds = w > 2 * kBlock && w <= 3 * kBlock && j.tw <= 2 * kBlock;
    const int wide = w > kBlock && !thirds ? 2 * kBlock : kBlock;
    const int columns = most > 1 ? (wide > kBlock ? 4 : 2) * wide
                                 : 2 * (w < kBlock ? w : wide);
    fixed = fixed_sums(j) && !j.acc64;
    staged = w >= kSsStagedWidth && j.tw <= columns &&
             blocks(j, kBlock) >= (most > 2 ? kSsStagedBlocks : kSsGatherBlocks + 1) &&
             (most == 1 || ss_row_bytes(j, most, true) <= kSsRowBytes);
    block = staged ? wide : (w > 64 ? kBlock : 64);
    const int lines = (j.tw + 7) / 8 < w ? (j.tw + 7) / 8 : w;  // 8 texels each
    const bool share = staged || (blocks(j, block) >= kSsGatherBlocks &&
                                  most * 2 * lines * 128 <= kSsGatherBytes);
    nit = 1;
    if (most > 1 && share) {
      const int left = j.niter - j.it;
      nit = j.it % kSsIters != 0 ? 0 : (left < kSsIters ? left : kSsIters);
    }
  }
  static ATMO_HD int64_t blocks(const Job& j, int block) {
    return static_cast<int64_t>(j.nr) * j.nmu * ((j.nnu * j.nmus + block - 1) / block);
  }
};
// PassLaunch::ss_kinds.
constexpr int ss_kind(bool f64, int nit, int block, bool staged) {
  return 1 << ((f64 ? nit : 0) +
               (block > kBlock ? 3 : staged ? 2 : block == kBlock ? 1 : 0) * (kSsIters + 1));
}
constexpr int kSsFixed = 1 << (4 * (kSsIters + 1));
ATMO_HD int ss_kind(const Job& j) {
  const SsTiling t(j);
  return t.nit == 0 ? 0
                    : t.fixed ? kSsFixed : ss_kind(j.acc64 != 0, t.nit, t.block, t.staged);
}
inline size_t ss_lds(const Job& j) {
  const SsTiling t(j);
  return ss_row_bytes(j, t.nit, t.staged);
}

// Scattering density of orders >= 3 (density_arcs.h): a block of 8 waves
// takes arc_cols mu_s columns and arc_mus mu rows of a layer, for the
// wavelengths of up to kArcIters Precompute iterations. Each wave has
// arc_tiles tiles of 64 (mu, nu) texels of a column: 512 rows of 2 columns,
// 256 of 4, or 128 or 64 of 8, so that the source texels of an angle (cols x
// kArcIters x NU) are at most one per thread. At most kArcMus mu rows' prefix
// sums fit a block's LDS: 13/16 of the rows or more have texels from NU = 7 on
// (all at 8, 16 and 32), 1/2 to 1 below.
constexpr int kArcMaxCols = 8;
constexpr int kArcMus = 16;
constexpr int kArcIters = 5;
ATMO_HD int arc_cols(int nnu) { return nnu >= 26 ? 2 : (nnu >= 13 ? 4 : 8); }
ATMO_HD int arc_tiles(int nnu) { return nnu * kArcMus > 64 ? 2 : 1; }
ATMO_HD int arc_mus(int nnu) {
  const int mus = 8 / arc_cols(nnu) * arc_tiles(nnu) * 64 / nnu;
  return mus < kArcMus ? mus : kArcMus;
}
// The instance that serves a job: its tiles per wave and the groups of 4
// wavelengths of its iterations (those of the kArcIters from j.it on).
ATMO_HD int arc_kind_bit(int tiles, int groups) { return 1 << (4 * (tiles - 1) + groups - 1); }
ATMO_HD int arc_kind(const Job& j) {
  const int left = j.niter - j.it;
  const int nit = left < kArcIters ? left : kArcIters;
  return arc_kind_bit(arc_tiles(j.nnu), (3 * nit + 3) / 4);
}

// Multiple scattering: packed rows of at most kMsMaxRow texels are processed
// through LDS by blocks of kMsTile[tile].block threads, each thread holding
// kMsTile[tile].tpt texels: ms_rows_per_block(W, capacity) whole rows per
// block, capacity = tpt x block texels (0: the row is too long for LDS and
// takes the gather kernel; -1: it does not fit this tile). Rows of up to
// 1024 texels take 2 texels per thread in 512-thread blocks rather than 4 in
// 256: the blocks hold the same rows and the kernel runs at more waves per
// SIMD (the high-resolution pass, rows of 1024 texels: 83.0 against 88.8 ms
// per Init with FP32 storage, 81.5 against 83.0 with FP16; 1 texel in
// 1024-thread blocks took 103-105 ms).
struct MsTile {
  int tpt, block;
};
constexpr int kMsTiles = 3;
constexpr MsTile kMsTile[kMsTiles] = {{1, 256}, {2, 256}, {2, 512}};
constexpr int kMsMaxRow = 4 * kBlock;
constexpr int ms_tile_capacity(int t) { return kMsTile[t].tpt * kMsTile[t].block; }
// Rows per block are capped at 4 (blocks of 256 texels) or 8, which keeps
// the block's LDS (2 x capacity RGB floats + 3.2 KB of samples per row)
// under 64 KB.
ATMO_HD int ms_rows_per_block(int w, int capacity) {
  if (w > kMsMaxRow) return 0;
  if (w > capacity) return -1;
  const int r = capacity / w;
  const int cap = capacity <= kBlock ? 4 : 8;
  return r < cap ? r : cap;
}
// Rows per block of a tile of tpt texels per thread, whose texels are in one row
// (odd rows of two-texel tiles leave a thread's second texel idle).
ATMO_HD int ms_tile_rows(int w, int tpt, int block) {
  const int r = ms_rows_per_block(w, tpt * block), m = block / ((w + tpt - 1) / tpt);
  return r < m ? r : m;
}
// Whether the threads of an FP16 job load two neighbouring texels of delta J. With
// one texel per thread, half of a block's waves then load, which a launch of few
// blocks waits for. Measured on MI355X, us, a texel at a time | two (15 wavelengths
// unless given):
//   rows of 256: 1024 blocks (3 wl) 48 | 48, 5120 171 | 168, 20480 645 | 620;
//     64 (3 wl) 31 | 35
//   rows of 64: 256 blocks (3 wl) 31 | 35, 1280 64 | 68, 5120 179 | 183
//   rows of 32: 2560 blocks 146 | 126, 640 52 | 51, 128 (3 wl) 29 | 32
//   rows of 96, in 192 of the 256 threads: 2048 blocks (3 wl) 65 | 69, 10240 279 | 290
// With two texels per thread every wave loads either way: rows of 1024, 64 rows
// (3 wl) 61 | 49.
constexpr int kMsPairBlocks = 2048;
constexpr int kMsPairShort = 32, kMsPairLong = 128;  // not the rows between
ATMO_HD bool ms_pairs(const Job& j) {
  if (j.half_luts == 0) return false;
  const MsTile t = kMsTile[j.ms_tile];
  if (t.tpt > 1) return true;
  const int w = j.nnu * j.nmus, rpb = ms_tile_rows(w, t.tpt, t.block);
  if (rpb <= 0 || (w > kMsPairShort && w < kMsPairLong)) return false;
  const int64_t rows = static_cast<int64_t>(j.nr) * j.nmu;
  return (rows + rpb - 1) / rpb * j.niter >= kMsPairBlocks;
}
// Whether the two texels of a thread are a block's width apart, so that all waves of
// a block with one row have texels, and not half a row, which leaves some waves idle
// and the others full. Better where a CU has one block: rows of 640 texels, FP32, us,
// half a row | a block apart: 64 blocks 53 | 47, 256 56 | 50, 320 62 | 68, 1024 119 |
// 125.
constexpr int kMsSpreadBlocks = 256;
ATMO_HD bool ms_spread(const Job& j) {
  const MsTile t = kMsTile[j.ms_tile];
  return j.half_luts == 0 && t.tpt > 1 && ms_tile_rows(j.nnu * j.nmus, t.tpt, t.block) == 1 &&
         static_cast<int64_t>(j.nr) * j.nmu * j.niter <= kMsSpreadBlocks;
}
ATMO_HD int dj_kind(const Job& j) {
  return j.half_luts == 0 ? kDjF32 : (j.ms_paired ? kDjPairs : kDjRgb21);
}
// The smallest tile that holds a row of w texels.
ATMO_HD int ms_default_tile(int w) {
  if (w <= kBlock) return 0;
  if (w <= 2 * kBlock) return 1;
  return 2;
}
// Row orders of the multiple-scattering blocks (Job::ms_row_order):
// 0 r-major (the LUT's own order), 1 mu-major, 2 ray order (rows sorted by
// the impact parameter of their view ray, Job::ms_rows). The samples of a
// row's ray lie on the ray's line, whose points have the same impact
// parameter r sqrt(1 - mu^2), so rows of nearly equal impact parameter read
// nearly the same source rows of the scattering density: in ray order the
// blocks resident on one XCD share their source rows in its L2.
constexpr int kMsRowOrders = 3;
// Default: ray order at every size. At the reference sizes (a 12.6 MB
// delta J per iteration) it fetches 0.25 GB per launch of 5 iterations
// against 1.05 GB in r-major order, and runs 1.4% faster.
ATMO_HD int ms_default_row_order(int nr, int nmu, int w) {
  (void)nr;
  (void)nmu;
  (void)w;
  return 2;
}

// Blocks one job needs for each pass.
int blocks_optical_depth(const Job& j);
int blocks_transmittance(const Job& j);
int blocks_direct_irradiance(const Job& j);
int blocks_single_scattering(const Job& j);
int blocks_scattering_density(const Job& j);
int blocks_density_arcs(const Job& j);
size_t arc_lds(const Job& j);  // LDS bytes of a block of launch_density_arcs
int blocks_indirect_irradiance(const Job& j);
int blocks_multiple_scattering(const Job& j);
int blocks_half_conversion(const Job& j);
int blocks_lookup_copy(const Job& j);
int blocks_combine(const Job& j);

// The optical depths of the jobs' transmittance texels into their OD (one
// job per model), read by launch_transmittance for jobs whose OD is set.
hipError_t launch_optical_depth(const PassLaunch& p, hipStream_t s);
hipError_t launch_transmittance(const PassLaunch& p, hipStream_t s);
hipError_t launch_direct_irradiance(const PassLaunch& p, hipStream_t s);
hipError_t launch_single_scattering(const PassLaunch& p, hipStream_t s);
// The scattering density direction by direction (order 2, and the orders >= 3
// of the jobs that are not arc_sums), and that of an order >= 3 by arc sums. In the
// latter the jobs of a model's Precompute iterations follow each other in
// p.jobs, and the blocks of the first of every kArcIters serve all of them.
hipError_t launch_scattering_density(const PassLaunch& p, int order, hipStream_t s);
hipError_t launch_density_arcs(const PassLaunch& p, hipStream_t s);
// 'order' is the order of the scattering read by the pass (>= 1).
hipError_t launch_indirect_irradiance(const PassLaunch& p, int order,
                                      hipStream_t s);
hipError_t launch_multiple_scattering(const PassLaunch& p, hipStream_t s);
// FP16 storage of the scattering LUTs of half-precision jobs:
// launch_clear_max (one block per job) resets the per-channel maxima, then
// launch_to_half (blocks_half_conversion blocks per job) computes the maxima
// and writes the scaled FP16 texels.
hipError_t launch_clear_max(const PassLaunch& p, hipStream_t s);
// Illuminance mode: sums the Precompute iterations' FP64 accumulators into S
// and SM, and their irradiance accumulators into E (blocks_combine blocks
// per job; the job's niter, S64, SM64 and E_it name the accumulators).
hipError_t launch_acc64_to_f32(const PassLaunch& p, hipStream_t s);
hipError_t launch_to_half(const PassLaunch& p, hipStream_t s);
// The lookup copy of S and SM, in quads (blocks_lookup_copy blocks per
// job).
hipError_t launch_interleave(const PassLaunch& p, hipStream_t s);

// Lookups (one ray / point per thread). 'job' is a device pointer, 'combined'
// its Job::combined, 'copy' whether it has a lookup copy (if that changes before a
// captured launch runs, the kernels read S and SM themselves). With
// 'luminance' the results are scaled by the job's radiance-to-luminance
// factors (the Luminance API of atmosphere/model.cc:252-281).
hipError_t launch_sky_radiance(const Job* job, bool combined, bool copy, int64_t n,
                               const float* camera, const float* view_ray,
                               const float* shadow_length,
                               const float* sun_direction, float* radiance,
                               float* transmittance, int luminance, hipStream_t s);
hipError_t launch_sky_radiance_to_point(const Job* job, bool combined, int64_t n,
                                        const float* camera,
                                        const float* point,
                                        const float* shadow_length,
                                        const float* sun_direction,
                                        float* radiance, float* transmittance,
                                        int luminance, hipStream_t s);
// Seeded synthetic query batch (camera, view ray, sun direction, point,
// normal: n x 3; shadow length: n).
hipError_t launch_generate_queries(uint64_t seed, int64_t n, double bottom_radius,
                                  double top_radius, double max_altitude,
                                  double max_distance, double max_sun_zenith,
                                  float* camera, float* view_ray, float* sun_direction,
                                  float* point, float* normal, float* shadow_length,
                                  hipStream_t s);
hipError_t launch_sun_and_sky_irradiance(const Job* job, int64_t n,
                                         const float* point,
                                         const float* normal,
                                         const float* sun_direction,
                                         float* sun_irradiance,
                                         float* sky_irradiance, int luminance,
                                         hipStream_t s);

}  // namespace atmo

#endif  // ATMO_KERNELS_H_
