// Scattering density of orders >= 3 (functions.glsl:1163-1260, :1348-1367)
// by arc sums on the matrix cores. Part of precompute.hip.
//
// At a texel (r, mu, mu_s, nu) and an incident zenith angle theta, the
// incident radiance is a function of the cosine nu1 between the incident
// direction and the sun only: linear interpolation in t = (nu1 + 1) / 2
// (NU - 1) between NU values of (r, mu_s, theta), plus, for directions that
// hit the ground, linear interpolation of a row of the irradiance LUT in a
// coordinate linear in nu1. Such a function is
//   f(t) = u + v (t - t_lo) + sum over breakpoints k of D_k max(0, t - k),
// D_k the change of slope at k. With t = tA + S (sx cos phi + sy sin phi)
// and phase function weights p(phi) of the outgoing direction, the quadrature
// over the 32 azimuths phi is
//   sum_m p_m f(t_m) = sum_k D_k G_k,
//   G_k / S = ((tA - k) / S) P + sx C + sy E,
// where P, C and E are the sums of p, p cos and p sin over the azimuths with
// t > k: an arc centred on the sun's azimuth phi_s = atan2(sy, sx), so a
// difference of two prefix sums over the azimuths. (u + v t is two terms of
// the same form over the whole circle.) The prefix sums depend on (r, mu,
// theta) only, G on the texel's geometry only, D on (r, mu_s, theta) and the
// wavelength: the densities of all wavelengths and texels of a (r, mu_s)
// plane are one matrix product G x D, with no per-direction work. It is the
// same quadrature as direction by direction: an azimuth within rounding of a
// breakpoint contributes max(0, t - k) = 0 within rounding on either side.
//
// Per texel and angle there are about 2 + 2/3 NU terms (11 at NU = 16, 6 at 8)
// instead of 32 azimuths, and their G serve all wavelengths of the model.
// (With one iteration and many NU the directions are faster: arc_sums.) Against the
// kernel that interpolated per direction, wavelength triple and
// texel (its FP32 arithmetic issued at 0.98 of the ceiling), per order, on
// MI355X:
//   texels, wavelengths          direction by direction   arcs
//   16.8M (NU 16), 15            14.2 ms                  4.7 ms
//   16.8M (NU 16), 3             2.99 ms                  2.93 ms
//   1.05M (NU 8), 15             0.92 ms                  0.21 ms
//   1.05M (NU 8), 3              0.23 ms                  0.146 ms
// At 16.8M texels with 15 wavelengths vector instructions issue in 61% of the
// cycles, the matrix units are busy 28%, and the LDS is busy 55%.
//
// The outgoing phase function is Rayleigh's plus Mie's with a factor per
// wavelength, so there are two G per term and two sums, combined at the end.
#ifndef ATMO_DENSITY_ARCS_H_
#define ATMO_DENSITY_ARCS_H_

#include <hip/hip_runtime.h>

#include "atmo_device.h"
#include "kernels.h"
#include "pass_common.h"

namespace atmo {
namespace {

using f32x4 = float __attribute__((ext_vector_type(4)));

constexpr int kArcWaves = 8;  // waves per block
// Prefix sums over the azimuths -16 .. 31 (the arcs reach half a turn from
// azimuths in [0, 16)): slot i holds the sums over azimuths < i - 16.
constexpr int kArcSlots = 49;
constexpr float kSteps = static_cast<float>(16.0 / kPi);  // azimuths per radian

// One incident zenith angle of a block's layer.
struct ArcTheta {
  double ct, ga;   // cos theta; ground normal . sun = ga mu_s + gb nu1
  float st, dw, wy, gb;
  int row0, row1;  // mu rows of the incident radiance
  int ground;
  int chunks;      // steps: chunks of terms of the column with most terms
};
// The terms of one (theta, mu_s column): two over the whole circle, then nv
// breakpoints klo + 1 .. klo + nv of the incident radiance and ne breakpoints
// jlo + 1 .. jlo + ne of the ground irradiance, whose texel coordinate is
// ea + eb t.
struct ArcColumn {
  double ta;
  float s, inv_rt;  // S, and 2 over the range of t
  float ea, eb, inv_eb;
  float e_at;       // ground irradiance coordinate at t = klo, from jlo
  short klo, nv;
  short jlo, ne;
};
struct alignas(16) ArcShared {
  ArcTheta th[kTheta];
  float gf[kTheta][16];  // ground: transmittance * albedo / pi * d_omega
  float cr[16], cm[16];  // scattering coefficients of both phase functions
  double mu[kArcMus], wx[kArcMus];
  double mu_s[kArcMaxCols], ws[kArcMaxCols];
};
// The rest of a block's LDS, sized by NU: byte offsets.
struct ArcLayout {
  int cols, terms, mus;  // mu_s columns, terms held per column, mu rows
  int term0;     // float [2][cols][terms][16]: wavelength n at 4 (n % 4) + n / 4
  int par0;      // float2 [2][cols][terms]: (tA - k) / S, half angle + 17
  int col0;      // ArcColumn [kTheta][cols]
  int count0;    // int [kTheta][cols]: terms
  // Prefix sums of p, p cos, p sin (Rayleigh) and p (Mie), float4
  // [2][mus][kArcSlots], then of p cos and p sin (Mie), float2. Lanes read
  // them at random within a half turn. 24-byte slots read by 8-byte loads took
  // 1.6 times the LDS cycles, 16-byte slots for the second part (one address
  // for both reads) 1.2 times.
  int prefix0;
  int node0;     // float [2][cols][NU][16]: incident radiance of two angles
  int bytes;
  ATMO_HD explicit ArcLayout(int nnu) {
    cols = arc_cols(nnu);
    mus = arc_mus(nnu);
    terms = cols == 8 ? 14 : (cols == 4 ? 28 : 36);  // all but some of the ground's
    const int held = cols * terms;
    term0 = static_cast<int>(sizeof(ArcShared));
    par0 = term0 + 2 * held * 64;
    col0 = par0 + 2 * held * 8;
    count0 = col0 + kTheta * cols * static_cast<int>(sizeof(ArcColumn));
    prefix0 = count0 + kTheta * cols * 4;
    node0 = prefix0 + 2 * mus * kArcSlots * 24;
    bytes = node0 + 2 * cols * nnu * 64;
    // The tiles on their way out take the place of the sums and nodes.
    const int stage = prefix0 + kArcWaves * 64 * 17 * 4;
    if (bytes < stage) bytes = stage;
  }
};
static_assert(sizeof(ArcShared) % 16 == 0 && sizeof(ArcColumn) == 40, "LDS layout");

// Inclusive sum over the lanes 0 .. l of each row of 16 lanes.
__device__ __forceinline__ float scan16(float v) {
#define ATMO_SCAN_STEP(ctrl)                                                  \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, \
                                                  0xf, 0xf, true));
  ATMO_SCAN_STEP(0x111)  // row_shr:1
  ATMO_SCAN_STEP(0x112)
  ATMO_SCAN_STEP(0x114)
  ATMO_SCAN_STEP(0x118)
#undef ATMO_SCAN_STEP
  return v;
}

// kTiles: tiles of 64 texels of a column per wave.
// kG: groups of 4 wavelengths, 3 x (the job group's iterations) rounded up.
//
// A block takes arc_cols consecutive mu_s columns and arc_mus mu rows of a
// layer. The product is v_mfma_f32_4x4x1: 16 blocks of 4 texels x 4
// wavelengths x 1 term, so a lane is a texel and a term is the same for the
// whole wave (no terms wasted on padding, and its place on the circle one
// value). It takes 8 cycles per 4 wavelengths. FP32 matrix instructions do
// not overlap vector arithmetic on gfx950 (their busy cycles and the vector
// instructions' add up to the kernel's time), so what counts is the sum of
// both.
template <int kTiles, int kG>
__global__ __launch_bounds__(kArcWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void
k_density_arcs(const Job* __restrict__ jobs, const int* __restrict__ first_block, int njobs) {
  extern __shared__ float4 arc_lds[];
  char* const lds = reinterpret_cast<char*>(arc_lds);
  ArcShared& sh = *reinterpret_cast<ArcShared*>(lds);
  const int ji = find_job(first_block, njobs, blockIdx.x);
  const Job& J = jobs[ji];
  if (arc_kind(J) != arc_kind_bit(kTiles, kG)) return;
  const int nnu = J.nnu, nmus = J.nmus, nmu = J.nmu;
  const ArcLayout L(nnu);
  const int cols = L.cols, mus = L.mus, held = L.terms;
  const int nit = min(kArcIters, J.niter - J.it);
  const int mu_tiles = (nmu + mus - 1) / mus, col_groups = (nmus + cols - 1) / cols;
  // Layer by layer, then mu rows, then columns: the blocks that write the
  // parts of a line of delta J, and those that read the same source rows,
  // follow each other on one XCD.
  const int lb = xcd_contiguous(blockIdx.x - first_block[ji], J.nr * mu_tiles * col_groups);
  const int rest = lb / col_groups;
  const int c0 = __builtin_amdgcn_readfirstlane((lb - rest * col_groups) * cols);
  const int k = __builtin_amdgcn_readfirstlane(rest / mu_tiles);
  const int y0 = __builtin_amdgcn_readfirstlane(rest - k * mu_tiles) * mus;
  const int W = nnu * nmus;
  const int64_t layer = static_cast<int64_t>(k) * nmu;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Term builders: wavelength and term of the lane (lanes past the last
  // whole term idle).
  constexpr int kLanes = 4 * kG, kUnit = 64 / kLanes;
  const int n = lane % kLanes, kk = lane / kLanes;

  float* const terms = reinterpret_cast<float*>(lds + L.term0);
  float2* const pars = reinterpret_cast<float2*>(lds + L.par0);
  ArcColumn* const columns = reinterpret_cast<ArcColumn*>(lds + L.col0);
  int* const counts = reinterpret_cast<int*>(lds + L.count0);
  float4* const prefix4 = reinterpret_cast<float4*>(lds + L.prefix0);
  float* const nodes = reinterpret_cast<float*>(lds + L.node0);
  const int prefix_size = mus * kArcSlots;
  float2* const prefix2 = reinterpret_cast<float2*>(prefix4 + 2 * prefix_size);

  double r, rho;
  s_layer_r(J, k, &r, &rho);
  // This lane's wavelength in the terms: channel ch of job it.
  const int it = n / 3, ch = n - 3 * it;
  const bool on = it < nit;
  // Its irradiance row: a model's iterations follow each other in memory, so
  // 32 bits from the first job's tell their places.
  const uint32_t esrc = 4 * static_cast<uint32_t>((&J)[on ? it : 0].dE - J.dE) + ch;
  auto irradiance = [&](int j) {
    return gload(reinterpret_cast<const float*>(J.dE), static_cast<int64_t>(esrc + 4 * j));
  };

  if (tid < kTheta) {
    const double theta = (tid + 0.5) * (kPi / kTheta);
    const double ct = cos(theta), st = sin(theta);
    const bool g = hits_ground(J, r, ct);
    const Taps ty = axis_taps(s_mu_texel(J, r, ct, g), nmu);
    ArcTheta& t = sh.th[tid];
    t.ct = ct;
    t.st = static_cast<float>(st);
    t.dw = static_cast<float>((kPi / kTheta) * (kPi / kTheta) * st);
    t.wy = ty.w;
    t.row0 = ty.i0;
    t.row1 = ty.i1;
    t.ground = g ? 1 : 0;
    const double dg = dist_bottom(J, r, ct);
    const double len = sqrt(r * r + 2.0 * r * dg * ct + dg * dg);
    t.ga = r / len;
    t.gb = static_cast<float>(dg / len);
  }
  if (tid >= 64 && tid < 64 + mus) {
    const int y = min(y0 + tid - 64, nmu - 1);
    double mu;
    bool ground;
    s_row_mu(J, y, r, rho, &mu, &ground);
    sh.mu[tid - 64] = mu;
    sh.wx[tid - 64] = sqrt(1.0 - mu * mu);
  }
  if (tid >= 128 && tid < 128 + cols) {
    const double mu_s = s_col_mus(J, min(c0 + tid - 128, nmus - 1));
    sh.mu_s[tid - 128] = mu_s;
    sh.ws[tid - 128] = sqrt(fmax(1.0 - mu_s * mu_s, 0.0));
  }
  if (tid >= 192 && tid < 192 + 16) {
    // Both phase functions' factors per wavelength.
    const int i = tid - 192, c = i % 3;
    float cr = 0.0f, cm = 0.0f;
    if (i < 3 * nit) {
      const Job& Jc = (&J)[i / 3];
      const double h = r - J.rb, g = J.g;
      cr = static_cast<float>(Jc.rayleigh[c] * profile_density(J.prof_r, h) *
                              (3.0 / (16.0 * kPi)));
      cm = static_cast<float>(Jc.mie_sca[c] * profile_density(J.prof_m, h) *
                              (3.0 / (8.0 * kPi)) * (1.0 - g * g) / (2.0 + g * g));
    }
    sh.cr[i] = cr;
    sh.cm[i] = cm;
  }
  if (tid >= 256 && tid < 256 + kTheta * nit) {
    // gf of angle i and the wavelengths of job j.
    const int i = (tid - 256) % kTheta, j = (tid - 256) / kTheta;
    const double theta = (i + 0.5) * (kPi / kTheta);
    const double ct = cos(theta), st = sin(theta);
    if (hits_ground(J, r, ct)) {
      const Job& Jc = (&J)[j];
      const float3 tg = transmittance(Jc, Jc.T, r, ct, dist_bottom(J, r, ct), true);
      const double f = 1.0 / kPi * ((kPi / kTheta) * (kPi / kTheta) * st);
      sh.gf[i][3 * j] = static_cast<float>(tg.x * Jc.albedo[0] * f);
      sh.gf[i][3 * j + 1] = static_cast<float>(tg.y * Jc.albedo[1] * f);
      sh.gf[i][3 * j + 2] = static_cast<float>(tg.z * Jc.albedo[2] * f);
    }
  }
  __syncthreads();
  if (tid < kTheta * cols) {
    const int l = tid / cols, s = tid % cols;
    const ArcTheta& t = sh.th[l];
    const double mu_s = sh.mu_s[s];
    const double hn = 0.5 * (nnu - 1);
    ArcColumn c;
    c.s = t.st * static_cast<float>(hn);
    c.ta = (1.0 + mu_s * t.ct) * hn;
    const double rt = sh.ws[s] * t.st * hn;
    c.inv_rt = 1.0f / static_cast<float>(rt);
    const int klo = min(max(static_cast<int>(floor(c.ta - rt)), 0), nnu - 2);
    const int khi = min(static_cast<int>(ceil(c.ta + rt)) - 1, nnu - 2);
    c.klo = static_cast<short>(klo);
    c.nv = static_cast<short>(max(khi - klo, 0));
    c.ea = c.eb = c.inv_eb = c.e_at = 0.0f;
    c.jlo = c.ne = 0;
    if (t.ground) {
      const double he = 0.5 * (J.ew - 1), eb = t.gb * he / hn;
      const double ea = (t.ga * mu_s - t.gb + 1.0) * he;
      const int jlo = min(max(static_cast<int>(floor(ea + eb * (c.ta - rt))), 0), J.ew - 2);
      const int jhi = min(static_cast<int>(ceil(ea + eb * (c.ta + rt))) - 1, J.ew - 2);
      c.jlo = static_cast<short>(jlo);
      c.ne = static_cast<short>(eb > 0.0 ? max(jhi - jlo, 0) : 0);
      c.eb = static_cast<float>(eb);
      c.inv_eb = static_cast<float>(1.0 / eb);
      c.ea = static_cast<float>(ea - jlo);
      c.e_at = static_cast<float>(ea + eb * klo - jlo);
    }
    columns[tid] = c;
    const int count = 2 + c.nv + c.ne;
    counts[tid] = count;
    int most = count;
    for (int i = 1; i < cols; i *= 2) most = max(most, __shfl_xor(most, i));
    sh.th[l].chunks = (most + held - 1) / held;
  }

  // The texels of this lane: rows 64 (tile0 + g) + lane of the block's rows,
  // in column col. With 4 or 2 columns, 2 or 4 waves share a column.
  const int col = wave % cols, tile0 = (wave / cols) * kTiles;
  float sx[kTiles], sy[kTiles], xs[kTiles];
  int base[kTiles];
#pragma unroll
  for (int g = 0; g < kTiles; ++g) {
    const int row = (tile0 + g) * 64 + lane;
    const int slot = row / nnu, nui = row - slot * nnu;
    const bool in = slot < mus;
    base[g] = in ? slot * kArcSlots : 0;
    const double mu = sh.mu[in ? slot : 0], wx = sh.wx[in ? slot : 0], mu_s = sh.mu_s[col];
    const double half_range = wx * sh.ws[col];
    const double grid = clamp_cos(static_cast<double>(nui) / (nnu - 1) * 2.0 - 1.0);
    const double nu = clamp_d(grid, mu * mu_s - half_range, mu * mu_s + half_range);
    const double x = wx == 0.0 ? 0.0 : (nu - mu * mu_s) / wx;
    sx[g] = static_cast<float>(x);
    sy[g] = sqrt_f(static_cast<float>(fmax(1.0 - x * x - mu_s * mu_s, 0.0)));
    // phi_s in azimuth steps, azimuth m at m: a multiple of 2^-18, so that
    // adding and subtracting a half turn is exact and the ends of a whole
    // circle are 32 azimuths apart.
    const float a = atan2f(sy[g], sx[g]) * kSteps - 0.5f;
    xs[g] = rintf(a * 262144.0f) * (1.0f / 262144.0f);
  }
  const float g1 = static_cast<float>(1.0 + J.g * J.g);
  const float mg2 = static_cast<float>(-2.0 * J.g);

  // The nodes of angle l (mu rows blended, times d_omega), at most one item
  // (node, job, column) per thread: loaded and, later, stored.
  const bool has_node = tid < cols * nit * nnu;
  const int is = tid % cols, ij = (tid / cols) % nit, inode = tid / (cols * nit);
  const uint32_t isrc = static_cast<uint32_t>((&J)[ij].dR - J.dR) +
                        static_cast<uint32_t>(layer * W) + min(inode, nnu - 1) * nmus +
                        min(c0 + is, nmus - 1);
  float* const iout = nodes + (is * nnu + inode) * 16 + 3 * ij;
  float3 va, vb;
  auto load_nodes = [&](int l) {
    if (!has_node) return;
    const int64_t src = isrc;
    va = make3(gload(J.dR, src + static_cast<uint32_t>(sh.th[l].row0 * W)));
    vb = make3(gload(J.dR, src + static_cast<uint32_t>(sh.th[l].row1 * W)));
  };
  auto store_nodes = [&](int l) {
    if (!has_node) return;
    const ArcTheta& t = sh.th[l];
    const float w1 = t.wy, w0 = 1.0f - w1;
    float* const o = iout + (l & 1) * cols * nnu * 16;
    o[0] = (w0 * va.x + w1 * vb.x) * t.dw;
    o[1] = (w0 * va.y + w1 * vb.y) * t.dw;
    o[2] = (w0 * va.z + w1 * vb.z) * t.dw;
  };
  // The prefix sums of angle l: 16 lanes per mu row.
  auto build_prefix = [&](int l) {
    const ArcTheta& t = sh.th[l];
    const int slot = wave * 4 + (lane >> 4), m = lane & 15;
    if (slot >= mus) return;
    const float fmu = static_cast<float>(sh.mu[slot]), fwx = static_cast<float>(sh.wx[slot]);
    const float c = kCosPhi[m], s = kSinPhi[m];
    const float nu2 = fmaf(fwx * t.st, c, fmu * static_cast<float>(t.ct));
    const float pr = fmaf(nu2, nu2, 1.0f);
    const float q = rsq_f(fmaf(mg2, nu2, g1));
    const float pm = pr * (q * q * q);
    float v[6] = {pr, pr * c, pr * s, pm, pm * c, pm * s};
    float all[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) v[i] = scan16(v[i]);
#pragma unroll
    for (int i = 0; i < 6; ++i) all[i] = 2.0f * __shfl(v[i], lane | 15);
    // Azimuths m, 31 - m and -1 - m have the same cosine and phase, and
    // opposite sines. The last lane's mirrored slot 32 is its slot above; it
    // writes the empty sum and the whole circle's instead.
    float4* const e4 = prefix4 + (l & 1) * prefix_size + slot * kArcSlots;
    float2* const e2 = prefix2 + (l & 1) * prefix_size + slot * kArcSlots;
    e4[17 + m] = make_float4(v[0], v[1], v[2], v[3]);
    e2[17 + m] = make_float2(v[4], v[5]);
    e4[15 - m] = make_float4(-v[0], -v[1], v[2], -v[3]);
    e2[15 - m] = make_float2(-v[4], v[5]);
    const bool last = m == 15;
    const int at = 47 - m + (last ? 16 : 0);
    e4[at] = last ? make_float4(all[0], all[1], 0.0f, all[3])
                  : make_float4(all[0] - v[0], all[1] - v[1], v[2], all[3] - v[3]);
    e2[at] = last ? make_float2(all[4], 0.0f) : make_float2(all[4] - v[4], v[5]);
    if (last) {
      e4[16] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      e2[16] = make_float2(0.0f, 0.0f);
    }
  };
  // The terms (held) chunk and on of the columns at angle l, in buffer b: a
  // wave makes kUnit terms of a column for all wavelengths; two waves make
  // the terms' places on the circle.
  const float inv_nnu = 1.0f / static_cast<float>(nnu);
  auto build_terms = [&](int b, int l, int chunk) {
    const ArcTheta& t = sh.th[l];
    const int i = tid - (kArcWaves - 2) * 64;
    if (i >= 0 && i < cols * held) {
      const int s = i / held, e = chunk * held + i % held;
      const ArcColumn& c = columns[l * cols + s];
      if (e < counts[l * cols + s]) {
        const float pos = e == 0 ? c.klo - nnu
                          : e < 2 + c.nv ? c.klo + e - 1
                                         : ((e - 1 - c.nv) - c.ea) * c.inv_eb;
        const float rel = static_cast<float>(c.ta - pos);
        const float q =
            e < 2 ? 16.0f : acosf(fminf(fmaxf(-rel * c.inv_rt, -1.0f), 1.0f)) * kSteps;
        pars[b * cols * held + i] = make_float2(rel / c.s, q + 17.0f);
      }
    }
    for (int u = (wave + 4) % kArcWaves; u < cols * ((held + kUnit - 1) / kUnit);
         u += kArcWaves) {
      const int s = u % cols, o = (u / cols) * kUnit + kk;
      const int count = counts[l * cols + s];
      if (chunk * held + o - kk >= count) continue;
      const ArcColumn& c = columns[l * cols + s];
      const int e = chunk * held + o;
      if (kk >= kUnit || o >= held) continue;
      float D = 0.0f;
      if (e < 2 + c.nv) {
        // Slopes above and below the term's place: the lowest piece
        // f0 + slope (t - klo) is reached from 0 at t = klo - NU.
        const float* const v =
            nodes + ((((l & 1) * cols + s) * nnu + c.klo + max(e - 1, 0)) * 16 + n);
        const float v0 = v[0], v1 = v[16];
        const float rise = e < 2 ? v0 * inv_nnu : v[-16];
        const float below = e < 2 ? rise : v0 - rise;
        D = e == 0 ? rise : (v1 - v0) - below;
        if (e < 2 && t.ground) {
          // The line of the ground irradiance.
          const float e0 = irradiance(c.jlo), de = irradiance(c.jlo + 1) - e0;
          const float gf = sh.gf[l][n];
          const float a = gf * fmaf(de, c.e_at, e0) * inv_nnu;
          D += e == 0 ? a : fmaf(gf * de, c.eb, -a);
        }
      } else if (e < count) {
        const int j = c.jlo + (e - 1 - c.nv);
        const float e0 = irradiance(j - 1), e1 = irradiance(j), e2 = irradiance(j + 1);
        D = sh.gf[l][n] * c.eb * ((e2 - e1) - (e1 - e0));
      }
      terms[((b * cols + s) * held + o) * 16 + 4 * (n & 3) + (n >> 2)] = on ? D * c.s : 0.0f;
    }
  };

  // Two sums per texel and wavelength, or (several groups of wavelengths, to
  // stay in registers) one with both factors in the terms.
  constexpr bool kOne = kG >= 2;
  f32x4 acc_r[kTiles][kG], acc_m[kTiles][kOne ? 1 : kG];
#pragma unroll
  for (int i = 0; i < kG; ++i)
#pragma unroll
    for (int g = 0; g < kTiles; ++g) {
      acc_r[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!kOne) acc_m[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  auto product = [&](int b, int l, int chunk) {
    const int count =
        min(__builtin_amdgcn_readfirstlane(counts[l * cols + col]) - chunk * held, held);
    const float2* par = pars + (b * cols + col) * held;
    const float* term = terms + (b * cols + col) * held * 16 + 4 * (lane & 3);
    float cr[kG], cm[kG];
    if (kOne)
#pragma unroll
      for (int i = 0; i < kG; ++i) {
        cr[i] = sh.cr[4 * i + (lane & 3)];
        cm[i] = sh.cm[4 * i + (lane & 3)];
      }
    const char *pre4[kTiles], *pre2[kTiles];
#pragma unroll
    for (int g = 0; g < kTiles; ++g) {
      pre4[g] = reinterpret_cast<const char*>(prefix4 + (l & 1) * prefix_size + base[g]);
      pre2[g] = reinterpret_cast<const char*>(prefix2 + (l & 1) * prefix_size + base[g]);
    }
    for (int e = 0; e < count; ++e, ++par, term += 16) {
      const float2 p = *par;
      const float qa = 34.0f - p.y;
      float d[kG];
#pragma unroll
      for (int i = 0; i < kG; ++i) d[i] = term[i];
      float4 a4[kTiles], b4[kTiles];
      float2 a2[kTiles], b2[kTiles];
#pragma unroll
      for (int g = 0; g < kTiles; ++g) {
        const int ib = static_cast<int>(xs[g] + p.y), ia = static_cast<int>(xs[g] + qa);
        b4[g] = *reinterpret_cast<const float4*>(pre4[g] + ib * 16);
        b2[g] = *reinterpret_cast<const float2*>(pre2[g] + ib * 8);
        a4[g] = *reinterpret_cast<const float4*>(pre4[g] + ia * 16);
        a2[g] = *reinterpret_cast<const float2*>(pre2[g] + ia * 8);
      }
#pragma unroll
      for (int g = 0; g < kTiles; ++g) {
        const float gr = fmaf(sy[g], b4[g].z - a4[g].z,
                              fmaf(sx[g], b4[g].y - a4[g].y, p.x * (b4[g].x - a4[g].x)));
        const float gm = fmaf(sy[g], b2[g].y - a2[g].y,
                              fmaf(sx[g], b2[g].x - a2[g].x, p.x * (b4[g].w - a4[g].w)));
#pragma unroll
        for (int i = 0; i < kG; ++i) {
          if (kOne) {
            acc_r[g][i] =
                __builtin_amdgcn_mfma_f32_4x4x1f32(gr, cr[i] * d[i], acc_r[g][i], 0, 0, 0);
            acc_r[g][i] =
                __builtin_amdgcn_mfma_f32_4x4x1f32(gm, cm[i] * d[i], acc_r[g][i], 0, 0, 0);
          } else {
            acc_r[g][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(gr, d[i], acc_r[g][i], 0, 0, 0);
            acc_m[g][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(gm, d[i], acc_m[g][i], 0, 0, 0);
          }
        }
      }
    }
  };

  load_nodes(0);
  store_nodes(0);
  __syncthreads();
  load_nodes(1);
  build_prefix(0);
  build_terms(0, 0, 0);
  store_nodes(1);
  __syncthreads();
  int l = 0, chunk = 0;
  for (int b = 0; l < kTheta; b ^= 1) {
    // The next step: the next terms of this angle if any column has more,
    // else the next angle. They are built in the other buffer, and the nodes
    // of the angle after it loaded, between the same barriers as this step's
    // products.
    const bool more = __builtin_amdgcn_readfirstlane(sh.th[l].chunks) > chunk + 1;
    const int l1 = more ? l : l + 1, chunk1 = more ? chunk + 1 : 0;
    if (l1 < kTheta) {
      const bool ahead = !more && l + 2 < kTheta;
      if (ahead) load_nodes(l + 2);
      if (!more) build_prefix(l1);
      build_terms(b ^ 1, l1, chunk1);
      if (ahead) store_nodes(l + 2);
    }
    product(b, l, chunk);
    __syncthreads();
    l = l1;
    chunk = chunk1;
  }

  // A lane holds wavelength 4 i + lane % 4 of the texels 4 (lane / 4) .. + 3
  // of each tile: through LDS, so that a thread stores the three channels of
  // a texel and neighbouring threads neighbouring columns.
  float* const stage = reinterpret_cast<float*>(prefix4);
#pragma unroll
  for (int g = 0; g < kTiles; ++g) {
    if (g > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < kG; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        stage[(wave * 64 + (lane & ~3) + q) * 17 + 4 * i + (lane & 3)] =
            kOne ? acc_r[g][i][q]
                 : fmaf(sh.cm[4 * i + (lane & 3)], acc_m[g][kOne ? 0 : i][q],
                        sh.cr[4 * i + (lane & 3)] * acc_r[g][i][q]);
    __syncthreads();
    for (int e = tid; e < kArcWaves * 64 * nit; e += kArcWaves * 64) {
      const int s = e % cols, row = (e / cols) % 64, part = (e / (cols * 64)) % (kArcWaves / cols),
                t = e / (kArcWaves * 64);
      const int at = (part * kTiles + g) * 64 + row;
      const int slot = at / nnu, nui = at - slot * nnu;
      if (slot >= mus || y0 + slot >= nmu || c0 + s >= nmus) continue;
      const float* const v = stage + ((part * cols + s) * 64 + row) * 17 + 3 * t;
      const int64_t o = (layer + y0 + slot) * W + nui * nmus + c0 + s;
      void* const dj = (&J)[t].dJ;
      if (J.half_luts)
        gstore(static_cast<uint2*>(dj), o, pack_f21x3(v[0], v[1], v[2]));
      else
        gstore(static_cast<float3*>(dj), o, make_float3(v[0], v[1], v[2]));
    }
  }
}

template <int kTiles, int kG>
void launch_arcs(const PassLaunch& p, hipStream_t s) {
  if (p.arc_kinds & arc_kind_bit(kTiles, kG))
    hipLaunchKernelGGL((k_density_arcs<kTiles, kG>), dim3(p.total_blocks), dim3(kArcWaves * 64),
                       p.arc_lds, s, p.jobs, p.first_block, p.njobs);
}

}  // namespace

int blocks_density_arcs(const Job& j) {
  if (j.it % kArcIters != 0) return 0;  // served with the first of its group
  const int mus = arc_mus(j.nnu), cols = arc_cols(j.nnu);
  return j.nr * ((j.nmu + mus - 1) / mus) * ((j.nmus + cols - 1) / cols);
}

size_t arc_lds(const Job& j) { return static_cast<size_t>(ArcLayout(j.nnu).bytes); }

hipError_t launch_density_arcs(const PassLaunch& p, hipStream_t s) {
  // One instance per kind of job; each skips the others.
  launch_arcs<1, 1>(p, s);
  launch_arcs<1, 2>(p, s);
  launch_arcs<1, 3>(p, s);
  launch_arcs<1, 4>(p, s);
  launch_arcs<2, 1>(p, s);
  launch_arcs<2, 2>(p, s);
  launch_arcs<2, 3>(p, s);
  launch_arcs<2, 4>(p, s);
  return hipGetLastError();
}

}  // namespace atmo

#endif  // ATMO_DENSITY_ARCS_H_
