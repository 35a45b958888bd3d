// Sky-shading lookups for gfx950: GetSkyRadiance, GetSkyRadianceToPoint and
// GetSunAndSkyIrradiance (atmosphere/functions.glsl:1633-1896) over batches
// of rays, one ray per thread. Texels are FP32; everything else is FP64: the
// scalar geometry (radius, ray/sphere discriminants, ground flag, LUT
// coordinates), where FP32 cancellation near the horizon flips the ground/sky
// choice or shifts a lookup, and the texel blending, so that the difference
// of two nearby lookups in GetSkyRadianceToPoint keeps the texels' precision.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "atmo_device.h"
#include "kernels.h"

namespace atmo {
namespace {

struct D3 {
  double x, y, z;
};
__device__ __forceinline__ D3 load3(const float* p, int64_t i) {
  return D3{p[3 * i], p[3 * i + 1], p[3 * i + 2]};
}
__device__ __forceinline__ void store3(float* p, int64_t i, D4 v) {
  p[3 * i] = static_cast<float>(v.x);
  p[3 * i + 1] = static_cast<float>(v.y);
  p[3 * i + 2] = static_cast<float>(v.z);
}
__device__ __forceinline__ double dot3(D3 a, D3 b) {
  return a.x * b.x + a.y * b.y + a.z * b.z;
}
__device__ __forceinline__ D4 mul(D4 a, D4 b) {
  return D4{a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w};
}
__device__ __forceinline__ D4 scale(D4 a, double s) {
  return D4{a.x * s, a.y * s, a.z * s, a.w * s};
}
__device__ __forceinline__ D4 sub(D4 a, D4 b) {
  return D4{a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w};
}
__device__ __forceinline__ D4 rgb(D4 a) { return D4{a.x, a.y, a.z, 0.0}; }

// functions.glsl:1633-1645
__device__ __forceinline__ D4 extrapolated_mie(const Job& J, D4 s) {
  if (s.x <= 0.0) return D4{0.0, 0.0, 0.0, 0.0};
  const double k = s.w / s.x * (J.rayleigh[0] / J.mie_sca[0]);
  return D4{s.x * k * (J.mie_sca[0] / J.rayleigh[0]),
            s.y * k * (J.mie_sca[1] / J.rayleigh[1]),
            s.z * k * (J.mie_sca[2] / J.rayleigh[2]), 0.0};
}

__device__ __forceinline__ void acc_q(D4* acc, double w, float4 v) { acc_d4(acc, w, v); }
__device__ __forceinline__ void acc_q(float4* acc, float w, float4 v) { acc_f4(acc, w, v); }
__device__ __forceinline__ D4 as_d4(D4 v) { return v; }
__device__ __forceinline__ D4 as_d4(float4 v) { return to_d4(v); }

// 16-byte parts of lookup copy lines that a wave holds in LDS: one line of
// each lane.
constexpr int kLineParts = 8;
constexpr int kStageParts = 64 * kLineParts;
// Lanes whose first line is their neighbour's from which on lanes load their
// own lines (neighbouring pixels of a frame).
constexpr int kNearLanes = 32;

__device__ __forceinline__ float4 as_floats(uint4 a) {
  return make_float4(__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z),
                     __uint_as_float(a.w));
}

// The lookup of S and SM in the lookup copy for the rays of a wave, whose
// lanes are all active. A ray reads 2 (FP16) or 4 lines of 128 bytes at random.
// Read by its own lane, a line takes 8 loads, each of them 64 lines for the
// wave: a scattered 16-byte load cost 50 cycles of the address unit, which
// was busy 70% of the time with the vector units at 49% and 2 waves per SIMD
// (226 VGPRs hold the loads in flight). Here 8 lanes read a line together, so
// that a load takes 8 whole lines, and each lane gets its own from LDS. Part k
// of a line is at k ^ (lane % 8), so that neighbouring lanes read different
// banks. Where most lanes' lines are their neighbours' (the pixels of a frame),
// the lanes load their own.
// 2.07M rays on MI355X, own lines | shared, us: GetSkyRadiance scattered 134 |
// 97 FP32, 85 | 78 FP16; GetSkyRadianceToPoint scattered 307 | 198 and 212 |
// 176, pixels 177 | 152 and 150 | 152.
template <class Real, bool kHalf>
__device__ __forceinline__ void lookup_lines(const Job& J, const SCoords& c, uint4* stage,
                                             D4* s, D4* m) {
  using Acc = typename std::conditional<sizeof(Real) == 8, D4, float4>::type;
  const QuadTaps<Real> t(J, c);
  const uint4* __restrict__ lines = static_cast<const uint4*>(J.Q);
  const int lane = threadIdx.x & 63, group = lane / kLineParts, part = lane % kLineParts;
  constexpr int kLines = kHalf ? 2 : 4;
  Acc as{}, am{};
  // Part k of line n of the lane.
  auto add = [&](int n, int k, uint4 u) {
    const int a = kHalf ? n : n / 2, b = kHalf ? k / 4 : n % 2, texel = kHalf ? k % 4 : k / 2;
    const Real w = t.wz[a] * t.wy[b] * t.wx[texel / 2] * t.ws[texel % 2];
    if (kHalf) {
      acc_q(&as, w, unpack_half4(make_uint2(u.x, u.y)));
      acc_q(&am, w, unpack_half4(make_uint2(u.z, u.w)));
    } else {
      acc_q(k % 2 ? &am : &as, w, as_floats(u));
    }
  };
  if (__popcll(__ballot(t.line[0] == __shfl_xor(t.line[0], 1))) >= kNearLanes) {
#pragma unroll
    for (int n = 0; n < kLines; ++n)
#pragma unroll
      for (int k = 0; k < kLineParts; ++k)
        add(n, k, gload(lines, static_cast<int64_t>(t.line[n]) * kLineParts + k));
  } else {
    uint4 v[kLineParts];
    auto fetch = [&](int n) {
#pragma unroll
      for (int k = 0; k < kLineParts; ++k) {
        const uint32_t line = __shfl(t.line[n], kLineParts * k + group);
        v[k] = gload(lines, static_cast<int64_t>(line) * kLineParts + part);
      }
    };
    fetch(0);
#pragma unroll
    for (int n = 0; n < kLines; ++n) {
#pragma unroll
      for (int k = 0; k < kLineParts; ++k)
        stage[(kLineParts * k + group) * kLineParts + (part ^ group)] = v[k];
      // (The lanes of a wave run in step and its LDS accesses in order.)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (n + 1 < kLines) fetch(n + 1);
#pragma unroll
      for (int k = 0; k < kLineParts; ++k)
        add(n, k, stage[lane * kLineParts + (k ^ part)]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (kHalf) {
    // Stored values, scaled after the sums as for F16Texels.
    const float* sc = J.scales;
    as = scaled(as, make_float4(1.0f / sc[0], 1.0f / sc[1], 1.0f / sc[2], 1.0f / sc[3]));
    am = scaled(am, make_float4(1.0f / sc[4], 1.0f / sc[5], 1.0f / sc[6], 0.0f));
  }
  *s = as_d4(as);
  *m = as_d4(am);
}

// functions.glsl:1658-1690. kF32: FP32 tap weights and sums (GetSkyRadiance, whose
// result is not a difference of two lookups); otherwise FP64. kSeparate: S and
// SM are separate. kLines: they may have a lookup copy; then all lanes of the wave
// call it, with the wave's kStageParts parts of LDS.
template <bool kF32, bool kSeparate, bool kLines>
__device__ D4 combined_scattering(const Job& J, double r, double mu, double mu_s,
                                  double nu, bool ground, uint4* stage, D4* single_mie) {
  using Real = typename std::conditional<kF32, float, double>::type;
  const SCoords c = s_coords<kF32>(J, r, mu, mu_s, nu, ground);
  auto lookup = [&](const auto& lut) {
    return kF32 ? s_lookup_f(J, lut, c) : s_lookup_d(J, lut, c);
  };
  D4 s;
  if (kLines && J.Q != nullptr) {
    // Lookup copy: the S and SM texels of the 4 (nu, mu_s) taps of each
    // (r, mu) tap in one contiguous quad.
    if (J.half_luts)
      lookup_lines<Real, true>(J, c, stage, &s, single_mie);
    else
      lookup_lines<Real, false>(J, c, stage, &s, single_mie);
    *single_mie = rgb(*single_mie);
    return s;
  }
  if (J.half_luts) {
    const float* sc = J.scales;
    const F16Texels st{J.S16, make_float4(1.0f / sc[0], 1.0f / sc[1], 1.0f / sc[2],
                                          1.0f / sc[3])};
    s = lookup(st);
    if (kSeparate) {
      const F16Texels mt{J.SM16, make_float4(1.0f / sc[4], 1.0f / sc[5], 1.0f / sc[6],
                                             0.0f)};
      *single_mie = rgb(lookup(mt));
    }
  } else {
    s = lookup(F32Texels{J.S});
    if (kSeparate) *single_mie = rgb(lookup(F32Texels{J.SM}));
  }
  if (!kSeparate) *single_mie = extrapolated_mie(J, s);
  return s;
}

// scattering * P_R(nu) + single_mie * P_M(nu), optionally times the sky
// radiance-to-luminance factors.
__device__ __forceinline__ D4 shade(const Job& J, D4 scat, D4 mie, double nu,
                                    int luminance) {
  const double pr = rayleigh_phase_d(nu);
  const double pm = mie_phase_d(J.g, nu);
  D4 l{scat.x * pr + mie.x * pm, scat.y * pr + mie.y * pm, scat.z * pr + mie.z * pm,
       0.0};
  if (luminance) l = D4{l.x * J.sky_k[0], l.y * J.sky_k[1], l.z * J.sky_k[2], 0.0};
  return l;
}

// kSeparate, kLines: as in combined_scattering. Three waves per SIMD take 168
// VGPRs with lines (175 unbounded, 8% slower); without, the loads in flight of
// fewer waves are worth more (2.07M scattered rays with 2 waves, and 3: combined FP16 121
// us, 131; separate without a copy 193, 241 FP16, 286, 313 FP32).
template <bool kSeparate, bool kLines>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kLines ? 3 : 2))) void
k_sky_radiance(
    const Job* __restrict__ job, int64_t n, const float* __restrict__ camera,
    const float* __restrict__ view_ray, const float* __restrict__ shadow_length,
    const float* __restrict__ sun_direction, float* __restrict__ radiance,
    float* __restrict__ transmittance_out, int luminance) {
  __shared__ uint4 stage_of[kLines ? kBlock / 64 : 1][kLines ? kStageParts : 1];
  uint4* const stage = stage_of[kLines ? threadIdx.x / 64 : 0];
  // All lanes of a wave take part in the lookups of lines: those past the end
  // repeat the last ray and store nothing.
  const int64_t ray = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (!kLines && ray >= n) return;
  const int64_t i = ray < n ? ray : n - 1;
  const Job& J = *job;
  D3 cam = load3(camera, i);
  const D3 v = load3(view_ray, i);
  const D3 sd = load3(sun_direction, i);
  const double shadow = shadow_length[i];
  // functions.glsl:1715-1729
  double r = sqrt(dot3(cam, cam));
  double rmu = dot3(cam, v);
  const double to_top = -rmu - sqrt(rmu * rmu - r * r + J.rt * J.rt);
  bool space = false;
  if (to_top > 0.0) {
    cam = D3{cam.x + v.x * to_top, cam.y + v.y * to_top, cam.z + v.z * to_top};
    r = J.rt;
    rmu += to_top;
  } else if (r > J.rt) {
    // In space, looking past the atmosphere.
    if (!kLines) {
      store3(transmittance_out, i, D4{1.0, 1.0, 1.0, 0.0});
      store3(radiance, i, D4{0.0, 0.0, 0.0, 0.0});
      return;
    }
    space = true;
    r = J.rt;
    rmu = r;
  }
  // With lines, a wave leaves together (most waves of a frame seen from space do:
  // 2.07M pixels 40 us, 60 where each stays for the lookups).
  if (kLines && __all(space)) {
    if (ray >= n) return;
    store3(transmittance_out, i, D4{1.0, 1.0, 1.0, 0.0});
    store3(radiance, i, D4{0.0, 0.0, 0.0, 0.0});
    return;
  }
  const double mu = rmu / r;
  const double mu_s = dot3(cam, sd) / r;
  const double nu = dot3(v, sd);
  const bool ground = hits_ground(J, r, mu);
  const D4 zero{0.0, 0.0, 0.0, 0.0};
  const D4 t = ground ? zero : t_lookup_d(J, J.T, r, mu);
  D4 mie, scat;
  if (kSeparate && !kLines && shadow == 0.0) {
    // (Without a copy, a lookup of its own for these rays: 300k scattered rays with
    // light shafts 65 us with one for both, high-resolution LUTs, 56 with two.)
    scat = combined_scattering<true, kSeparate, kLines>(J, r, mu, mu_s, nu, ground, stage, &mie);
  } else {
    double r_p = r, mu_p = mu, mu_s_p = mu_s;
    if (shadow != 0.0) {
      // Light shafts (functions.glsl:1746-1766).
      const double d = shadow;
      r_p = clamp_radius(J, sqrt(d * d + 2.0 * r * mu * d + r * r));
      mu_p = (r * mu + d) / r_p;
      mu_s_p = (r * mu_s + d * nu) / r_p;
    }
    scat = combined_scattering<true, kSeparate, kLines>(J, r_p, mu_p, mu_s_p, nu, ground, stage,
                                                        &mie);
  }
  scat = rgb(scat);
  if (ray >= n) return;
  if (shadow != 0.0) {
    const D4 st = transmittance_d(J, J.T, r, mu, shadow, ground);
    scat = mul(scat, st);
    mie = mul(mie, st);
  }
  store3(radiance, i, space ? zero : shade(J, scat, mie, nu, luminance));
  store3(transmittance_out, i, space ? D4{1.0, 1.0, 1.0, 0.0} : t);
}

// (Two waves per SIMD: with lines its FP64 sums take 227 VGPRs, and 3 spill;
// without, 3 waves make scattered lookups 4% slower.)
template <bool kLines>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_sky_radiance_to_point(
    const Job* __restrict__ job, int64_t n, const float* __restrict__ camera,
    const float* __restrict__ point, const float* __restrict__ shadow_length,
    const float* __restrict__ sun_direction, float* __restrict__ radiance,
    float* __restrict__ transmittance_out, int luminance) {
  __shared__ uint4 stage_of[kLines ? kBlock / 64 : 1][kLines ? kStageParts : 1];
  uint4* const stage = stage_of[kLines ? threadIdx.x / 64 : 0];
  const int64_t ray = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (!kLines && ray >= n) return;
  const int64_t i = ray < n ? ray : n - 1;  // as in k_sky_radiance
  const Job& J = *job;
  D3 cam = load3(camera, i);
  const D3 p = load3(point, i);
  const D3 sd = load3(sun_direction, i);
  const double shadow = shadow_length[i];
  // functions.glsl:1797-1808
  D3 v = D3{p.x - cam.x, p.y - cam.y, p.z - cam.z};
  const double inv_len = 1.0 / sqrt(dot3(v, v));
  v = D3{v.x * inv_len, v.y * inv_len, v.z * inv_len};
  double r = sqrt(dot3(cam, cam));
  double rmu = dot3(cam, v);
  const double to_top = -rmu - sqrt(rmu * rmu - r * r + J.rt * J.rt);
  if (to_top > 0.0) {
    cam = D3{cam.x + v.x * to_top, cam.y + v.y * to_top, cam.z + v.z * to_top};
    r = J.rt;
    rmu += to_top;
  }
  const double mu = rmu / r;
  const double mu_s = dot3(cam, sd) / r;
  const double nu = dot3(v, sd);
  const D3 pc = D3{p.x - cam.x, p.y - cam.y, p.z - cam.z};
  double d = sqrt(dot3(pc, pc));
  const bool ground = hits_ground(J, r, mu);
  // Both transmittances below are quotients with the lookup at the camera.
  const D4 here = t_lookup_d(J, J.T, r, ground ? -mu : mu);
  const D4 t = transmittance_from_d(J, J.T, here, r, mu, d, ground);
  D4 mie;
  D4 scat =
      rgb(combined_scattering<false, kLines, kLines>(J, r, mu, mu_s, nu, ground, stage, &mie));
  // functions.glsl:1831-1840
  d = d - shadow > 0.0 ? d - shadow : 0.0;
  const double r_p = clamp_radius(J, sqrt(d * d + 2.0 * r * mu * d + r * r));
  const double mu_p = (r * mu + d) / r_p;
  const double mu_s_p = (r * mu_s + d * nu) / r_p;
  D4 mie_p;
  const D4 scat_p =
      rgb(combined_scattering<false, kLines, kLines>(J, r_p, mu_p, mu_s_p, nu, ground, stage,
                                                     &mie_p));
  if (ray >= n) return;
  D4 st = t;
  if (shadow > 0.0) st = transmittance_from_d(J, J.T, here, r, mu, d, ground);
  scat = sub(scat, mul(st, scat_p));
  mie = sub(mie, mul(st, mie_p));
  if (!kLines) mie = extrapolated_mie(J, D4{scat.x, scat.y, scat.z, mie.x});
  // functions.glsl:1857-1859
  mie = scale(mie, smoothstep_d(0.0, 0.01, mu_s));
  store3(radiance, i, shade(J, scat, mie, nu, luminance));
  store3(transmittance_out, i, t);
}

__global__ __launch_bounds__(kBlock) void k_sun_and_sky_irradiance(
    const Job* __restrict__ job, int64_t n, const float* __restrict__ point,
    const float* __restrict__ normal, const float* __restrict__ sun_direction,
    float* __restrict__ sun_out, float* __restrict__ sky_out, int luminance) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const Job& J = *job;
  const D3 p = load3(point, i);
  const D3 nrm = load3(normal, i);
  const D3 sd = load3(sun_direction, i);
  const double r = sqrt(dot3(p, p));
  const double mu_s = dot3(p, sd) / r;
  // Two lookups, neither a difference: FP32 weights and sums (as in
  // GetSkyRadiance).
  D4 sky = scale(e_lookup_d<float>(J, J.E, r, mu_s), (1.0 + dot3(nrm, p) / r) * 0.5);
  const D4 ts = transmittance_to_sun_d<float>(J, J.T, r, mu_s);
  const double c = dot3(nrm, sd);
  const double cf = c > 0.0 ? c : 0.0;
  D4 sun{J.solar[0] * ts.x * cf, J.solar[1] * ts.y * cf, J.solar[2] * ts.z * cf, 0.0};
  if (luminance) {
    // GetSunAndSkyIlluminance (atmosphere/model.cc:273-281).
    sky = D4{sky.x * J.sky_k[0], sky.y * J.sky_k[1], sky.z * J.sky_k[2], 0.0};
    sun = D4{sun.x * J.sun_k[0], sun.y * J.sun_k[1], sun.z * J.sun_k[2], 0.0};
  }
  store3(sky_out, i, sky);
  store3(sun_out, i, sun);
}

// Seeded synthetic query batches. Variate k of ray i is output number
// 6 i + k + 1 of the SplitMix64 sequence started at 'seed' (Steele, Lea and
// Flood, "Fast splittable pseudorandom number generators", OOPSLA 2014): the
// sequence's n-th output is the finalizer applied to seed + n * golden gamma.
__device__ __forceinline__ double splitmix_uniform(uint64_t seed, uint64_t n) {
  uint64_t z = seed + n * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return static_cast<double>(z >> 11) * 0x1.0p-53;
}

__global__ __launch_bounds__(kBlock) void k_generate_queries(
    uint64_t seed, int64_t n, double rb, double rt, double max_altitude,
    double max_distance, double max_sun_zenith, float* __restrict__ camera,
    float* __restrict__ view_ray, float* __restrict__ sun_direction,
    float* __restrict__ point, float* __restrict__ normal,
    float* __restrict__ shadow_length) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint64_t base = 6ull * static_cast<uint64_t>(i) + 1ull;
  const double alt = max_altitude * splitmix_uniform(seed, base);
  const double vz = 2.0 * splitmix_uniform(seed, base + 1) - 1.0;
  const double vphi = 2.0 * kPi * splitmix_uniform(seed, base + 2);
  const double zen = max_sun_zenith * splitmix_uniform(seed, base + 3);
  const double az = 2.0 * kPi * splitmix_uniform(seed, base + 4);
  const double dist = max_distance * splitmix_uniform(seed, base + 5);
  const double vs = sqrt(fmax(0.0, 1.0 - vz * vz));
  const double v[3] = {vs * cos(vphi), vs * sin(vphi), vz};
  const double cz = rb + alt;
  double p[3] = {v[0] * dist, v[1] * dist, cz + v[2] * dist};
  const double pr = sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
  // Points are kept 1e-3 length units inside the atmosphere's shell.
  const double lo = rb + 1e-3, hi = rt - 1e-3;
  const double k = (pr < lo ? lo : (pr > hi ? hi : pr)) / pr;
  p[0] *= k;
  p[1] *= k;
  p[2] *= k;
  const double pn = sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
  const double sun[3] = {sin(zen) * cos(az), sin(zen) * sin(az), cos(zen)};
  for (int c = 0; c < 3; ++c) {
    camera[3 * i + c] = c == 2 ? static_cast<float>(cz) : 0.0f;
    view_ray[3 * i + c] = static_cast<float>(v[c]);
    sun_direction[3 * i + c] = static_cast<float>(sun[c]);
    point[3 * i + c] = static_cast<float>(p[c]);
    normal[3 * i + c] = static_cast<float>(p[c] / pn);
  }
  shadow_length[i] = 0.0f;
}

inline unsigned grid_for(int64_t n) {
  return static_cast<unsigned>((n + kBlock - 1) / kBlock);
}

}  // namespace

hipError_t launch_sky_radiance(const Job* job, bool combined, bool copy, int64_t n,
                               const float* camera, const float* view_ray,
                               const float* shadow_length,
                               const float* sun_direction, float* radiance,
                               float* transmittance, int luminance, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const auto kernel = combined ? k_sky_radiance<false, false>
                      : copy ? k_sky_radiance<true, true> : k_sky_radiance<true, false>;
  hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kBlock), 0, s, job, n, camera, view_ray,
                     shadow_length, sun_direction, radiance, transmittance, luminance);
  return hipGetLastError();
}

hipError_t launch_sky_radiance_to_point(const Job* job, bool combined, int64_t n,
                                        const float* camera,
                                        const float* point,
                                        const float* shadow_length,
                                        const float* sun_direction,
                                        float* radiance, float* transmittance,
                                        int luminance, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const auto kernel = combined ? k_sky_radiance_to_point<false> : k_sky_radiance_to_point<true>;
  hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kBlock), 0, s, job, n, camera, point,
                     shadow_length, sun_direction, radiance, transmittance, luminance);
  return hipGetLastError();
}

hipError_t launch_sun_and_sky_irradiance(const Job* job, int64_t n,
                                         const float* point,
                                         const float* normal,
                                         const float* sun_direction,
                                         float* sun_irradiance,
                                         float* sky_irradiance, int luminance,
                                         hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sun_and_sky_irradiance, dim3(grid_for(n)), dim3(kBlock), 0, s,
                     job, n, point, normal, sun_direction, sun_irradiance,
                     sky_irradiance, luminance);
  return hipGetLastError();
}

hipError_t launch_generate_queries(uint64_t seed, int64_t n, double bottom_radius,
                                  double top_radius, double max_altitude,
                                  double max_distance, double max_sun_zenith,
                                  float* camera, float* view_ray, float* sun_direction,
                                  float* point, float* normal, float* shadow_length,
                                  hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_generate_queries, dim3(grid_for(n)), dim3(kBlock), 0, s, seed, n,
                     bottom_radius, top_radius, max_altitude, max_distance,
                     max_sun_zenith, camera, view_ray, sun_direction, point, normal,
                     shadow_length);
  return hipGetLastError();
}

}  // namespace atmo
