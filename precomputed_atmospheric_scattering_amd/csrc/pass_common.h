// Device helpers shared by the precompute kernels (precompute.hip,
// density_arcs.h).
#ifndef ATMO_PASS_COMMON_H_
#define ATMO_PASS_COMMON_H_

#include <hip/hip_runtime.h>

namespace atmo {
namespace {

// Workgroups are dispatched to the 8 XCDs (each with its own L2) round-robin
// by workgroup id. This permutation of a job's nb blocks gives the blocks of
// one XCD (same id mod 8) a contiguous range of the job's work, so that the
// blocks resident on an XCD at a time work on neighbouring rows and share
// their L2 lines.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_contiguous(int lb, int nb) {
  const int q = nb / kXcds, rem = nb % kXcds;
  const int g = lb % kXcds;
  return g * q + (g < rem ? g : rem) + lb / kXcds;
}

// Block b's job: the last i with first_block[i] <= b (a job without blocks
// in a launch repeats its successor's entry). The search is uniform across
// the block.
__device__ __forceinline__ int find_job(const int* __restrict__ first_block,
                                        int njobs, int b) {
  int lo = 0, hi = njobs;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (first_block[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ float rcp_f(float x) {
  return __builtin_amdgcn_rcpf(x);
}
__device__ __forceinline__ float rsq_f(float x) {
  return __builtin_amdgcn_rsqf(x);
}
__device__ __forceinline__ float sqrt_f(float x) {
  return __builtin_amdgcn_sqrtf(x);
}
__device__ __forceinline__ float clampf(float x, float lo, float hi) {
  return fminf(fmaxf(x, lo), hi);
}

// cos and sin of (m + 1/2) * pi / 16 for m = 0..15, evaluated at compile time
// (Taylor series in FP64, converged to the last bit for |x| <= pi).
constexpr double cx_sin(double x) {
  double term = x, sum = x;
  for (int n = 1; n < 24; ++n) {
    term *= -x * x / ((2.0 * n) * (2.0 * n + 1.0));
    sum += term;
  }
  return sum;
}
constexpr double cx_cos(double x) {
  double term = 1.0, sum = 1.0;
  for (int n = 1; n < 24; ++n) {
    term *= -x * x / ((2.0 * n - 1.0) * (2.0 * n));
    sum += term;
  }
  return sum;
}
#define ATMO_PHI(m) ((m + 0.5) * 3.14159265358979323846 / 16.0)
__device__ constexpr float kCosPhi[16] = {
    float(cx_cos(ATMO_PHI(0))),  float(cx_cos(ATMO_PHI(1))),
    float(cx_cos(ATMO_PHI(2))),  float(cx_cos(ATMO_PHI(3))),
    float(cx_cos(ATMO_PHI(4))),  float(cx_cos(ATMO_PHI(5))),
    float(cx_cos(ATMO_PHI(6))),  float(cx_cos(ATMO_PHI(7))),
    float(cx_cos(ATMO_PHI(8))),  float(cx_cos(ATMO_PHI(9))),
    float(cx_cos(ATMO_PHI(10))), float(cx_cos(ATMO_PHI(11))),
    float(cx_cos(ATMO_PHI(12))), float(cx_cos(ATMO_PHI(13))),
    float(cx_cos(ATMO_PHI(14))), float(cx_cos(ATMO_PHI(15)))};
__device__ constexpr float kSinPhi[16] = {
    float(cx_sin(ATMO_PHI(0))),  float(cx_sin(ATMO_PHI(1))),
    float(cx_sin(ATMO_PHI(2))),  float(cx_sin(ATMO_PHI(3))),
    float(cx_sin(ATMO_PHI(4))),  float(cx_sin(ATMO_PHI(5))),
    float(cx_sin(ATMO_PHI(6))),  float(cx_sin(ATMO_PHI(7))),
    float(cx_sin(ATMO_PHI(8))),  float(cx_sin(ATMO_PHI(9))),
    float(cx_sin(ATMO_PHI(10))), float(cx_sin(ATMO_PHI(11))),
    float(cx_sin(ATMO_PHI(12))), float(cx_sin(ATMO_PHI(13))),
    float(cx_sin(ATMO_PHI(14))), float(cx_sin(ATMO_PHI(15)))};
#undef ATMO_PHI

// Incident zenith angles of the scattering density and the indirect
// irradiance.
constexpr int kTheta = 16;

}  // namespace
}  // namespace atmo

#endif  // ATMO_PASS_COMMON_H_
