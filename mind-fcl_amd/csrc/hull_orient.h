// The hull builder's orientation test in 32 bits: which side of a face's
// plane a point lies on, where 32 bits are sure of it.  Plain C++ but for the
// qualifiers, so that a test can compare it with 64 bits on the CPU.
#pragma once

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define MFCL_HD __host__ __device__ __forceinline__
#else
#include <math.h>
#define MFCL_HD inline
#endif

namespace mfcl {

// Of u, v, w, n and the products each operation rounds by at most 2^-24 of
// its size, eight times along any path to the volume, and every term is at
// most |u||v||w| in 1-norms: the error is below 2^-20 of that product (half
// of it is left over, which is also far above the 64-bit test's 1e-12), plus
// what underflows.  A value that overflows on the way turns the volume, which
// is of cubic size, into an infinity or NaN (no later operation makes either
// finite again) while the bound can still be finite, from coordinates of
// about 5e12 on: a volume that is not finite is not sure.
constexpr float kFloatMax = 3.40282347e+38f;
struct HullPlane {
  float ax, ay, az, nx, ny, nz, err;
};
MFCL_HD HullPlane planeOf(const float* A, const float* B, const float* C) {
  HullPlane q;
  q.ax = A[0];
  q.ay = A[1];
  q.az = A[2];
  const float ux = B[0] - q.ax, uy = B[1] - q.ay, uz = B[2] - q.az;
  const float vx = C[0] - q.ax, vy = C[1] - q.ay, vz = C[2] - q.az;
  q.nx = uy * vz - uz * vy;
  q.ny = uz * vx - ux * vz;
  q.nz = ux * vy - uy * vx;
  q.err = ((fabsf(ux) + fabsf(uy) + fabsf(uz)) * (fabsf(vx) + fabsf(vy) + fabsf(vz)) + 1e-30f) * 0x1p-20f;
  return q;
}
// 1 sees, 0 does not, -1 not sure
MFCL_HD int sees32(const HullPlane& q, const float* P) {
  const float wx = P[0] - q.ax, wy = P[1] - q.ay, wz = P[2] - q.az;
  const float o = q.nx * wx + q.ny * wy + q.nz * wz;
  const float e = q.err * (fabsf(wx) + fabsf(wy) + fabsf(wz)) + 1e-36f;
  if (!(fabsf(o) > e && fabsf(o) <= kFloatMax)) return -1;
  return o > 0 ? 1 : 0;
}

}  // namespace mfcl
