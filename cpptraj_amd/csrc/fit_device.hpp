// fit_device.hpp -- device code shared by the fit kernels (k_fit.hip,
// k_fit_fused.hip): moments of one atom, the solve of one frame and the
// coordinate update of one atom.
#pragma once
// Multiply-adds contracted by expression, not by what the compiler happens to
// see around them: the same source gives the same bits in every kernel of the
// files that include this, so a frame's fit does not depend on which of them
// took it.
#pragma clang fp contract(on)
#include "rmsd_device.hpp"
#include "rmsd_kernels.hpp"

namespace fit_dev {

// Adds one atom (x shifted, reference y) to the 13 moments of its frame:
// w x (3), w x y^T (9), w |x|^2.
template <bool WEIGHTED>
__device__ __forceinline__ void accum(double (&v)[13], double x0, double x1, double x2, double w,
                                      double y0, double y1, double y2) {
  double wx0 = x0, wx1 = x1, wx2 = x2;
  if (WEIGHTED) {
    wx0 = w * x0;
    wx1 = w * x1;
    wx2 = w * x2;
  }
  v[0] += wx0;
  v[1] += wx1;
  v[2] += wx2;
  v[3] += wx0 * y0; v[4] += wx0 * y1; v[5] += wx0 * y2;
  v[6] += wx1 * y0; v[7] += wx1 * y1; v[8] += wx1 * y2;
  v[9] += wx2 * y0; v[10] += wx2 * y1; v[11] += wx2 * y2;
  v[12] += wx0 * x0 + wx1 * x1 + wx2 * x2;
}

// RMSD, U (Kabsch) and t1 = -centroid of one frame from its 13 moments m (about
// the shift s) and the reference constants K; W < 1e-14: -1, identity, 0.
__device__ __forceinline__ double solve(const double* m, const double* K, double s0, double s1,
                                        double s2, int clamp, double (&U)[9], double (&t1)[3]) {
  const double W = K[4];
#pragma unroll
  for (int k = 0; k < 9; ++k) U[k] = k % 4 == 0 ? 1.0 : 0.0;
  t1[0] = t1[1] = t1[2] = 0.0;
  if (W < RMSD_SMALL) return -1.0;
  // centroid in shifted coordinates, then the centred moments
  const double c0 = m[0] / W, c1 = m[1] / W, c2 = m[2] / W;
  double R[9];
  R[0] = m[3] - c0 * K[0]; R[1] = m[4] - c0 * K[1]; R[2] = m[5] - c0 * K[2];
  R[3] = m[6] - c1 * K[0]; R[4] = m[7] - c1 * K[1]; R[5] = m[8] - c1 * K[2];
  R[6] = m[9] - c2 * K[0]; R[7] = m[10] - c2 * K[1]; R[8] = m[11] - c2 * K[2];
  const double sx = m[12] - W * (c0 * c0 + c1 * c1 + c2 * c2);
  const double E0 = 0.5 * (sx + K[3]);
  const rmsd_dev::QcpCoef co = rmsd_dev::qcp_coefficients(R);
  const double lam = rmsd_dev::qcp_lambda(co, E0);
  const double r = rmsd_dev::rmsd_from_lambda(E0, lam, W, clamp);
  rmsd_dev::qcp_rotation(R, lam, U);
  t1[0] = -(c0 + s0);
  t1[1] = -(c1 + s1);
  t1[2] = -(c2 + s2);
  return r;
}

// X = U (9), t1 (3), t2 (3).  mode 1: x' = U (x + t1) + t2
// (Frame::Trans_Rot_Trans, in its operation order); mode 2: x' = x + (t1 + t2).
__device__ __forceinline__ void move_atom(const double* X, int mode, float& px, float& py,
                                          float& pz) {
#pragma clang fp contract(off)
  if (mode == 1) {
    const double x = (double)px + X[9];
    const double y = (double)py + X[10];
    const double z = (double)pz + X[11];
    px = (float)(x * X[0] + y * X[1] + z * X[2] + X[12]);
    py = (float)(x * X[3] + y * X[4] + z * X[5] + X[13]);
    pz = (float)(x * X[6] + y * X[7] + z * X[8] + X[14]);
  } else {
    px = (float)((double)px + (X[9] + X[12]));
    py = (float)((double)py + (X[10] + X[13]));
    pz = (float)((double)pz + (X[11] + X[14]));
  }
}

// Four consecutive atoms as three 16-byte pieces with 4-byte alignment: global
// memory instructions take any dword address, so neither the frames' base nor
// their stride or row length needs to be a multiple of 16 bytes.
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// Atoms 4q ... 4q + 3 of a frame: SoA (ld > 0) or AoS.
__device__ __forceinline__ void load_step(const float* fr, int64_t ld, int q, float (&x)[4],
                                          float (&y)[4], float (&z)[4]) {
  const auto p = gp(fr);
  typedef const __attribute__((address_space(1))) f32x4_a4* vp;
  if (ld) {
    const f32x4_a4 a = *(vp)(p + 4 * q), b = *(vp)(p + ld + 4 * q), c = *(vp)(p + 2 * ld + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = a[e];
      y[e] = b[e];
      z[e] = c[e];
    }
  } else {
    const vp v = (vp)(p + 12 * (int64_t)q);
    const f32x4_a4 a = v[0], b = v[1], c = v[2];
    x[0] = a.x; y[0] = a.y; z[0] = a.z;
    x[1] = a.w; y[1] = b.x; z[1] = b.y;
    x[2] = b.z; y[2] = b.w; z[2] = c.x;
    x[3] = c.y; y[3] = c.z; z[3] = c.w;
  }
}

__device__ __forceinline__ void store_step(float* fr, int64_t ld, int q, const float (&x)[4],
                                           const float (&y)[4], const float (&z)[4]) {
  const auto p = gp(fr);
  typedef __attribute__((address_space(1))) f32x4_a4* vp;
  if (ld) {
    *(vp)(p + 4 * q) = f32x4_a4{x[0], x[1], x[2], x[3]};
    *(vp)(p + ld + 4 * q) = f32x4_a4{y[0], y[1], y[2], y[3]};
    *(vp)(p + 2 * ld + 4 * q) = f32x4_a4{z[0], z[1], z[2], z[3]};
  } else {
    const vp v = (vp)(p + 12 * (int64_t)q);
    v[0] = f32x4_a4{x[0], y[0], z[0], x[1]};
    v[1] = f32x4_a4{y[1], z[1], x[2], y[2]};
    v[2] = f32x4_a4{z[2], x[3], y[3], z[3]};
  }
}

// One atom.
__device__ __forceinline__ void load_step(const float* fr, int64_t ld, int k, float (&x)[1],
                                          float (&y)[1], float (&z)[1]) {
  const auto p = gp(fr);
  if (ld) {
    x[0] = p[k];
    y[0] = p[ld + k];
    z[0] = p[2 * ld + k];
  } else {
    const f32x3_a4 v = *(const __attribute__((address_space(1))) f32x3_a4*)(p + 3 * (int64_t)k);
    x[0] = v.x;
    y[0] = v.y;
    z[0] = v.z;
  }
}

__device__ __forceinline__ void store_step(float* fr, int64_t ld, int k, const float (&x)[1],
                                           const float (&y)[1], const float (&z)[1]) {
  const auto p = gp(fr);
  if (ld) {
    p[k] = x[0];
    p[ld + k] = y[0];
    p[2 * ld + k] = z[0];
  } else {
    *(__attribute__((address_space(1))) f32x3_a4*)(p + 3 * (int64_t)k) = f32x3_a4{x[0], y[0], z[0]};
  }
}

}  // namespace fit_dev
