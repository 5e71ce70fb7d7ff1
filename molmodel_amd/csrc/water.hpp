// water.hpp -- rigid-water constraint solver shared by the integrator and
// the replica-exchange velocity moves: two O-H length constraints
// (value 0.5 (r^2 - l^2), constraint.cpp:30-66) and one H-O-H angle
// constraint (constraint.cpp:68-112, geograd.cpp:59-103), solved with the
// reference's Newton iteration (constraint.cpp:295-358) in FP64.
//
// The solver is one chain of FP64 instructions in a kernel that has less than
// one wavefront per SIMD, so its time is their number.  Gradients are
// therefore kept as the five vectors they consist of (the O-H1 length reaches
// O and H1, the O-H2 length O and H2, the angle all three sites) instead of
// three rows of nine; masses enter as reciprocals; the angle's deviation is
// taken from the sine of the difference, not from an arc cosine; the 3x3
// system is solved by cofactors with one division; and the velocity step
// hands its gradients at the unmoved positions on to the position step.
// Rattle and three Newton passes were some 3000 instructions and are 1200.
#pragma once
#include <hip/hip_runtime.h>

namespace mmamd {

// target geometry: O-H length, H-O-H angle (radians)
struct WaterGeom {
  double bond, t0, cos0, sin0;
};
inline WaterGeom water_geom(double bond, double angle_deg) {
  const double t0 = angle_deg * (M_PI / 180.0);
  return {bond, t0, cos(t0), sin(t0)};
}

// gradients of one configuration: length 1 is r1 on O and -r1 on H1, length 2
// r2 on O and -r2 on H2, the angle o on O, p on H1 and q on H2
struct WaterGrad {
  double r1[3], r2[3], o[3], p[3], q[3];
};

__device__ __forceinline__ double dot3(const double *a, const double *b) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// gradients and, if val is given, constraint values
// (constraint.cpp:30-112, geograd.cpp:59-103)
template <bool VALUES>
__device__ __forceinline__ void water_constraints(const double *x, const WaterGeom &w, WaterGrad &c,
                                                  double *val) {
  // angle H1-O-H2: a = H1 - O = -r1, b = H2 - O = -r2
#pragma unroll
  for (int d = 0; d < 3; d++) { c.r1[d] = x[d] - x[3 + d]; c.r2[d] = x[d] - x[6 + d]; }
  const double a2 = dot3(c.r1, c.r1), b2 = dot3(c.r2, c.r2), ab = dot3(c.r1, c.r2);
  const double ma = rsqrt(a2), mb = rsqrt(b2), t0a = ma * mb;
  const double t3 = -t0a * ab * ma * ma, t4 = -t0a * ab * mb * mb;
  double ct = ab * t0a;
  ct = ct > 1 ? 1 : (ct < -1 ? -1 : ct);
  const double s2t = 1 - ct * ct;
  const bool flat = s2t < 64.0 * 2.220446049250313e-16;
  const double is = flat ? 0 : rsqrt(s2t);
#pragma unroll
  for (int d = 0; d < 3; d++) {   // -1/sin times the derivative of cos
    c.p[d] = (c.r2[d] * t0a + c.r1[d] * t3) * is;
    c.q[d] = (c.r1[d] * t0a + c.r2[d] * t4) * is;
    c.o[d] = -c.p[d] - c.q[d];
  }
  if constexpr (VALUES) {
    val[0] = 0.5 * (a2 - w.bond * w.bond);
    val[1] = 0.5 * (b2 - w.bond * w.bond);
    // t - t0 from z = sin(t - t0): near the target the arc sine's series
    // (through z^9; the next term is below 2^-65 of z at |z| = 1/64),
    // elsewhere, and where t - t0 is not within a quarter turn, the angle
    const double st = s2t * is, z = st * w.cos0 - ct * w.sin0;
    if (!flat && fabs(z) < 0.015625 && ct * w.cos0 + st * w.sin0 > 0) {
      const double z2 = z * z;
      val[2] = z + z * z2 * (1.0 / 6 + z2 * (3.0 / 40 + z2 * (15.0 / 336 + z2 * (105.0 / 3456))));
    } else {
      val[2] = (flat ? (ct > 0 ? 0 : M_PI) : acos(ct)) - w.t0;
    }
  }
}

// 3x3 Gaussian elimination with partial pivoting
__device__ inline bool solve3_pivot(double s[3][3], double *x) {
  for (int c = 0; c < 3; c++) {
    int piv = c;
    for (int r = c + 1; r < 3; r++)
      if (fabs(s[r][c]) > fabs(s[piv][c])) piv = r;
    if (s[piv][c] == 0) return false;
    if (piv != c) {
      for (int k = 0; k < 3; k++) { const double t = s[c][k]; s[c][k] = s[piv][k]; s[piv][k] = t; }
      const double t = x[c]; x[c] = x[piv]; x[piv] = t;
    }
    for (int r = c + 1; r < 3; r++) {
      const double m = s[r][c] / s[c][c];
      for (int k = c; k < 3; k++) s[r][k] -= m * s[c][k];
      x[r] -= m * x[c];
    }
  }
  for (int c = 2; c >= 0; c--) {
    double t = x[c];
    for (int k = c + 1; k < 3; k++) t -= s[c][k] * x[k];
    x[c] = t / s[c][c];
  }
  return true;
}

// By cofactors where the determinant is of the size of the diagonal's product
// (a water's is 0.997 of it), by elimination where it is not: a bent molecule
// stretched flat, masses of very different size.
__device__ __forceinline__ bool solve3(double s[3][3], double *x) {
  const double c0 = s[1][1] * s[2][2] - s[1][2] * s[2][1];
  const double c1 = s[1][2] * s[2][0] - s[1][0] * s[2][2];
  const double c2 = s[1][0] * s[2][1] - s[1][1] * s[2][0];
  const double det = s[0][0] * c0 + s[0][1] * c1 + s[0][2] * c2;
  if (!(fabs(det) > 0.01 * fabs(s[0][0] * s[1][1] * s[2][2]))) return solve3_pivot(s, x);
  const double id = 1.0 / det, b0 = x[0], b1 = x[1], b2 = x[2];
  x[0] = (b0 * c0 + b1 * (s[0][2] * s[2][1] - s[0][1] * s[2][2]) +
          b2 * (s[0][1] * s[1][2] - s[0][2] * s[1][1])) * id;
  x[1] = (b0 * c1 + b1 * (s[0][0] * s[2][2] - s[0][2] * s[2][0]) +
          b2 * (s[0][2] * s[1][0] - s[0][0] * s[1][2])) * id;
  x[2] = (b0 * c2 + b1 * (s[0][1] * s[2][0] - s[0][0] * s[2][1]) +
          b2 * (s[0][0] * s[1][1] - s[0][1] * s[1][0])) * id;
  return true;
}

// s[a][b] = (gradient a of c) . (gradient b of c0) / masses
__device__ __forceinline__ void water_matrix(const WaterGrad &c, const WaterGrad &c0, const double *im,
                                             double s[3][3]) {
  s[0][0] = dot3(c.r1, c0.r1) * (im[0] + im[1]);
  s[0][1] = dot3(c.r1, c0.r2) * im[0];
  s[0][2] = dot3(c.r1, c0.o) * im[0] - dot3(c.r1, c0.p) * im[1];
  s[1][0] = dot3(c.r2, c0.r1) * im[0];
  s[1][1] = dot3(c.r2, c0.r2) * (im[0] + im[2]);
  s[1][2] = dot3(c.r2, c0.o) * im[0] - dot3(c.r2, c0.q) * im[2];
  s[2][0] = dot3(c.o, c0.r1) * im[0] - dot3(c.p, c0.r1) * im[1];
  s[2][1] = dot3(c.o, c0.r2) * im[0] - dot3(c.q, c0.r2) * im[2];
  s[2][2] = dot3(c.o, c0.o) * im[0] + dot3(c.p, c0.p) * im[1] + dot3(c.q, c0.q) * im[2];
}

// sum over the constraints of x[a] (gradient a) / masses
__device__ __forceinline__ void water_shift(const WaterGrad &c, const double *im, const double *x,
                                            double *dx) {
#pragma unroll
  for (int d = 0; d < 3; d++) {
    dx[d] = (x[0] * c.r1[d] + x[1] * c.r2[d] + x[2] * c.o[d]) * im[0];
    dx[3 + d] = (x[2] * c.p[d] - x[0] * c.r1[d]) * im[1];
    dx[6 + d] = (x[2] * c.q[d] - x[1] * c.r2[d]) * im[2];
  }
}

// constraint.cpp:295-335 from the gradients c0 at the old positions (im:
// reciprocal masses); returns false if not converged
__device__ inline bool shake_water(double *x, double *v, const WaterGrad &c0, const double *im, double dt,
                                   const WaterGeom &w, double tol, int maxit) {
  const double invdt = dt > 0 ? 1 / dt : 0;
  for (int it = 0; it < maxit; it++) {
    WaterGrad c;
    double xs[3], s[3][3], dx[9];
    water_constraints<true>(x, w, c, xs);
    bool sat = true;
#pragma unroll
    for (int a = 0; a < 3; a++) { xs[a] = -xs[a]; if (fabs(xs[a]) > tol) sat = false; }
    if (sat) return true;
    water_matrix(c, c0, im, s);
    if (!solve3(s, xs)) return false;
    water_shift(c0, im, xs, dx);
#pragma unroll
    for (int d = 0; d < 9; d++) { x[d] += dx[d]; v[d] += dx[d] * invdt; }
  }
  return false;
}

// constraint.cpp:336-358 from the gradients at the positions
__device__ __forceinline__ void rattle_water(double *v, const WaterGrad &c, const double *im) {
  double xs[3], s[3][3], dx[9];
  xs[0] = xs[1] = xs[2] = 0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    xs[0] -= c.r1[d] * (v[d] - v[3 + d]);
    xs[1] -= c.r2[d] * (v[d] - v[6 + d]);
    xs[2] -= c.o[d] * v[d] + c.p[d] * v[3 + d] + c.q[d] * v[6 + d];
  }
  water_matrix(c, c, im, s);
  if (!solve3(s, xs)) return;
  water_shift(c, im, xs, dx);
#pragma unroll
  for (int d = 0; d < 9; d++) v[d] += dx[d];
}

}  // namespace mmamd
