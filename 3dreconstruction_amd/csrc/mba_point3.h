// Damped 3 x 3 point blocks V + D^2 (xx xy xz yy yz zz): one test of positive
// definiteness, and from the same leading minors the inverse (right-hand side,
// back substitution, matvecs) and the triangular factor (rows of the explicit
// S).  The fused multiply-adds are written out, so every kernel that includes
// this -- and a host build -- rounds alike and decides alike.
#ifndef MBA_POINT3_H_
#define MBA_POINT3_H_

#include <cmath>

#if defined(__HIPCC__)
#define MBA_POINT3 __host__ __device__ __forceinline__
#else
#define MBA_POINT3 inline
#endif

namespace mba {

// V with its LM diagonal, diag(V) clamped, over the radius
// (levenberg_marquardt_strategy.cc:104-111).
MBA_POINT3 void damp3(const double v[6], double min_diag, double max_diag, double inv_radius, double a[6]) {
  a[0] = fma(fmin(fmax(v[0], min_diag), max_diag), inv_radius, v[0]);
  a[1] = v[1];
  a[2] = v[2];
  a[3] = fma(fmin(fmax(v[3], min_diag), max_diag), inv_radius, v[3]);
  a[4] = v[4];
  a[5] = fma(fmin(fmax(v[5], min_diag), max_diag), inv_radius, v[5]);
}

// Cofactors and determinant; ok: positive definite by Sylvester's criterion
// (a00 > 0, leading 2 x 2 minor > 0, det > 0).
struct Minors3 {
  double c00, c01, c02, c11, c12, c22, det;
  bool ok;
  MBA_POINT3 explicit Minors3(const double a[6]) {
    c00 = fma(a[3], a[5], -(a[4] * a[4]));
    c01 = fma(a[2], a[4], -(a[1] * a[5]));
    c02 = fma(a[1], a[4], -(a[2] * a[3]));
    c11 = fma(a[0], a[5], -(a[2] * a[2]));
    c12 = fma(a[1], a[2], -(a[0] * a[4]));
    c22 = fma(a[0], a[3], -(a[1] * a[1]));
    det = fma(a[2], c02, fma(a[0], c00, a[1] * c01));
    ok = a[0] > 0.0 && c22 > 0.0 && det > 0.0;
  }
};

// FP64 inverse: adjugate over the determinant, one division; false if the block
// is not positive definite.
MBA_POINT3 bool inv3_spd(const double a[6], double o[6]) {
  const Minors3 m(a);
  if (!m.ok) return false;
  const double id = 1.0 / m.det;
  o[0] = m.c00 * id;
  o[1] = m.c01 * id;
  o[2] = m.c02 * id;
  o[3] = m.c11 * id;
  o[4] = m.c12 * id;
  o[5] = m.c22 * id;
  return true;
}

// L^-T's three columns applied on the right, for V + D^2 = L L': the squared
// pivots are the ratios a00, c22 / a00, det / c22 of the leading minors that
// inv3_spd tests, so a block has a factor exactly when it has an inverse.  A
// Cholesky of the block decides by differences that round otherwise: of 20,000
// two-view blocks with a baseline of 1e-8 of the depth, at radius 1e16, 1,361
// had an inverse (in the right-hand side) and no factor (in S), and where both
// existed they disagreed by 35 % along the weak direction; these agree to
// 4e-16 (medians).  A block without one gives zeros: the pass or the
// re-damping has flagged it by the same test.
struct Factor3 {
  double i00 = 0.0, i11 = 0.0, i22 = 0.0, l10 = 0.0, l20 = 0.0, l21 = 0.0;
  // rsqrt(d) = 1 / sqrt(d)
  template <typename F>
  MBA_POINT3 bool of(const double a[6], F&& rsqrt) {
    const Minors3 m(a);
    if (!m.ok) return false;
    const double r0 = rsqrt(a[0]), r1 = rsqrt(m.c22), r2 = rsqrt(m.det);
    i00 = r0;
    i11 = a[0] * r0 * r1;
    i22 = m.c22 * r1 * r2;
    l10 = a[1] * r0;
    l20 = a[2] * r0;
    l21 = -m.c12 * r0 * r1;
    return true;
  }
  // z with z L' = w (forward substitution along the row).
  template <typename T>
  MBA_POINT3 void solve(const T w[3], T z[3]) const {
    const double z0 = (double)w[0] * i00;
    const double z1 = fma(-l10, z0, (double)w[1]) * i11;
    const double z2 = fma(-l21, z1, fma(-l20, z0, (double)w[2])) * i22;
    z[0] = (T)z0;
    z[1] = (T)z1;
    z[2] = (T)z2;
  }
};

}  // namespace mba

#endif  // MBA_POINT3_H_
