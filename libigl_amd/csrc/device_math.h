// device_math.h -- FP32 device helpers shared by the traversal kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace gwn {

// Lane masks of a wavefront held in scalar registers.  (A condition kept as a
// bool and balloted later costs two VALU instructions more.)
__device__ __forceinline__ uint64_t lanes_at_most(uint32_t v, uint32_t i) {
  return __builtin_amdgcn_uicmp(v, i, 37);  // ICMP_ULE
}
__device__ __forceinline__ uint64_t lanes_beyond(float l2, float r2) {
  return __builtin_amdgcn_fcmpf(l2, r2, 10);  // FCMP_UGT: !(l2 <= r2)
}
__device__ __forceinline__ uint64_t lanes_beyond(double l2, double r2) { return __builtin_amdgcn_fcmp(l2, r2, 10); }
__device__ __forceinline__ uint64_t lanes_above(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, 2); }  // OGT
__device__ __forceinline__ uint64_t lanes_below_value(float a, float b) {
  return __builtin_amdgcn_fcmpf(a, b, 4);  // OLT
}
__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// atan on [0,1] as a * P(a^2), P of degree 8: a weighted least-squares /
// Lawson fit to atan(x)/x on 4000 Chebyshev nodes (computed for this
// library); max error 1.2e-8 in exact arithmetic, ~1e-7 rad when evaluated in
// FP32 (comparable to a correctly rounded atan2f).
__device__ __forceinline__ float atan01(float a) {
  const float s = a * a;
  float p = 0.0028501534834504128f;
  p = fmaf(p, s, -0.016069747507572174f);
  p = fmaf(p, s, 0.04269346594810486f);
  p = fmaf(p, s, -0.07504474371671677f);
  p = fmaf(p, s, 0.10641028732061386f);
  p = fmaf(p, s, -0.14203672111034393f);
  p = fmaf(p, s, 0.1999262422323227f);
  p = fmaf(p, s, -0.33333075046539307f);
  p = fmaf(p, s, 1.0f);
  return a * p;
}

// atan2 (not both arguments zero; for y = 0 it takes the sign of y).
__device__ __forceinline__ float atan2_fast(float y, float x) {
  const float ax = fabsf(x), ay = fabsf(y);
  const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
  float r = atan01(mn * __builtin_amdgcn_rcpf(mx));
  if (ay > ax) r = 1.57079632679489662f - r;
  if (x < 0.0f) r = 3.14159265358979324f - r;
  return copysignf(r, y);
}

// Far field of an order-0/1/2 Taylor expansion written as one polynomial in
// the direction to the query.  For the offset q (l2 = |q|^2), x = q/|q| (kept
// normalised so that the cubic cannot overflow for distant queries) and
// m = 1/|q| the value is
//   m^2 [ x.b + m ( Qf(x) + m G(x) ) ]
// with b = b.xyz.  |x| = 1 takes z^2 out of the quadratic form and of the
// cubic, which leaves a constant and three linear terms in its place and
// fewer operations (31 with the reciprocal square root, against 36 with both
// in homogeneous form):
//   Qf(x) = c.z + x (c.x x + c.w y + d.y z) + y (c.y y + d.x z)
//   G(x)  = x (f.y + x (d.z x + e.y y + e.z z) + y (e.w y + f.w z))
//         + y (f.z + y (d.w y + f.x z)) + e.x z
// The soup's slot records (k_write_slots) and the cloud's cell records
// (k_rec_poly) store their expansions in this form, through pack_far_field.

// m and m^2, and the bracket of the formula above
template <int ORDER, typename T, typename V4>
__device__ __forceinline__ T far_field_bracket(T x, T y, T z, T m, const V4& b, const V4& c, const V4& d, const V4& e,
                                               const V4& f) {
  // explicit multiply-adds (no compiler contraction): every kernel that
  // inlines this computes each term bit for bit the same
  x *= m;
  y *= m;
  z *= m;
  T t = fma(z, b.z, fma(y, b.y, x * b.x));  // x.b
  if (ORDER >= 1) {
    const T q1 = fma(d.y, z, fma(c.w, y, c.x * x)), q2 = fma(d.x, z, c.y * y);
    T qf = fma(x, q1, fma(y, q2, c.z));
    if (ORDER >= 2) {
      const T g1 = fma(e.z, z, fma(e.y, y, d.z * x)), g2 = fma(f.w, z, e.w * y), g3 = fma(f.x, z, d.w * y);
      const T gx = fma(x, g1, fma(y, g2, f.y)), gy = fma(y, g3, f.z);
      qf = fma(m, fma(x, gx, fma(y, gy, e.x * z)), qf);
    }
    t = fma(m, qf, t);
  }
  return t;
}

// the FP32 value; a caller that sums it may add m * m * bracket by itself
template <int ORDER>
__device__ __forceinline__ float far_field_poly(float x, float y, float z, float l2, const float4& b,
                                                const float4& c, const float4& d, const float4& e,
                                                const float4& f) {
  const float m = __builtin_amdgcn_rsqf(l2);
  return (m * m) * far_field_bracket<ORDER>(x, y, z, m, b, c, d, e, f);
}

// Coefficients of an expansion in the record form of far_field_bracket:
// b.xyz; the quadratic form by xx yy zz xy yz xz; the cubic by
// x^3 y^3 z^3 x^2y x^2z xy^2 y^2z xz^2 yz^2 xyz.  r: the 20 values of
// b c d e f (r[3], the free fourth value of b, is not written).
template <typename T>
__device__ __forceinline__ void pack_far_field(const double* b, const double* q, const double* g, T* r) {
  for (int k = 0; k < 3; ++k) r[k] = (T)b[k];
  r[4] = (T)(q[0] - q[2]);   // c.x  x^2
  r[5] = (T)(q[1] - q[2]);   // c.y  y^2
  r[6] = (T)q[2];            // c.z  1
  r[7] = (T)q[3];            // c.w  xy
  r[8] = (T)q[4];            // d.x  yz
  r[9] = (T)q[5];            // d.y  xz
  r[10] = (T)(g[0] - g[7]);  // d.z  x^3
  r[11] = (T)(g[1] - g[8]);  // d.w  y^3
  r[12] = (T)g[2];           // e.x  z
  r[13] = (T)(g[3] - g[8]);  // e.y  x^2y
  r[14] = (T)(g[4] - g[2]);  // e.z  x^2z
  r[15] = (T)(g[5] - g[7]);  // e.w  xy^2
  r[16] = (T)(g[6] - g[2]);  // f.x  y^2z
  r[17] = (T)g[7];           // f.y  x
  r[18] = (T)g[8];           // f.z  y
  r[19] = (T)g[9];           // f.w  xyz
}

// 1/sqrt(x) to FP64 rounding: with the hardware estimate r (about 2^-26
// relative) and e = 1 - x r^2 it is r (1 - e)^(-1/2), the binomial series of
// which is taken to e^2: 1 + e/2 + 3 e^2/8
__device__ __forceinline__ double rsqrt64(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * r), r, 1.0);
  return fma(r * e, fma(0.375, e, 0.5), r);
}

// A running sum of angles atan2(y, x), kept as the product of the x + i y
// scaled by powers of two and the number of full turns: the sum is
// 2 pi turns + atan2(im, re).  A term costs a complex multiplication, a
// rescaling and the turn count (16 operations) where an atan2 of its own
// costs about 25 in FP32 and over 100 in FP64, and each multiplication moves
// the angle by at most about one unit of rounding of 1 rad, where a running
// sum of angles rounds at the size of the sum.
template <typename T>
struct AngleSum {
  T re = T(1), im = T(0);
  int32_t turns = 0;

  // Adds atan2(y, x) (y, x not NaN, not both zero, their product with the
  // unit-sized sum not overflowing, and far enough above the denormals that
  // its parts round as the sum does) and returns true; otherwise leaves the
  // sum as it is and returns false.
  __device__ __forceinline__ bool add(T y, T x) {
    constexpr T least = sizeof(T) == 4 ? T(1e-30) : T(1e-290);  // smallest normal / epsilon: 1.0e-31, 1.0e-292
    const T r = fma(-im, y, re * x), i = fma(re, y, im * x);
    const T s = fmax(fabs(r), fabs(i));
    if (!(s > least && s < T(INFINITY))) return false;
    // both arguments on one side of the real axis and the product on the
    // other: the sum of the two left [-pi, pi]
    const int32_t a = sign_word(im), b = sign_word(y), c = sign_word(i);
    turns += ((~(a ^ b) & (a ^ c)) >> 31) & ((a >> 31) | 1);
    const int e = -frexp_exponent(s);
    re = scale(r, e);
    im = scale(i, e);
    return true;
  }
  __device__ __forceinline__ double total() const {
    return fma((double)turns, 6.283185307179586476925286766559, (double)argument(im, re));
  }

 private:
  static __device__ __forceinline__ float argument(float y, float x) { return atan2_fast(y, x); }
  static __device__ __forceinline__ double argument(double y, double x) { return atan2(y, x); }
  static __device__ __forceinline__ int32_t sign_word(float v) { return __float_as_int(v); }
  static __device__ __forceinline__ int32_t sign_word(double v) { return __double2hiint(v); }
  static __device__ __forceinline__ int frexp_exponent(float v) { return __builtin_amdgcn_frexp_expf(v); }
  static __device__ __forceinline__ int frexp_exponent(double v) { return __builtin_amdgcn_frexp_exp(v); }
  static __device__ __forceinline__ float scale(float v, int e) { return __builtin_ldexpf(v, e); }
  static __device__ __forceinline__ double scale(double v, int e) { return __builtin_ldexp(v, e); }
};

}  // namespace gwn
