// z-pass loader with the Y_lm(x) weighting of the Yamamoto correlator
// (correlator.h:435-436).
#pragma once

#include "ylm_device.h"

namespace fc {

// 1 / d for normal d > 0 well inside the exponent range: the hardware's
// estimate and two Newton steps (to about 1 ulp), without the scaling and the
// special cases of the division.  With one reciprocal per two samples the
// weighted z pass of 1024 x 1024 x 768 takes 1634 us instead of 1777 (the plain
// copy 1260).
__device__ __forceinline__ double inv_normal(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  return fma(r, fma(-d, r, 1.0), r);
}

// Along a row x and y are fixed, so Y_lm c is a polynomial of degree l in z
// over r^l: the row's coefficients are formed once per thread (one switch over
// (l, m)) and a sample costs four multiply-adds and half a reciprocal instead of
// the whole formula of ylm_eval with its switch (256^3 FP64 weighted z pass 53.2
// -> 49.7 us, still with a division per sample, the plain copy taking 48.6).
// FP64; differs from ylm_eval by rounding (a few ulp).
//
// Several transforms of one l may share a launch: output rows g rows_per + r
// are the grid's row r weighted with m + g.
struct LoadYlm {
  int ell, m, n1;
  double c0, c;          // normalisation of m = 0 and of the others
  double x0, y0, z0;     // cell centres relative to the observer: x0 + i etc.
  uint32_t rows_per, nm;
  int i0 = 0;            // x slab of row 0
  void shift_x(int dx) { i0 += dx; }
  struct Row {
    int ell;
    double s, z0;  // x^2 + y^2 (+ the reference's 1e-20), z of sample 0
    double a[5];
    __device__ __forceinline__ double weight(double z, double ir2) const {
      if (ell == 2) return ((a[2] * z + a[1]) * z + a[0]) * ir2;
      return ((((a[4] * z + a[3]) * z + a[2]) * z + a[1]) * z + a[0]) * ir2 * ir2;
    }
    __device__ __forceinline__ double operator()(double v, int k) const {
      if (ell == 0) return v * a[0];
      const double z = z0 + (double)k;
      return v * weight(z, inv_normal(s + z * z));
    }
    // Samples k and k + 1: one reciprocal, of the product of their r^2.
    __device__ __forceinline__ double2 pair(double v, double w, int k) const {
      if (ell == 0) return make_double2(v * a[0], w * a[0]);
      const double z = z0 + (double)k, y = z + 1.0;
      const double dz = s + z * z, dy = s + y * y;
      const double ir = inv_normal(dz * dy);
      return make_double2(v * weight(z, ir * dy), w * weight(y, ir * dz));
    }
  };
  // Block order over nb blocks: the members' blocks of one range of rows follow
  // each other on one XCD, so the grid's rows are read from memory once (256^3
  // FP64, five members: 245 -> 203 us; the mixed-radix rows, which their stages
  // bound, lose 4% by it and keep the plain order).
  __device__ __forceinline__ uint32_t block(uint32_t b, uint32_t nb) const {
    if (nm <= 1) return b;
    const uint32_t per = nb / nm;
    if (per * nm != nb || per % 8) return b;
    const uint32_t t = b >> 3, q = t / nm;
    return (t - q * nm) * per + q * 8 + (b & 7);
  }
  __device__ __forceinline__ uint32_t member(int64_t r) const {
    return r < (int64_t)rows_per ? 0u : (uint32_t)r / rows_per;
  }
  __device__ __forceinline__ int64_t src(int64_t r) const {
    return r - (int64_t)member(r) * rows_per;
  }
  __device__ __forceinline__ Row row(int64_t r) const {
    const int g = (int)member(r);
    r -= (int64_t)g * rows_per;
    const int i = i0 + (int)(r / n1), j = (int)(r % n1);
    const double x = x0 + (double)i * 1.0, y = y0 + (double)j * 1.0;
    Row w;
    w.ell = ell;
    w.s = x * x + y * y + 1e-20;
    w.z0 = z0;
    ylm_row(ell, m + g, x, y, m + g == 0 ? c0 : c, w.a);
    return w;
  }
};

}  // namespace fc
