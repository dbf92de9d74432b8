// z-pass loader with the Y_lm(x) weighting of the Yamamoto correlator
// (correlator.h:435-436).
#pragma once

#include "ylm_device.h"

namespace fc {

// Along a row x and y are fixed, so Y_lm c is a polynomial of degree l in z
// over r^l: the row's coefficients are formed once per thread (one switch over
// (l, m)) and a sample costs four multiply-adds and a division instead of the
// whole formula of ylm_eval with its switch (256^3 FP64 weighted z pass 53.2 ->
// 49.7 us, the plain copy taking 48.6).  FP64; differs from ylm_eval by
// rounding (a few ulp).
//
// Several transforms of one l may share a launch: output rows g rows_per + r
// are the grid's row r weighted with m + g.
struct LoadYlm {
  int ell, m, n1;
  double c0, c;          // normalisation of m = 0 and of the others
  double x0, y0, z0;     // cell centres relative to the observer: x0 + i etc.
  uint32_t rows_per;
  int i0 = 0;            // x slab of row 0
  void shift_x(int dx) { i0 += dx; }
  struct Row {
    int ell;
    double s, z0;  // x^2 + y^2 (+ the reference's 1e-20), z of sample 0
    double a[5];
    __device__ __forceinline__ double operator()(double v, int k) const {
      if (ell == 0) return v * a[0];
      const double z = z0 + (double)k;
      const double ir2 = 1.0 / (s + z * z);
      if (ell == 2) return v * (((a[2] * z + a[1]) * z + a[0]) * ir2);
      return v * (((((a[4] * z + a[3]) * z + a[2]) * z + a[1]) * z + a[0]) * ir2 * ir2);
    }
  };
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
