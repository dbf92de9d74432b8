// Fused x pass of the mixed-radix lengths (see fused_x.h for the pass and
// fft_gen.h for the engine).
#pragma once

#include "fft_gen.h"
#include "fused_x.h"

namespace fc {

// One launch over nb members (member i reads A, B at i a_bstride and writes
// pk, q at i pk_bstride, q_bstride; B is shared in cross mode).  T: storage of
// the spectra and pk; TI: combine, inverse and q.
template <typename T>
struct GenPx {
  const cplx<T>*A, *B;
  int n1, n2h;
  int64_t ldc;
  const double2 *ph0, *ph1, *ph2;
  T* pk;
  KSlots ks;
  void* q;
  int64_t ldq;
  int rs, offm, nb;
  int64_t a_bstride, pk_bstride, q_bstride;
};
// Whether the pass takes a length: no chirp convolution, one column's threads
// and both grids' column (interlaced) within a workgroup.
inline bool gen_px_ok(const GenAxis& ax) {
  return !ax.blue && ax.tcol <= 512 && (size_t)ax.N * 2 * sizeof(double2) <= 65536;
}
template <typename T, typename TI, int MODE>
void launch_gen_px(const GenAxis& ax, const GenPx<T>& p, hipStream_t s);

}  // namespace fc
