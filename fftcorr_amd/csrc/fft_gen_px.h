// Fused x pass of the mixed-radix lengths (see fused_x.h for the pass and
// fft_gen.h for the engine).
#pragma once

#include "fft_gen.h"
#include "fused_x.h"

namespace fc {

// Whether the pass takes a length: no chirp convolution, one column's threads
// and both grids' column (interlaced) within a workgroup.
inline bool gen_px_ok(const GenAxis& ax) {
  return !ax.blue && ax.tcol <= 512 && (size_t)ax.N * 2 * sizeof(double2) <= 65536;
}
template <typename T, typename TI, int MODE>
void launch_gen_px(const GenAxis& ax, const PxArgs<T>& p, hipStream_t s);

}  // namespace fc
