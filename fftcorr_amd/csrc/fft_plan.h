// Host side of the 3D R2C/C2R FFT: plan (twiddle tables + tile shapes per
// axis) and launchers.  A plan replaces FftGrid::plan_fft
// (cc/grid/fft_grid.cc:69-115); the execute calls replace execute_fft /
// execute_ifft (:125-178), split into the z (rows) and y/x (columns) passes so
// callers can fuse their own loads into the z pass.
#pragma once

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "fc_internal.h"
#include "fft_gen.h"
#include "fft_kernels.h"

namespace fc {

constexpr int kMaxFftLen = 4096;
// Default z+y chunk (KiB of complex output per chunk; 0 = no chunking).
constexpr int kDefaultZyChunkKiB = 0;
constexpr size_t kLdsBudget = 65536;  // bytes of LDS per workgroup we allow

// Tile shape chosen for one transform axis (autotuned; see fft.hip).
struct AxisTiles {
  int tc = 0;  // columns (or rows) per workgroup
};

struct FftPlan {
  int device = 0;
  int n[3] = {0, 0, 0};
  int n2h = 0;
  // Complex row stride of the work grid: n2/2+1 rounded up to 128 bytes so
  // every row (and every tile of TC columns) starts on a 128-byte boundary.
  int ldc = 0;
  int prec = FC_FP64;
  bool fast[3] = {false, false, false};  // axis 2: the half-length row FFT
  int tile[3] = {0, 0, 0};
  // Register-chained plan variant per axis (FftCfgV; axis 2: the row FFT of
  // length n2/2) of the forward passes, which the autotuner times; 0 unless
  // it or imported wisdom chose another.  Inverse passes use variant 0.
  int var[3] = {0, 0, 0};
  // x slabs per z+y chunk: the y pass of a chunk reads the z pass's output
  // while it is still in the last-level cache (0: the whole grid at once).
  int zy_chunk = 0;
  int zy_chunk_kib = 0;
  // Twiddle tables exp(-2 pi i m / L) in the plan's precision.
  DeviceBuffer tw0, tw1;      // lengths n0, n1
  // Mixed-radix tables of the axes without a compile-time plan (axis 2: the
  // whole row length n2); null where fast[] or where only the direct DFT is left.
  std::shared_ptr<GenAxis> gen[3];
  DeviceBuffer tw2M, tw2N;    // lengths n2/2 (fast rows) and n2 (post-process / DFT)
  size_t csize() const { return prec == FC_FP64 ? sizeof(double2) : sizeof(float2); }
  int64_t nrows() const { return (int64_t)n[0] * n[1]; }
  size_t complex_bytes() const { return (size_t)n[0] * n[1] * ldc * csize(); }
};

// Values per thread of the register-chained plan of length L.
int fft_len_e(int L);
// Whether the register-chained kernels have plan variant var for length L.
bool fft_var_ok(int L, int var);

// Plan cache keyed by (device, shape, precision).
std::shared_ptr<FftPlan> get_fft_plan(int device, const int shape[3], int prec);
// An uncached plan built with the current wisdom (the autotuner's scratch plan).
std::shared_ptr<FftPlan> make_private_plan(int device, const int shape[3], int prec);
void set_tile_wisdom(int L, int prec, int kind, int tile);
int default_col_tile(int L, size_t cs);
int default_row_tile(int M, size_t cs);

// ---- launchers -------------------------------------------------------------
// Column view [A][L][G][B] for k_fft_cols_rc / k_dft_cols (see fft_kernels.h).
template <typename T, typename Tin = T>
struct ColView {
  const cplx<Tin>* in;
  int64_t inA, inL, inG;
  cplx<T>* out;
  int64_t outA, outL, outG;
  int A, G, B;
  int nout = 0, off = 0;  // nout == 0: all L outputs
};

// Compute units of the current device (queried once per device).
inline int current_device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  FC_HIP(hipGetDevice(&dev));
  int n = dev >= 0 && dev < 64 ? cache[dev].load(std::memory_order_relaxed) : 0;
  if (n <= 0) {
    FC_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    if (dev >= 0 && dev < 64) cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Column pass of the L outputs (or the pruned ones) of a view: the compile-time
// plan where the length has one and the tile's offsets fit 32 bits, else the
// mixed-radix pass (gen, FP64 arithmetic), else direct sums.
template <typename T, int DIR, typename Tin = T>
void launch_cols(int L, const ColView<T, Tin>& v, int tc, const cplx<T>* tw, hipStream_t s,
                 const GenAxis* gen, int var = 0);

// Column pass stored in T with arithmetic in the wider A where the
// register-chained kernel takes L (tw_a: twiddles in A), else as launch_cols
// (tw_t).
template <typename T, int DIR, typename A>
void launch_cols_wide(int L, const ColView<T>& v, int tc, const cplx<A>* tw_a,
                      const cplx<T>* tw_t, hipStream_t s, const GenAxis* gen, int var = 0);

// In-place y pass over the work grid [n0][n1][ldc].
template <typename T>
ColView<T> y_view(const FftPlan& p, cplx<T>* d) {
  const int64_t ldc = p.ldc;
  return ColView<T>{d, (int64_t)p.n[1] * ldc, ldc, 0, d, (int64_t)p.n[1] * ldc, ldc, 0,
                    p.n[0], 1, p.n2h};
}
// In-place x pass over the work grid: L = n0, groups = the n1 rows of each slab.
template <typename T>
ColView<T> x_view(const FftPlan& p, cplx<T>* d) {
  const int64_t ldc = p.ldc;
  return ColView<T>{d, 0, (int64_t)p.n[1] * ldc, ldc, d, 0, (int64_t)p.n[1] * ldc, ldc,
                    1, p.n[1], p.n2h};
}

// z pass (R2C rows) stored in T.  With A wider than T, the register-chained
// kernel computes in A with the twiddles of the A-precision plan *pa (same
// shape), exchanging through LDS in T.
// in2 / nrows1 (optional): rows from nrows1 on are read from in2 (a second
// grid of the same shape), register-chained row lengths only.
template <typename T, typename Tin, class Loader, typename A = T>
void launch_rows_r2c(const FftPlan& p, const Tin* in, int64_t ldi, cplx<T>* out, int64_t ldo,
                     Loader ld, hipStream_t s, int64_t nrows = -1, const FftPlan* pa = nullptr,
                     const Tin* in2 = nullptr, int64_t nrows1 = 0);

// nrows rows of ldi complex -> real rows of ldo; nsel > 0 keeps only samples
// (o - off) mod n2, o < nsel (pruned inverse).  grp: rows of one batch member
// (0: one member), where rows are transformed in pairs.
template <typename T, typename Tout>
void launch_rows_c2r(const FftPlan& p, const cplx<T>* in, int64_t ldi, Tout* out, int64_t ldo,
                     hipStream_t s, int64_t nrows = -1, int nsel = 0, int off = 0,
                     int64_t grp = 0);

// y then x forward passes over the complex work grid [n0][n1][ldc].
template <typename T>
void fft_yx_forward(const FftPlan& p, cplx<T>* data, hipStream_t s) {
  launch_cols<T, -1>(p.n[1], y_view<T>(p, data), p.tile[1], p.tw1.as<cplx<T>>(), s,
                     p.gen[1].get(), p.var[1]);
  launch_cols<T, -1>(p.n[0], x_view<T>(p, data), p.tile[0], p.tw0.as<cplx<T>>(), s,
                     p.gen[0].get(), p.var[0]);
}

// x then y inverse passes.
template <typename T>
void fft_xy_inverse(const FftPlan& p, cplx<T>* data, hipStream_t s) {
  launch_cols<T, +1>(p.n[0], x_view<T>(p, data), p.tile[0], p.tw0.as<cplx<T>>(), s,
                     p.gen[0].get());
  launch_cols<T, +1>(p.n[1], y_view<T>(p, data), p.tile[1], p.tw1.as<cplx<T>>(), s,
                     p.gen[1].get());
}

}  // namespace fc
