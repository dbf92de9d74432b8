// Mixed-radix FFT passes for lengths without a compile-time plan: every
// length up to 4096 whose prime factors are at most 13, and (as a chirp
// convolution) every other length up to kGenMaxBlue.  The stage sequence is
// data (GenStage tables in device memory), the butterflies are compile-time
// radices selected by a wave-uniform switch, so one kernel serves all lengths.
// Arithmetic is FP64 whatever the storage type; see fft_gen_kernels.h.
#pragma once

#include <algorithm>
#include <memory>
#include <vector>

#include "fc_internal.h"
#include "fft_kernels.h"

namespace fc {

// One Stockham stage: butterfly j (j < nb) of radix R reads elements
// j + r nb and writes (j / NS) NS R + j % NS + r NS; twiddle step tws =
// N / (NS R); dm, ds: division by NS as (umulhi(j, dm) + j) >> ds.
struct GenStage {
  int R, nb, NS, tws;
  uint32_t dm;
  int ds, pad0, pad1;
};

constexpr int kGenMaxLen = 4096;   // longest length of the stages
constexpr int kGenMaxBlue = 2048;  // longest length taken as a chirp convolution (N <= 4096)
constexpr int kGenRadSmall = 10;   // largest radix of the small-register kernels

// Device tables of one length L.  Stages of the length-N FFT in order, then
// (for a transform followed by its inverse in the same kernel) stages 1 ..
// ns - 1 of the plan with the radices reversed, whose first stage has the
// radix of the last forward one.  blue: N >= 2 L - 1, the transform is the
// convolution with chirp[e] = exp(-i pi e^2 / L) through filt = FFT_N of the
// conjugate chirp / N.
struct GenAxis {
  int L = 0, N = 0, ns = 0;
  bool blue = false;
  int tcol = 0;  // threads per column: the largest nb
  int rmax = 0;  // largest radix
  std::vector<int> radices;
  DeviceBuffer stages, W, chirp, filt;
};

// Radices of a length (all prime factors <= 13), smallest first; empty if it
// has another factor.  Fewest stages, then the largest smallest radix (the
// threads per column), then the smallest largest one (registers).
std::vector<int> gen_radices(int L);
// Whether this engine takes a length, its stages (no tables; N = 0 if it does
// not take it) and its tables on the current device.
bool gen_len_ok(int L);
GenAxis gen_axis_stages(int L);
std::shared_ptr<GenAxis> make_gen_axis(int L);
// LDS bytes of a workgroup of the row passes of a length, rows stored in
// complex values of cs bytes.
size_t gen_row_lds(const GenAxis& ax, size_t cs);

// Columns of [A][L][G][B] (ColView of fft_plan.h): outputs as k_fft_cols_rc.
struct GenCols {
  int64_t inA, inL, inG, outA, outL, outG;
  int A, G, B, nout, offm;
};
template <typename Tin, typename Tout>
void launch_gen_cols(const GenAxis& ax, const cplx<Tin>* in, cplx<Tout>* out, const GenCols& v,
                     int dir, hipStream_t s);

// Real rows of n2 samples (ax: the length n2) <-> the n2/2+1 Hermitian half,
// two rows per complex transform, paired within groups of grp rows (grp divides
// nrows).  nsel, offm as k_fft_rows_c2r_rc.
template <typename Tin, typename Tout, class Loader>
void launch_gen_r2c(const GenAxis& ax, const Tin* in, int64_t ldi, cplx<Tout>* out, int64_t ldo,
                    int64_t nrows, int64_t grp, Loader ld, hipStream_t s);
template <typename T, typename Tout>
void launch_gen_c2r(const GenAxis& ax, const cplx<T>* in, int64_t ldi, Tout* out, int64_t ldo,
                    int64_t nrows, int64_t grp, int nsel, int offm, hipStream_t s);

}  // namespace fc
