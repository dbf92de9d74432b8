// Mixed-radix row passes (fft_gen.h): real rows <-> Hermitian half rows.
#include "fft_gen_kernels.h"
#include "load_ylm.h"

namespace fc {
namespace {

// First row of pair `item` (rows in groups of grp); true if it has a second.
__device__ __forceinline__ bool row_pair(int64_t item, int64_t grp, int64_t nrows, int64_t* r0) {
  const int64_t ppg = (grp + 1) / 2;
  const int64_t q = grp == nrows ? 0 : item / ppg;
  const int64_t in = 2 * (item - q * ppg);
  *r0 = q * grp + in;
  return in + 1 < grp && *r0 + 1 < nrows;
}

// Block (tcol, tr): tr pairs of rows.  The two rows of a pair are the real and
// imaginary part of one complex row of n2, so odd and even lengths take the
// same path and no half-length post-processing is needed.  Rows come in groups
// (batch members) of grp, and a pair never spans two groups: a member's
// results do not depend on its place.  LDS tr rows of lay.rs.
template <typename Tin, typename Tout, class Loader, bool BLUE, int RM>
__global__ void __launch_bounds__(gen_max_threads<RM>())
    k_gen_r2c(const Tin* in, int64_t ldi, cplx<Tout>* out, int64_t ldo, int64_t nrows, int64_t grp,
              LayGenRow lay, Loader ld, GenDev g) {
  using CL = cplx<typename std::conditional<BLUE, double, Tout>::type>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  CL* lds = reinterpret_cast<CL*>(smem_raw);
  const int c = threadIdx.y, j = threadIdx.x;
  const int L = g.L;
  int64_t r0;
  const bool two = row_pair((int64_t)blockIdx.x * blockDim.y + c, grp, nrows, &r0);
  const int64_t ra = r0 < nrows ? r0 : 0;  // rows past the end read row 0 (discarded)
  const int64_t rb = two ? r0 + 1 : 0;
  const auto la = ld.row(ra);
  const auto lb = ld.row(rb);
  const Tin* pa = in + ld.src(ra) * ldi + j;
  const Tin* pb = in + ld.src(rb) * ldi + j;
  // A row without a partner is paired with zeros: a partner's values would
  // enter its rounding.
  auto load = [&](int r, int u) {
    const double b = lb((double)pb[r * u], j + r * u);
    return double2{la((double)pa[r * u], j + r * u), two ? b : 0.0};
  };
  auto put = [&](int r, int u, double2 v) {
    lds[lay(c, j + r * u)] = to_cplx<typename ScalarOf<CL>::type>(v);
  };
  if constexpr (BLUE)
    gen_run_blue<RM>(lds, g.stg, g.ns, g.W, g.chirp, g.filt, L, c, j, lay, load, put, true);
  else
    gen_run<RM, 0>(lds, g.stg, g.ns, g.W, c, j, lay, load, NoMid{}, put, true);
  __syncthreads();
  if (r0 >= nrows) return;
  cplx<Tout>* da = out + r0 * ldo;
  // X_a = (Z[k] + conj Z[n-k]) / 2, X_b = -i (Z[k] - conj Z[n-k]) / 2.
  for (int k = j; k <= L / 2; k += blockDim.x) {
    const double2 zk = to_cplx<double>(lds[lay(c, k)]);
    const double2 zm = to_cplx<double>(lds[lay(c, k == 0 ? 0 : L - k)]);
    st_stream(da + k, to_cplx<Tout>(double2{0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y)}));
    if (two)
      st_stream(da + ldo + k, to_cplx<Tout>(double2{0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x)}));
  }
}

// Pairs of Hermitian half rows -> pairs of real rows (unnormalised; imaginary
// parts of the DC and Nyquist terms ignored).  nsel == 0: whole rows; else
// sample (o - off) mod n2 at o < nsel (offm = off mod n2).  Every input of a
// row is read in the first stage, so the real rows may overlay the complex
// ones.
template <typename T, typename Tout, bool BLUE, int RM>
__global__ void __launch_bounds__(gen_max_threads<RM>())
    k_gen_c2r(const cplx<T>* in, int64_t ldi, Tout* out, int64_t ldo, int64_t nrows, int64_t grp,
              LayGenRow lay, int nsel, int offm, GenDev g) {
  using CL = cplx<typename std::conditional<BLUE, double, T>::type>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  CL* lds = reinterpret_cast<CL*>(smem_raw);
  const int c = threadIdx.y, j = threadIdx.x;
  const int L = g.L;
  int64_t r0;
  const bool okb = row_pair((int64_t)blockIdx.x * blockDim.y + c, grp, nrows, &r0);
  const bool oka = r0 < nrows;
  const cplx<T>* xa = in + (oka ? r0 : 0) * ldi;
  const cplx<T>* xb = in + (okb ? r0 + 1 : 0) * ldi;
  // Z[k] = X_a[k] + i X_b[k] (k > n2/2: from the conjugates), conjugated for
  // the stages' sign.
  auto load = [&](int r, int u) {
    const int e = j + r * u;
    const bool low = 2 * e <= L;
    const int k = low ? e : L - e;
    double2 a = to_cplx<double>(xa[k]), b = to_cplx<double>(xb[k]);
    if (e == 0 || 2 * e == L) a.y = b.y = 0.0;
    if (!low) a.y = -a.y, b.y = -b.y;
    if (!okb) b = double2{0.0, 0.0};
    return double2{a.x - b.y, -(a.y + b.x)};
  };
  Tout* da = out + r0 * ldo;
  const int last = nsel == 0 ? L : nsel;
  const int shift = nsel == 0 ? 0 : offm;
  auto put = [&](int r, int u, double2 v) {
    int o = j + r * u + shift;
    if (o >= L) o -= L;
    for (; o < last; o += L) {
      if (oka) da[o] = Tout(v.x);
      if (okb) da[ldo + o] = Tout(-v.y);
    }
  };
  if constexpr (BLUE)
    gen_run_blue<RM>(lds, g.stg, g.ns, g.W, g.chirp, g.filt, L, c, j, lay, load, put, false);
  else
    gen_run<RM, 0>(lds, g.stg, g.ns, g.W, c, j, lay, load, NoMid{}, put, false);
}

constexpr size_t kRowLds = 65536;  // of a workgroup (gen_row_tile's limit)
struct RowShape {
  LayGenRow lay;
  int tr;
  size_t lds;
  unsigned nb;
};
RowShape row_shape(const GenAxis& ax, size_t cl, int64_t nrows, int64_t grp) {
  RowShape r;
  const int64_t items = (nrows + grp - 1) / grp * ((grp + 1) / 2);
  // A gap after every eighth element, so that neither the stages' strides nor
  // neighbouring rows meet in one bank; where one row with its gaps exceeds the
  // budget (FP64 values, more than 3640 of them), as many as it leaves room
  // for: a gap after every 16th to 128th element, none at 4096 points.
  r.lay = LayGenRow{ax.N + ax.N / 8 + 1, 3};
  while ((size_t)r.lay.rs * cl > kRowLds && r.lay.sh < 16)
    r.lay.rs = ax.N + ((ax.N - 1) >> ++r.lay.sh);
  r.tr = gen_row_tile(ax, (size_t)r.lay.rs * cl);
  r.lds = (size_t)r.tr * r.lay.rs * cl;
  if (r.lds > kRowLds) fail(FC_ERR_RUNTIME, "internal: row tile exceeds the LDS budget");
  const int64_t nb = (items + r.tr - 1) / r.tr;
  if (nb > INT32_MAX) fail(FC_ERR_INVALID, "transform too large for one launch");
  r.nb = (unsigned)nb;
  return r;
}

}  // namespace

size_t gen_row_lds(const GenAxis& ax, size_t cs) {
  return row_shape(ax, ax.blue ? sizeof(double2) : cs, 1, 1).lds;
}

template <typename Tin, typename Tout, class Loader>
void launch_gen_r2c(const GenAxis& ax, const Tin* in, int64_t ldi, cplx<Tout>* out, int64_t ldo,
                    int64_t nrows, int64_t grp, Loader ld, hipStream_t s) {
  const RowShape r = row_shape(ax, ax.blue ? sizeof(double2) : sizeof(cplx<Tout>), nrows, grp);
  if (r.nb == 0) return;
  auto go = [&](auto blue, auto rm) {
    hipLaunchKernelGGL(
        (k_gen_r2c<Tin, Tout, Loader, decltype(blue)::value, decltype(rm)::value>), dim3(r.nb),
        dim3((unsigned)ax.tcol, (unsigned)r.tr), r.lds, s, in, ldi, out, ldo, nrows, grp, r.lay,
        ld, gen_dev(ax));
  };
  gen_dispatch(ax, go);
  FC_LAUNCH_CHECK();
}

template <typename T, typename Tout>
void launch_gen_c2r(const GenAxis& ax, const cplx<T>* in, int64_t ldi, Tout* out, int64_t ldo,
                    int64_t nrows, int64_t grp, int nsel, int offm, hipStream_t s) {
  const RowShape r = row_shape(ax, ax.blue ? sizeof(double2) : sizeof(cplx<T>), nrows, grp);
  if (r.nb == 0) return;
  auto go = [&](auto blue, auto rm) {
    hipLaunchKernelGGL((k_gen_c2r<T, Tout, decltype(blue)::value, decltype(rm)::value>), dim3(r.nb),
                       dim3((unsigned)ax.tcol, (unsigned)r.tr), r.lds, s, in, ldi, out, ldo,
                       nrows, grp, r.lay, nsel, offm, gen_dev(ax));
  };
  gen_dispatch(ax, go);
  FC_LAUNCH_CHECK();
}

#define FC_GEN_R2C(Tin, Tout, Loader)                                                         \
  template void launch_gen_r2c<Tin, Tout, Loader>(const GenAxis&, const Tin*, int64_t,        \
                                                  cplx<Tout>*, int64_t, int64_t, int64_t,     \
                                                  Loader, hipStream_t);
FC_GEN_R2C(float, float, LoadCopy)
FC_GEN_R2C(double, float, LoadCopy)
FC_GEN_R2C(float, double, LoadCopy)
FC_GEN_R2C(double, double, LoadCopy)
FC_GEN_R2C(float, float, LoadYlm)
FC_GEN_R2C(double, float, LoadYlm)
FC_GEN_R2C(float, double, LoadYlm)
FC_GEN_R2C(double, double, LoadYlm)
#undef FC_GEN_R2C
#define FC_GEN_C2R(T, Tout)                                                                \
  template void launch_gen_c2r<T, Tout>(const GenAxis&, const cplx<T>*, int64_t, Tout*,     \
                                        int64_t, int64_t, int64_t, int, int, hipStream_t);
FC_GEN_C2R(float, float)
FC_GEN_C2R(double, double)
FC_GEN_C2R(float, double)
#undef FC_GEN_C2R

}  // namespace fc
