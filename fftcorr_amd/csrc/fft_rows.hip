// Row (z) passes with a compile-time plan and the choice between them, the
// mixed-radix pass and the direct sums.
#include "fft_plan.h"
#include "load_ylm.h"

namespace fc {

template <typename T, typename Tin, class Loader, typename A>
void launch_rows_r2c(const FftPlan& p, const Tin* in, int64_t ldi, cplx<T>* out, int64_t ldo,
                     Loader ld, hipStream_t s, int64_t nrows, const FftPlan* pa,
                     const Tin* in2, int64_t nrows1) {
  const size_t cs = sizeof(cplx<T>);
  if (nrows < 0) nrows = p.nrows();
  const int M = p.n[2] / 2;
  const int tr = p.tile[2];
  const cplx<T>* twN = p.tw2N.as<cplx<T>>();
  if (in2 && !(p.fast[2]))
    fail(FC_ERR_RUNTIME, "internal: two-grid z pass needs the register-chained rows");
  if (p.gen[2])
    return launch_gen_r2c<Tin, T>(*p.gen[2], in, ldi, out, ldo, nrows,
                                  std::min(nrows, p.nrows()), ld, s);
  if (p.fast[2]) {
    const FftPlan& pt = std::is_same<T, A>::value ? p : *pa;
    const cplx<A>* twMa = pt.tw2M.as<cplx<A>>();
    const cplx<A>* twNa = pt.tw2N.as<cplx<A>>();
    const int var = fft_var_ok(M, p.var[2]) ? p.var[2] : 0;
    // Wider arithmetic: at most two waves per workgroup (4 rows of M = 256):
    // small workgroups wait at few barriers of other waves (the 512^3 mixed
    // z pass: 0.375 ms with two waves against 0.384 with one; four waves
    // were slower than one in an earlier form of the kernel).
    const int cap = std::max(1, 128 / (M / (var == 1 ? 16 : fft_len_e(M))));
    int trc = std::is_same<T, A>::value ? tr : (tr < cap ? tr : cap);
    while (trc > 1 && (size_t)trc * row_pad_len(M) * cs > kLdsBudget) trc /= 2;
    auto go = [&](auto vtag, auto mtag) {
      constexpr int V = decltype(vtag)::value, Mv = decltype(mtag)::value;
      dim3 g((unsigned)((nrows + trc - 1) / trc));
      hipLaunchKernelGGL((k_fft_rows_r2c_rc<A, Tin, Mv, Loader, T, V>), g,
                         dim3(trc * (Mv / FftCfgV<Mv, V>::E)),
                         (size_t)trc * row_pad_len(Mv) * cs, s, in, ldi, out, ldo, nrows, trc,
                         twMa, twNa, ld, in2, nrows1);
    };
#define FC_R2C_RC_CASE(Mv)                                                       \
  case Mv:                                                                       \
    if constexpr (FftCfgV<Mv, 1>::fast) {                                        \
      if (var == 1) {                                                            \
        go(std::integral_constant<int, 1>{}, std::integral_constant<int, Mv>{}); \
        break;                                                                   \
      }                                                                          \
    }                                                                            \
    go(std::integral_constant<int, fft_plan_of<A, Mv>()>{},                      \
       std::integral_constant<int, Mv>{});                                       \
    break;
    switch (M) {
      FC_R2C_RC_CASE(8)
      FC_R2C_RC_CASE(16)
      FC_R2C_RC_CASE(32)
      FC_R2C_RC_CASE(64)
      FC_R2C_RC_CASE(128)
      FC_R2C_RC_CASE(192)
      FC_R2C_RC_CASE(256)
      FC_R2C_RC_CASE(384)
      FC_R2C_RC_CASE(512)
      FC_R2C_RC_CASE(768)
      FC_R2C_RC_CASE(1024)
      FC_R2C_RC_CASE(1536)
      FC_R2C_RC_CASE(2048)
    }
#undef FC_R2C_RC_CASE
  } else {
    dim3 g((unsigned)nrows);
    hipLaunchKernelGGL((k_dft_rows_r2c<T, Tin, Loader>), g, dim3(256),
                       (size_t)p.n[2] * sizeof(T), s, in, ldi, out, ldo, p.n[2], twN, ld);
  }
  FC_LAUNCH_CHECK();
}


template <typename T, typename Tout>
void launch_rows_c2r(const FftPlan& p, const cplx<T>* in, int64_t ldi, Tout* out, int64_t ldo,
                     hipStream_t s, int64_t nrows, int nsel, int off, int64_t grp) {
  const size_t cs = sizeof(cplx<T>);
  if (nrows < 0) nrows = p.nrows();
  const int M = p.n[2] / 2;
  const int tr = p.tile[2];
  const cplx<T>* twM = p.tw2M.as<cplx<T>>();
  const cplx<T>* twN = p.tw2N.as<cplx<T>>();
  if (p.gen[2])
    return launch_gen_c2r<T, Tout>(*p.gen[2], in, ldi, out, ldo, nrows, grp ? grp : nrows, nsel,
                             nsel ? ((off % p.n[2]) + p.n[2]) % p.n[2] : 0, s);
  if (p.fast[2]) {
    int trc = tr;
    while (trc > 1 && (size_t)trc * row_pad_len(M) * cs > kLdsBudget) trc /= 2;
    const int offm = nsel ? ((off % (2 * M)) + 2 * M) % (2 * M) : 0;
    // The radix-8 plans (plan variants are tuned on the forward passes).
#define FC_C2R_RC_CASE(Mv)                                                                   \
  case Mv: {                                                                                 \
    dim3 g((unsigned)((nrows + trc - 1) / trc));                                             \
    hipLaunchKernelGGL((k_fft_rows_c2r_rc<T, Tout, Mv, fft_plan_of<T, Mv>()>), g,             \
                       dim3(trc * (Mv / FftCfgV<Mv, fft_plan_of<T, Mv>()>::E)),              \
                       (size_t)trc * row_pad_len(Mv) * cs, s, in, ldi, out, ldo, nrows, trc,  \
                       twM, twN, nsel, offm);                                                \
    break;                                                                                   \
  }
    switch (M) {
      FC_C2R_RC_CASE(8)
      FC_C2R_RC_CASE(16)
      FC_C2R_RC_CASE(32)
      FC_C2R_RC_CASE(64)
      FC_C2R_RC_CASE(128)
      FC_C2R_RC_CASE(192)
      FC_C2R_RC_CASE(256)
      FC_C2R_RC_CASE(384)
      FC_C2R_RC_CASE(512)
      FC_C2R_RC_CASE(768)
      FC_C2R_RC_CASE(1024)
      FC_C2R_RC_CASE(1536)
      FC_C2R_RC_CASE(2048)
    }
#undef FC_C2R_RC_CASE
  } else {
    dim3 g((unsigned)nrows);
    const int nh = p.n[2] / 2 + 1;
    hipLaunchKernelGGL((k_dft_rows_c2r<T, Tout>), g, dim3(256), (size_t)nh * cs, s, in, ldi,
                       out, ldo, p.n[2], twN, nsel, off);
  }
  FC_LAUNCH_CHECK();
}


#define FC_R2C(T, Tin, Loader, A)                                                              \
  template void launch_rows_r2c<T, Tin, Loader, A>(                                            \
      const FftPlan&, const Tin*, int64_t, cplx<T>*, int64_t, Loader, hipStream_t, int64_t,    \
      const FftPlan*, const Tin*, int64_t);
#define FC_R2C_ALL(Loader)            \
  FC_R2C(double, double, Loader, double) \
  FC_R2C(double, float, Loader, double)  \
  FC_R2C(float, double, Loader, float)   \
  FC_R2C(float, float, Loader, float)    \
  FC_R2C(float, double, Loader, double)  \
  FC_R2C(float, float, Loader, double)
FC_R2C_ALL(LoadCopy)
FC_R2C_ALL(LoadYlm)
#undef FC_R2C_ALL
#undef FC_R2C
#define FC_C2R(T, Tout)                                                                       \
  template void launch_rows_c2r<T, Tout>(const FftPlan&, const cplx<T>*, int64_t, Tout*,       \
                                         int64_t, hipStream_t, int64_t, int, int, int64_t);
FC_C2R(double, double)
FC_C2R(float, float)
FC_C2R(float, double)
#undef FC_C2R

}  // namespace fc
