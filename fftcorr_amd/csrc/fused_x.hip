// Launches of the fused x pass with a compile-time plan (fused_x.h).
#include "fused_x.h"

#include <type_traits>

#include "fft_plan.h"

namespace fc {

template <typename T, typename TI, int MODE>
bool launch_px_rc(int n0, const PxArgs<T>& p, const cplx<T>* tw, const cplx<TI>* twi,
                  hipStream_t s) {
  // The kernel addresses pk and q with 32-bit byte offsets, the spectra with 32
  // bits while one is below 4 GB.
  const uint64_t lim = 0xffffffffull;
  const uint64_t q1 = (uint64_t)p.rs * p.n1 * p.ldq * sizeof(cplx<TI>);
  const uint64_t npk = (uint64_t)p.ks.ks0 * p.ks.ks1 * (p.ks.ks2 / 2 + 1) * 8;
  const uint64_t spec = (uint64_t)n0 * p.n1 * p.ldc * sizeof(cplx<T>);
  if (!px_len_ok(n0) || q1 > lim || npk > lim) return false;
  if constexpr (std::is_same<T, float>::value && MODE == kModeCross) {
    // Cross mode, 512-point x over FP32 spectra, one correlation: the
    // persistent prefetching form, when each tile's 64-byte row segments lie
    // inside the row pitch and its in-tile offsets fit 32 bits.
    constexpr int TC = px_tc<T, TI, 512, MODE>();
    const int tilesC = (p.n2h + TC - 1) / TC;
    const int64_t ntiles = (int64_t)p.n1 * tilesC;
    const uint64_t pitch = (uint64_t)p.n1 * p.ldc * sizeof(cplx<T>);
    if (n0 == 512 && p.nb == 1 && (int64_t)tilesC * TC <= p.ldc && pitch * 16 < (1ull << 32) &&
        ntiles <= INT32_MAX) {
      const int grid = (int)std::min<int64_t>(ntiles, current_device_cus());
      hipLaunchKernelGGL((k_periodic_x2_cross_pipe<TI, 512>), dim3((unsigned)grid),
                         dim3(px_threads<T, TI, 512, MODE>()), 0, s, p.A, p.B, p.n1, p.n2h, p.ldc,
                         tilesC, tw, twi, p.pk, p.ks, static_cast<cplx<TI>*>(p.q), p.ldq, p.rs,
                         p.offm, (int)ntiles);
      FC_LAUNCH_CHECK();
      return true;
    }
  }
  auto go = [&](auto ltag, auto off) {
    constexpr int L = decltype(ltag)::value;
    using Off = decltype(off);
    // Two grids' columns of 4096 FP64 values do not fit: separate passes.
    if constexpr (px_lds_bytes<T, TI, L, MODE>() <= 65536) {
    constexpr int TC = px_tc<T, TI, L, MODE>();
    const int tilesC = (p.n2h + TC - 1) / TC;
    const int64_t per = (int64_t)p.n1 * tilesC;
    const int64_t nblocks = per * p.nb;
    if (nblocks > INT32_MAX) fail(FC_ERR_INVALID, "grid too large for the fused x pass");
    hipLaunchKernelGGL((k_periodic_x2<T, TI, L, MODE, Off>), dim3((unsigned)nblocks),
                       dim3(px_threads<T, TI, L, MODE>()), (px_lds_bytes<T, TI, L, MODE>()), s,
                       p.A, p.B, p.n1, p.n2h, p.ldc, tilesC, tw, twi, p.ph0, p.ph1, p.ph2, p.pk,
                       p.ks, static_cast<cplx<TI>*>(p.q), p.ldq, p.rs, p.offm, (int)per,
                       p.a_bstride, p.pk_bstride, p.q_bstride);
    return true;
    } else {
      return false;
    }
  };
#define FC_PX2_CASE(Lv)                                        \
  case Lv:                                                     \
    if (!go(std::integral_constant<int, Lv>{}, uint32_t(0))) return false; \
    break;
#define FC_PX2_WIDE(Lv)                                        \
  case Lv:                                                     \
    if (!go(std::integral_constant<int, Lv>{}, uint64_t(0))) return false; \
    break;
  if (spec <= lim) {
    switch (n0) {
      FC_PX2_CASE(8)
      FC_PX2_CASE(16)
      FC_PX2_CASE(32)
      FC_PX2_CASE(64)
      FC_PX2_CASE(128)
      FC_PX2_CASE(192)
      FC_PX2_CASE(256)
      FC_PX2_CASE(384)
      FC_PX2_CASE(512)
      FC_PX2_CASE(768)
      FC_PX2_CASE(1024)
      FC_PX2_CASE(1536)
      FC_PX2_CASE(2048)
      FC_PX2_CASE(3072)
      FC_PX2_CASE(4096)
      default:
        return false;
    }
  } else {
    switch (n0) {
      FC_PX2_WIDE(512)
      FC_PX2_WIDE(768)
      FC_PX2_WIDE(1024)
      default:
        return false;
    }
  }
#undef FC_PX2_CASE
#undef FC_PX2_WIDE
  FC_LAUNCH_CHECK();
  return true;
}

#define FC_PX_RC(T, TI, MODE)                                                              \
  template bool launch_px_rc<T, TI, MODE>(int, const PxArgs<T>&, const cplx<T>*,            \
                                          const cplx<TI>*, hipStream_t);
#define FC_PX_RC_ALL(T, TI)         \
  FC_PX_RC(T, TI, kModeAuto)        \
  FC_PX_RC(T, TI, kModeCross)       \
  FC_PX_RC(T, TI, kModeInterlaced)
FC_PX_RC_ALL(double, double)
FC_PX_RC_ALL(float, float)
FC_PX_RC_ALL(float, double)
#undef FC_PX_RC_ALL
#undef FC_PX_RC

}  // namespace fc
