// Column passes with a compile-time plan (k_fft_cols_rc, k_fft_cols_pipe) and
// the choice between them, the mixed-radix pass and the direct sums.
#include "fft_plan.h"

namespace fc {
namespace {

// Tiles of tc columns a workgroup holds (E values per thread): 16, 8 or 4
// columns within 64 KB (two workgroups per CU), 4 or fewer of the longest
// lengths within 128 KB (one workgroup of up to 16 waves, but twice the row
// segment: 16 or 32 bytes of each line are read at a time otherwise).
constexpr bool rc_tile_fits(int L, int E, int tc, size_t cs) {
  return (size_t)L * tc * cs <= (tc > 4 ? kLdsBudget : 2 * kLdsBudget) && tc * (L / E) <= 1024;
}
constexpr bool rc_tile_ok(int L, int E, int tc, size_t cs) {
  return rc_tile_fits(L, E, tc, cs) && (tc >= 4 || !rc_tile_fits(L, E, 2 * tc, cs));
}
// The widest such tile of at most tc columns (at least the narrowest).
int rc_tile(int L, int E, int tc, size_t cs) {
  int t = tc >= 16 ? 16 : tc >= 8 ? 8 : 4;
  while (t > 1 && !rc_tile_fits(L, E, t, cs)) t /= 2;
  return t;
}

template <typename T, int DIR, typename Tin, int TC, typename A, int Lv, int V>
void launch_cols_rc_v(const ColView<T, Tin>& v, int64_t nb, int tilesB, int nout, int offm,
                      const cplx<A>* tw, hipStream_t s) {
  hipLaunchKernelGGL((k_fft_cols_rc<A, Lv, DIR, TC, Tin, T, V>), dim3((unsigned)nb),
                     dim3(TC * (Lv / FftCfgV<Lv, V>::E)),
                     (size_t)Lv * TC * sizeof(cplx<T>) <= kLdsBudget
                         ? (size_t)Lv * TC * sizeof(cplx<T>)
                         : 0,
                     s,
                     v.in, v.inA, v.inL, v.inG, v.out, v.outA, v.outL, v.outG, v.B, tilesB, v.G,
                     nout, offm, tw);
}

// Whether k_fft_cols_pipe takes a column view: one group per slab, all L
// outputs in order, each tile's 128-byte row segments inside the row pitch
// (the rows of the work-grid layouts are allocated at full pitch), and its
// 32-bit in-tile offsets in range.
template <typename T, typename Tin>
bool pipe_view_ok(const ColView<T, Tin>& v, int L, int tc, int nout, int offm) {
  const uint64_t cs = sizeof(cplx<T>);
  return std::is_same<T, Tin>::value && v.G == 1 && nout == L && offm == 0 &&
         (int64_t)((v.B + tc - 1) / tc) * tc <= v.inL && (uint64_t)v.inL * cs * 8 < (1ull << 32) &&
         (uint64_t)v.outL * cs * 64 < (1ull << 32);
}

// The persistent prefetching column pass (k_fft_cols_pipe): one workgroup
// per CU (its two tiles and the twiddles take most of the CU's LDS).
template <typename T, int DIR, int TC, typename A, int Lv>
void launch_cols_pipe(const ColView<T, T>& v, int tilesB, int64_t nb, const cplx<A>* tw,
                      hipStream_t s) {
  static_assert(2 * pipe_lds_bytes<Lv, TC, T>() > 80 * 1024, "one workgroup per CU");
  const int grid = (int)std::min<int64_t>(nb, current_device_cus());
  hipLaunchKernelGGL((k_fft_cols_pipe<A, Lv, DIR, TC, T>), dim3((unsigned)grid),
                     dim3(TC * (Lv / 8)), 0, s, v.in, v.inA, v.inL, v.out, v.outA, v.outL, v.B,
                     tilesB, (int)nb, tw);
}

// Register-chained column pass with plan variant var: arithmetic in A
// (twiddles tw in A), loads Tin, LDS and stores in T.  Full 512-point passes
// over FP32 storage (16-column tiles, plan variant 0) run as k_fft_cols_pipe;
// with FP64 storage its 8-column tiles leave one 8-wave workgroup per CU,
// which measured no faster than two workgroups of the plain pass.
template <typename T, int DIR, typename Tin, int TC, typename A = T>
void launch_cols_rc(int L, const ColView<T, Tin>& v, const cplx<A>* tw, hipStream_t s,
                    int var = 0) {
  const int nout = v.nout ? v.nout : L;
  const int offm = ((v.off % L) + L) % L;
  const int tilesB = (v.B + TC - 1) / TC;
  const int64_t nb = (int64_t)v.A * v.G * tilesB;
  if (nb > INT32_MAX) fail(FC_ERR_INVALID, "transform too large for one launch");
  if constexpr (std::is_same<T, Tin>::value && std::is_same<T, float>::value &&
                TC * sizeof(cplx<T>) == 128) {
    if (L == 512 && var == 0 && pipe_view_ok(v, L, TC, nout, offm)) {
      launch_cols_pipe<T, DIR, TC, A, 512>(v, tilesB, nb, tw, s);
      FC_LAUNCH_CHECK();
      return;
    }
  }
#define FC_COLS_RC_LEN(Lv)                                                               \
  case Lv:                                                                               \
    if constexpr (rc_tile_ok(Lv, FftCfgV<Lv, fft_plan_of<A, Lv>()>::E, TC,               \
                             sizeof(cplx<T>))) {                                         \
      if constexpr (FftCfgV<Lv, 1>::fast) {                                              \
        if (var == 1) {                                                                  \
          launch_cols_rc_v<T, DIR, Tin, TC, A, Lv, 1>(v, nb, tilesB, nout, offm, tw, s); \
          break;                                                                         \
        }                                                                                \
      }                                                                                  \
      launch_cols_rc_v<T, DIR, Tin, TC, A, Lv, fft_plan_of<A, Lv>()>(v, nb, tilesB, nout, \
                                                                     offm, tw, s);       \
      break;                                                                             \
    }                                                                                    \
    fail(FC_ERR_RUNTIME, "internal: no such tile");
  switch (L) {
    FC_COLS_RC_LEN(8)
    FC_COLS_RC_LEN(16)
    FC_COLS_RC_LEN(32)
    FC_COLS_RC_LEN(64)
    FC_COLS_RC_LEN(128)
    FC_COLS_RC_LEN(192)
    FC_COLS_RC_LEN(256)
    FC_COLS_RC_LEN(384)
    FC_COLS_RC_LEN(512)
    FC_COLS_RC_LEN(768)
    FC_COLS_RC_LEN(1024)
    FC_COLS_RC_LEN(1536)
    FC_COLS_RC_LEN(2048)
    FC_COLS_RC_LEN(3072)
    FC_COLS_RC_LEN(4096)
    default:
      fail(FC_ERR_RUNTIME, "internal: no register-chained column kernel for this length");
  }
#undef FC_COLS_RC_LEN
  FC_LAUNCH_CHECK();
}

// Runs the register-chained pass if it takes the view.
template <typename T, int DIR, typename Tin, typename A>
bool try_cols_rc(int L, const ColView<T, Tin>& v, int tc, const cplx<A>* tw, hipStream_t s,
                 int var) {
  if (!rc_len_ok(L)) return false;
  const int E = sizeof(A) == 4 && L % 3 == 0 ? 24 : fft_len_e(L);  // fft_plan_of
  const int t = rc_tile(L, E, tc, sizeof(cplx<T>));
  if (!rc_offsets_fit<T, Tin>(L, t, v.inL, v.outL, v.nout ? v.nout : L)) return false;
  const int vr = fft_var_ok(L, var) ? var : 0;
  switch (t) {
    case 16:
      launch_cols_rc<T, DIR, Tin, 16, A>(L, v, tw, s, vr);
      break;
    case 8:
      launch_cols_rc<T, DIR, Tin, 8, A>(L, v, tw, s, vr);
      break;
    case 4:
      launch_cols_rc<T, DIR, Tin, 4, A>(L, v, tw, s, vr);
      break;
    case 2:
      launch_cols_rc<T, DIR, Tin, 2, A>(L, v, tw, s, vr);
      break;
    default:
      launch_cols_rc<T, DIR, Tin, 1, A>(L, v, tw, s, vr);
  }
  return true;
}

}  // namespace

template <typename T, int DIR, typename Tin>
void launch_cols(int L, const ColView<T, Tin>& v, int tc, const cplx<T>* tw, hipStream_t s,
                 const GenAxis* gen, int var) {
  if (try_cols_rc<T, DIR, Tin, T>(L, v, tc, tw, s, var)) return;
  const int nout = v.nout ? v.nout : L;
  if (gen) {
    const GenCols gc{v.inA, v.inL, v.inG, v.outA, v.outL, v.outG,
                     v.A,   v.G,   v.B,   nout,   ((v.off % L) + L) % L};
    return launch_gen_cols<Tin, T>(*gen, v.in, v.out, gc, DIR, s);
  }
  dim3 g((unsigned)(v.G * v.B), v.A);
  hipLaunchKernelGGL((k_dft_cols<T, DIR, Tin>), g, dim3(256), (size_t)L * sizeof(cplx<T>), s,
                     v.in, v.inA, v.inL, v.inG, v.out, v.outA, v.outL, v.outG, v.B, L, nout,
                     v.off, tw);
  FC_LAUNCH_CHECK();
}

template <typename T, int DIR, typename A>
void launch_cols_wide(int L, const ColView<T>& v, int tc, const cplx<A>* tw_a,
                      const cplx<T>* tw_t, hipStream_t s, const GenAxis* gen, int var) {
  if constexpr (!std::is_same<T, A>::value)
    if (try_cols_rc<T, DIR, T, A>(L, v, tc, tw_a, s, var)) return;
  launch_cols<T, DIR>(L, v, tc, tw_t, s, gen, var);
}

#define FC_COLS(T, DIR, Tin)                                                                    \
  template void launch_cols<T, DIR, Tin>(int, const ColView<T, Tin>&, int, const cplx<T>*,       \
                                         hipStream_t, const GenAxis*, int);
FC_COLS(double, -1, double)
FC_COLS(double, 1, double)
FC_COLS(float, -1, float)
FC_COLS(float, 1, float)
FC_COLS(double, 1, float)
#undef FC_COLS
#define FC_COLS_WIDE(T, A)                                                                      \
  template void launch_cols_wide<T, -1, A>(int, const ColView<T>&, int, const cplx<A>*,          \
                                           const cplx<T>*, hipStream_t, const GenAxis*, int);
FC_COLS_WIDE(double, double)
FC_COLS_WIDE(float, float)
FC_COLS_WIDE(float, double)
#undef FC_COLS_WIDE

}  // namespace fc
