// Fused x pass, mixed radix: forward transform, combine, the compact k values,
// the inverse transform and the pruned store in one kernel.  The inverse runs
// the forward plan with its radices reversed: its first stage then takes
// exactly the elements that the forward transform's last stage left in the
// thread's registers, so the power spectrum never goes through LDS.
#include "fft_gen_kernels.h"
#include "fft_gen_px.h"

namespace fc {
namespace {

// WAVES: waves per SIMD the registers are held for.  Four (128 registers) leave
// room for two workgroups of up to eight waves on a CU; free, they take 137 in
// interlaced mode and 162 in cross mode, and a CU runs one (interlaced, 500
// points FP64: 483 us, held 337).  In cross mode holding them costs spills
// that workgroups of up to four waves, of which three fit anyway, do not earn
// back (100 points FP64 41 us, held 48; 400 points, seven and a half waves, 291
// and 222).  Radices above 10 need more than 128.
template <typename T, typename TI, int MODE, int RM, int WAVES>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(WAVES)))
    k_gen_px(PxArgs<T> p, int tilesC, int tiles_per_batch, GenDev g) {
  using C = cplx<T>;
  using CI = cplx<TI>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  CI* lds = reinterpret_cast<CI*>(smem_raw);
  const int tile_all = xcd_tile(blockIdx.x, gridDim.x);
  const int bat = tile_all / tiles_per_batch;
  const int tile = tile_all - bat * tiles_per_batch;
  const int y = tile / tilesC;
  const int c0 = (tile - y * tilesC) * (int)blockDim.x;
  const int c = threadIdx.x, j = threadIdx.y;
  const int cg = c0 + c;
  const bool colok = cg < p.n2h;
  const int64_t sL = (int64_t)p.n1 * p.ldc;
  // Per-thread bases at element j; element j + r u adds the scalar r u sL.
  const int64_t base = (int64_t)y * p.ldc + (colok ? cg : c0) + (int64_t)j * sL;
  const C* A = p.A + bat * p.a_bstride + base;
  const C* B = MODE == kModeAuto ? nullptr
                                 : p.B + (MODE == kModeInterlaced ? bat * p.a_bstride : 0) + base;
  CI* q = static_cast<CI*>(p.q) + bat * p.q_bstride + (int64_t)y * p.ldq + cg;
  const int64_t sq = (int64_t)p.n1 * p.ldq;
  const int L = g.L;
  const LayGenCol lay{blockDim.x};
  // The k slots of this row and column (put_pk's rule): element e goes to x
  // slots e + ox (e <= ox) and e - L + ox (e >= L - ox).
  const int ox = p.ks.ks0 / 2, oy = p.ks.ks1 / 2, nz = p.ks.oz() + 1;
  const int sy0 = slot_a(y, oy);
  int sy1 = slot_b(y, p.n1, oy);
  if (sy1 == sy0) sy1 = -1;
  const bool keep = colok && cg < nz && (sy0 >= 0 || sy1 >= 0);
  const int64_t sp = (int64_t)p.ks.ks1 * nz;
  T* pk = p.pk + bat * p.pk_bstride + cg + (int64_t)(j + ox) * sp;
  const int64_t py0 = (int64_t)sy0 * nz, py1 = (int64_t)sy1 * nz;
  auto put = [&](int64_t off, T val) {
    if (sy0 >= 0) pk[off + py0] = val;
    if (sy1 >= 0) pk[off + py1] = val;
  };

  // Interlaced: the second grid's transform waits in LDS behind the tile, each
  // thread reading back what it wrote.
  C* ldsb = reinterpret_cast<C*>(lds + (size_t)g.N * blockDim.x);
  double2 pyc = make_double2(1.0, 0.0);
  if constexpr (MODE == kModeInterlaced) {
    gen_run<RM, 0>(
        lds, g.stg, g.ns, g.W, c, j, lay,
        [&](int r, int u) {
          if (r > 0) B += (int64_t)u * sL;
          return to_cplx<double>(*B);
        },
        NoMid{},
        [&](int r, int u, double2 v) { ldsb[lay(c, j + r * u)] = to_cplx<T>(v); }, false);
    __syncthreads();  // its last LDS reads precede the next transform's writes
    pyc = cmul(p.ph1[y], p.ph2[colok ? cg : 0]);
  }
  gen_run<RM, 1>(
      lds, g.stg, g.ns, g.W, c, j, lay,
      [&](int r, int u) {
        if (r > 0) A += (int64_t)u * sL;
        return to_cplx<double>(*A);
      },
      [&](int r, int u, double2 v) {
#pragma clang fp contract(off)
        const int e = j + r * u;
        double2 w;
        if constexpr (MODE == kModeInterlaced) {
          const double2 ph = cmul(p.ph0[e], pyc);
          const double2 fb = to_cplx<double>(ldsb[lay(c, e)]);
          const double fx = 0.5 * (v.x + (fb.x * ph.x - fb.y * ph.y));
          const double fy = 0.5 * (v.y + (fb.x * ph.y + fb.y * ph.x));
          w = double2{fx * fx + fy * fy, 0.0};
        } else if constexpr (MODE == kModeCross) {
          if (r > 0) B += (int64_t)u * sL;
          const double2 b = to_cplx<double>(*B);
          w = double2{v.x * b.x + v.y * b.y, v.y * b.x - v.x * b.y};
        } else {
          w = double2{v.x * v.x + v.y * v.y, 0.0};
        }
        if (r > 0) pk += (int64_t)u * sp;
        if (keep) {
          if (e <= ox) put(0, T(w.x));
          if (e - L + ox >= 0) put(-(int64_t)L * sp, T(w.x));
        }
        return cconj(w);
      },
      [&](int r, int u, double2 v) {
        if (!colok) return;
        int o = j + r * u + p.offm;
        if (o >= L) o -= L;
        for (; o < p.rs; o += L) st_stream(q + o * sq, to_cplx<TI>(cconj(v)));
      },
      false);
}

}  // namespace

template <typename T, typename TI, int MODE>
void launch_gen_px(const GenAxis& ax, const PxArgs<T>& p, hipStream_t s) {
  if (!gen_px_ok(ax)) fail(FC_ERR_RUNTIME, "internal: no fused x pass for this length");
  const size_t cl = sizeof(cplx<TI>) + (MODE == kModeInterlaced ? sizeof(cplx<T>) : 0);
  const int tc = gen_px_tile(ax, cl, sizeof(cplx<T>), 512);
  const int tilesC = (p.n2h + tc - 1) / tc;
  const int64_t per = (int64_t)p.n1 * tilesC;
  const int64_t nblocks = per * p.nb;
  if (nblocks > INT32_MAX) fail(FC_ERR_INVALID, "grid too large for the fused x pass");
  const dim3 blk((unsigned)tc, (unsigned)ax.tcol);
  const size_t lds = (size_t)ax.N * tc * cl;
  auto go = [&](auto rm, auto waves) {
    hipLaunchKernelGGL((k_gen_px<T, TI, MODE, decltype(rm)::value, decltype(waves)::value>),
                       dim3((unsigned)nblocks), blk, lds, s, p, tilesC, (int)per, gen_dev(ax));
  };
  using Free = std::integral_constant<int, 2>;
  using Held = std::integral_constant<int, 4>;
  using Small = std::integral_constant<int, kGenRadSmall>;
  if (ax.rmax > kGenRadSmall)
    go(std::integral_constant<int, 16>{}, Free{});
  else if (MODE == kModeCross && tc * ax.tcol <= 256)
    go(Small{}, Free{});
  else
    go(Small{}, Held{});
  FC_LAUNCH_CHECK();
}

#define FC_GEN_PX(T, TI)                                                                       \
  template void launch_gen_px<T, TI, kModeAuto>(const GenAxis&, const PxArgs<T>&, hipStream_t);  \
  template void launch_gen_px<T, TI, kModeCross>(const GenAxis&, const PxArgs<T>&, hipStream_t); \
  template void launch_gen_px<T, TI, kModeInterlaced>(const GenAxis&, const PxArgs<T>&, hipStream_t);
FC_GEN_PX(double, double)
FC_GEN_PX(float, float)
FC_GEN_PX(float, double)
#undef FC_GEN_PX

}  // namespace fc
