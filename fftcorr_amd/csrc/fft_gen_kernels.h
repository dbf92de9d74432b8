// Device side of the mixed-radix passes (fft_gen.h): FP64 butterflies of
// radix 2 .. 16 and the stage loop.
//
// A workgroup owns a tile of columns (or rows); thread (c, j) runs butterfly j
// of column c in every stage, so a stage holds one butterfly (R values) in
// registers and a length L needs max(L / R) threads per column.  The first
// stage reads global memory and the last one's outputs leave from registers;
// in between the tile sits in LDS once (each stage reads, synchronises,
// writes back).  The radix is a wave-uniform switch: the cost of an integer
// plan instead of a compile-time one is a scalar branch per stage, an integer
// division by multiplication per thread and the idle lanes of the stages with
// fewer butterflies than threads.  400^3 in FP64, against the direct O(L^2)
// sums these lengths ran before: rows 12.3 -> 0.24 ms (1.03 GB, 4.4 TB/s),
// y columns 12.2 -> 0.31 ms (1.03 GB, 3.3 TB/s), fused x pass (was separate
// passes, 14 ms) 0.36 ms (0.65 GB), bound by VALU issue (about 0.17 ms) that
// overlaps the loads only as far as 128 registers (16 waves a CU) allow.
#pragma once

#include "fft_gen.h"
#include "hist_device.h"

namespace fc {

// ---- FP64 butterflies, sign -1 (inverse transforms conjugate in and out) ----
template <int P>
struct OddRoots;
template <>
struct OddRoots<5> {
  static constexpr double c[2] = {0.30901699437494742408, -0.8090169943749474241};
  static constexpr double s[2] = {0.9510565162951535721, 0.58778525229247312913};
};
template <>
struct OddRoots<7> {
  static constexpr double c[3] = {0.6234898018587335305, -0.22252093395631440434,
                                  -0.9009688679024191263};
  static constexpr double s[3] = {0.78183148246802980873, 0.974927912181823607,
                                  0.4338837391175581203};
};
template <>
struct OddRoots<11> {
  static constexpr double c[5] = {0.84125353283118116886, 0.4154150130018864255,
                                  -0.14231483827328514046, -0.6548607339452850641,
                                  -0.9594929736144973899};
  static constexpr double s[5] = {0.5406408174555975821, 0.9096319953545183714,
                                  0.98982144188093273236, 0.7557495743542582837,
                                  0.28173255684142969765};
};
template <>
struct OddRoots<13> {
  static constexpr double c[6] = {0.88545602565320989587, 0.5680647467311558025,
                                  0.12053668025532305325, -0.354604887042535626,
                                  -0.7485107481711010987, -0.9709418174260520272};
  static constexpr double s[6] = {0.46472317204376854566, 0.8229838658936563946,
                                  0.99270887409805399284, 0.93501624268541482345,
                                  0.6631226582407952023, 0.23931566428755776695};
};

template <int R>
struct GBfly;

// Powers of two and 3: the butterflies of the compile-time plans.
template <>
struct GBfly<2> {
  static __host__ __device__ __forceinline__ void run(double2* v) { Bfly<2, -1, double>::run(v); }
};
template <>
struct GBfly<3> {
  static __host__ __device__ __forceinline__ void run(double2* v) { Bfly<3, -1, double>::run(v); }
};
template <>
struct GBfly<4> {
  static __host__ __device__ __forceinline__ void run(double2* v) { Bfly<4, -1, double>::run(v); }
};
template <>
struct GBfly<8> {
  static __host__ __device__ __forceinline__ void run(double2* v) { Bfly<8, -1, double>::run(v); }
};
template <>
struct GBfly<16> {
  static __host__ __device__ __forceinline__ void run(double2* v) { Bfly<16, -1, double>::run(v); }
};

// Odd primes by the pair sums a_k = x_k + x_(P-k), b_k = x_k - x_(P-k):
// X_m, X_(P-m) = x_0 + sum a_k cos(2 pi m k / P) -+ i sum b_k sin(2 pi m k / P).
template <int P>
struct GBflyOdd {
  static __host__ __device__ __forceinline__ void run(double2* v) {
    constexpr int H = (P - 1) / 2;
    double2 a[H], b[H];
    double2 sum = v[0];
#pragma unroll
    for (int k = 0; k < H; ++k) {
      a[k] = cadd(v[k + 1], v[P - 1 - k]);
      b[k] = csub(v[k + 1], v[P - 1 - k]);
      sum = cadd(sum, a[k]);
    }
    const double2 x0 = v[0];
    v[0] = sum;
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      double2 u = x0, w = double2{0.0, 0.0};
#pragma unroll
      for (int k = 1; k <= H; ++k) {
        const int q = (m * k) % P;
        const double c = q <= H ? OddRoots<P>::c[q - 1] : OddRoots<P>::c[P - q - 1];
        const double s = q <= H ? OddRoots<P>::s[q - 1] : -OddRoots<P>::s[P - q - 1];
        u.x += c * a[k - 1].x;
        u.y += c * a[k - 1].y;
        w.x += s * b[k - 1].x;
        w.y += s * b[k - 1].y;
      }
      v[m] = double2{u.x + w.y, u.y - w.x};
      v[P - m] = double2{u.x - w.y, u.y + w.x};
    }
  }
};
template <>
struct GBfly<5> : GBflyOdd<5> {};
template <>
struct GBfly<7> : GBflyOdd<7> {};
template <>
struct GBfly<11> : GBflyOdd<11> {};
template <>
struct GBfly<13> : GBflyOdd<13> {};

// Coprime products A B without inner twiddles (Good 1958): input
// n = (B n1 + A n2) mod R, output k with k = k1 mod A and k = k2 mod B.
template <int A, int B>
struct GBflyPrime {
  static __host__ __device__ constexpr int crt(int k1, int k2) {
    for (int k = 0; k < A * B; ++k)
      if (k % A == k1 && k % B == k2) return k;
    return 0;
  }
  static __host__ __device__ __forceinline__ void run(double2* v) {
    double2 t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
      GBfly<A>::run(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      double2 u[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) u[n2] = t[n2][k1];
      GBfly<B>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[crt(k1, k2)] = u[k2];
    }
  }
};
template <>
struct GBfly<6> : GBflyPrime<2, 3> {};
template <>
struct GBfly<10> : GBflyPrime<2, 5> {};
template <>
struct GBfly<12> : GBflyPrime<4, 3> {};
template <>
struct GBfly<15> : GBflyPrime<3, 5> {};

// 9 = 3 x 3 with the inner twiddles W9^(n2 k1).
template <>
struct GBfly<9> {
  static __host__ __device__ __forceinline__ void run(double2* v) {
    constexpr double c1 = 0.7660444431189780352, s1 = 0.6427876096865393263;
    constexpr double c2 = 0.1736481776669303488, s2 = 0.9848077530122080594;
    constexpr double c4 = -0.9396926207859083841, s4 = 0.34202014332566873297;
    double2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 3; ++n1) t[n2][n1] = v[3 * n1 + n2];
      GBfly<3>::run(t[n2]);
    }
    t[1][1] = cmul(t[1][1], double2{c1, -s1});
    t[1][2] = cmul(t[1][2], double2{c2, -s2});
    t[2][1] = cmul(t[2][1], double2{c2, -s2});
    t[2][2] = cmul(t[2][2], double2{c4, -s4});
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      double2 u[3] = {t[0][k1], t[1][k1], t[2][k1]};
      GBfly<3>::run(u);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = u[k2];
    }
  }
};

// v[r] *= w^r (powers by halving: error ~ log2 R roundings of FP64).
template <int R>
__host__ __device__ __forceinline__ void gen_twiddle(double2* v, double2 w) {
  double2 p[R];
  p[1] = w;
#pragma unroll
  for (int r = 2; r < R; ++r) p[r] = cmul(p[r / 2], p[r - r / 2]);
#pragma unroll
  for (int r = 1; r < R; ++r) v[r] = cmul(v[r], p[r]);
}

__host__ __device__ __forceinline__ double2 cconj(double2 a) { return double2{a.x, -a.y}; }

// ---- the stage loop ---------------------------------------------------------
// lds: the tile, element e of column c at lay(c, e), values of type CL.
// MODE 0: one transform; src(r, u) gives input j + r u, sink(r, u, v) takes
// output j + r u (r a compile-time constant after unrolling, u wave-uniform, so
// a caller's address is a per-thread base plus a scalar).
// MODE 1: a transform, then w = mid(r, u, v) on every output j + r u, then a
// second transform of w with the radices reversed; sink takes its outputs.
// Both transforms have sign -1.
// bar_sink: the caller's sink writes the tile, so the last stage's reads are
// fenced from it.  RM: the largest radix the kernel has code for (kGenRadSmall
// or 16): the registers of radix 11 .. 16 are not held by plans without them.
// Every thread of the workgroup calls this; those with j >= nb only take part
// in the barriers.
template <int RM, int MODE, class CL, class Lay, class Src, class Mid, class Sink>
__device__ __forceinline__ void gen_run(CL* lds, const GenStage* __restrict__ stg, int ns,
                                        const double2* __restrict__ W, int c, int j, Lay lay,
                                        Src src, Mid mid, Sink sink, bool bar_sink) {
  using TL = typename ScalarOf<CL>::type;
  const int total = MODE == 1 ? 2 * ns - 1 : ns;
  // The next stage's descriptor (scalar loads) and this thread's twiddle of it
  // are fetched while the current stage runs: without that each stage began
  // with two dependent memory latencies (400-point rows: 306 -> 258 us).
  GenStage st = stg[0];
  int k = 0, q = j;  // j mod NS and j / NS (NS = 1 in the first stage)
  double2 w = double2{1.0, 0.0};
  for (int s = 0; s < total; ++s) {
    const bool act = j < st.nb;
    const bool first = s == 0, last = s == total - 1;
    const GenStage nx = stg[last ? s : s + 1];
    int kn = 0, qn = 0;
    double2 wn = double2{1.0, 0.0};
    auto prefetch = [&] {
      // j / NS and j mod NS of the next stage.
      qn = (int)(uint32_t)(((uint64_t)__umulhi((uint32_t)j, nx.dm) + (uint32_t)j) >> nx.ds);
      kn = j - qn * nx.NS;
      wn = W[j < nx.nb ? kn * nx.tws : 0];
    };
    auto stage = [&](auto tag) {
      constexpr int R = decltype(tag)::value;
      double2 v[R];
      // A transform's last stage has NS R = N, so its outputs are j + r NS
      // (and a single stage's, where j = 0, r).
      int base = q * st.NS * R + k, step = st.NS;
      if (act) {
        if (first) {
#pragma unroll
          for (int r = 0; r < R; ++r) v[r] = src(r, st.nb);
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) v[r] = to_cplx<double>(lds[lay(c, j + r * st.nb)]);
        }
      }
      if (!last) prefetch();
      if (act) {
        if (st.NS > 1) gen_twiddle<R>(v, w);
        GBfly<R>::run(v);
        if (MODE == 1 && s == ns - 1) {
#pragma unroll
          for (int r = 0; r < R; ++r) v[r] = mid(r, st.NS, v[r]);
          GBfly<R>::run(v);
          base = j * R;
          step = 1;
        }
      }
      if (!last || bar_sink) {
        if (!first) __syncthreads();
      }
      if (act) {
        if (last) {
#pragma unroll
          for (int r = 0; r < R; ++r) sink(r, step, v[r]);
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) lds[lay(c, base + r * step)] = to_cplx<TL>(v[r]);
        }
      }
      if (!last) __syncthreads();
    };
    switch (__builtin_amdgcn_readfirstlane(st.R)) {
#define FC_GEN_R(Rv)                                                   \
  case Rv:                                                             \
    if constexpr (Rv <= RM) stage(std::integral_constant<int, Rv>{});  \
    break;
      FC_GEN_R(2)
      FC_GEN_R(3)
      FC_GEN_R(4)
      FC_GEN_R(5)
      FC_GEN_R(6)
      FC_GEN_R(7)
      FC_GEN_R(8)
      FC_GEN_R(9)
      FC_GEN_R(10)
      FC_GEN_R(11)
      FC_GEN_R(12)
      FC_GEN_R(13)
      FC_GEN_R(15)
      FC_GEN_R(16)
#undef FC_GEN_R
      default:
        stage(std::integral_constant<int, 1>{});
    }
    st = nx;
    k = kn;
    q = qn;
    w = wn;
  }
}
template <>
struct GBfly<1> {
  static __host__ __device__ __forceinline__ void run(double2*) {}
};

struct NoMid {
  __device__ __forceinline__ double2 operator()(int, int, double2 v) const { return v; }
};

// Chirp convolution on top of MODE 1 (Bluestein 1970): inputs x[e] b[e] padded
// with zeros to N, transform, times filt = FFT(conj b) / N, inverse transform
// (conjugate, transform, conjugate), outputs times b[e], e < L.
template <int RM, class CL, class Lay, class Src, class Sink>
__device__ __forceinline__ void gen_run_blue(CL* lds, const GenStage* __restrict__ stg, int ns,
                                             const double2* __restrict__ W,
                                             const double2* __restrict__ chirp,
                                             const double2* __restrict__ filt, int L, int c,
                                             int j, Lay lay, Src src, Sink sink, bool bar_sink) {
  gen_run<RM, 1>(
      lds, stg, ns, W, c, j, lay,
      [&](int r, int u) {
        const int e = j + r * u;
        return e < L ? cmul(src(r, u), chirp[e]) : double2{0.0, 0.0};
      },
      [&](int r, int u, double2 v) { return cconj(cmul(v, filt[j + r * u])); },
      [&](int r, int u, double2 v) {
        const int e = j + r * u;
        if (e < L) sink(r, u, cmul(cconj(v), chirp[e]));
      },
      bar_sink);
}

// Row tile: row c of rs slots, element e at e + e / 2^sh (sh = 3: as LayRowPad).
struct LayGenRow {
  int rs, sh;
  __device__ __forceinline__ int operator()(int c, int e) const { return c * rs + e + (e >> sh); }
};
// Column tile of tc columns: element e of column c at e tc + c.
struct LayGenCol {
  uint32_t tc;
  __device__ __forceinline__ int operator()(int c, int e) const {
    return (int)(__umul24((uint32_t)e, tc) + (uint32_t)c);
  }
};

// Threads per workgroup: radices up to 10 fit 128 registers (16 waves), the
// larger ones do not.
template <int RM>
constexpr int gen_max_threads() {
  return RM <= kGenRadSmall ? 1024 : 512;
}

struct GenDev {
  const GenStage* stg;
  const double2 *W, *chirp, *filt;
  int L, N, ns;
};
inline GenDev gen_dev(const GenAxis& ax) {
  return GenDev{ax.stages.as<GenStage>(), ax.W.as<double2>(), ax.chirp.as<double2>(),
                ax.filt.as<double2>(), ax.L, ax.N, ax.ns};
}

// Largest workgroup of the kernel variant gen_dispatch picks for ax.
inline int gen_axis_threads(const GenAxis& ax) {
  return !ax.blue && ax.rmax <= kGenRadSmall ? gen_max_threads<kGenRadSmall>()
                                             : gen_max_threads<16>();
}
// How full a workgroup of `threads` leaves the CU's four SIMDs: its waves are
// dealt to them in turn, so a fifth wave doubles the load of the first SIMD
// (400-point columns, 80 threads each, fused x pass: 457 us with five waves,
// 362 with 3.75 of four; rows in pairs: 306 us with five, 236 with 3.75).
inline double gen_fill(int threads) {
  return (double)threads / (256.0 * ((threads + 255) / 256));
}

// Columns per workgroup of the column pass: 128-byte row segments (its stores
// fill whole lines: 400 points FP64, 183 us against 209 at 64 bytes and 258 at
// 96), fewer where the tile or the workgroup would be too large, more where a
// short column would leave less than two waves.
inline int gen_col_tile(const GenAxis& ax, size_t cl, size_t cs, int maxthr) {
  auto fits = [&](int tc) { return (size_t)ax.N * cl * tc <= 65536 && ax.tcol * tc <= maxthr; };
  int tc = (int)(128 / cs);
  while (tc > 1 && !fits(tc)) tc /= 2;
  while (tc < 64 && ax.tcol * tc < 128 && fits(2 * tc)) tc *= 2;
  return tc;
}

// Columns per workgroup of the fused x pass, which reads the spectra and
// writes only the pruned rows: the fullest SIMDs first, then 64-byte segments
// (narrower or unaligned ones cost part of each line), the smallest of equals.
inline int gen_px_tile(const GenAxis& ax, size_t cl, size_t cs, int maxthr) {
  int best = 1;
  double score = 0.0;
  for (int tc = 1; tc <= 64; ++tc) {
    if ((size_t)ax.N * cl * tc > 65536 || ax.tcol * tc > maxthr) break;
    const int seg = (int)(tc * cs);
    const double width = seg >= 64 ? 1.0 : seg >= 48 ? 0.9 : seg >= 32 ? 0.75 : 0.5;
    const double v = gen_fill(ax.tcol * tc) * width * (seg % 64 ? 0.95 : 1.0);
    if (v > score + 1e-9) score = v, best = tc;
  }
  return best;
}

// Row pairs per workgroup: the fullest four waves.
inline int gen_row_tile(const GenAxis& ax, size_t row_bytes) {
  int best = 1;
  double score = 0.0;
  for (int tr = 1; tr * ax.tcol <= 256 && tr * row_bytes <= 65536; ++tr)
    if (gen_fill(tr * ax.tcol) > score + 1e-9) score = gen_fill(tr * ax.tcol), best = tr;
  return best;
}

// go(blue, rm) with the kernel variant of a length's tables.
template <class F>
void gen_dispatch(const GenAxis& ax, F go) {
  using Small = std::integral_constant<int, kGenRadSmall>;
  using Big = std::integral_constant<int, 16>;
  if (ax.blue)
    go(std::true_type{}, Big{});
  else if (ax.rmax <= kGenRadSmall)
    go(std::false_type{}, Small{});
  else
    go(std::false_type{}, Big{});
}

}  // namespace fc
