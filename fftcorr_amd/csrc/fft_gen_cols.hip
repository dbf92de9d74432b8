// Mixed-radix column passes (fft_gen.h) and the host tables of a length.
#include <complex>
#include <mutex>

#include "fft_gen_kernels.h"

namespace fc {
namespace {

// Tile of tc adjacent columns; block (tc, tcol).
// Reads the whole tile in the first stage and writes it in the last one, so
// in and out may be the same array.  CL: the tile's values (the storage type;
// FP64 for a chirp convolution, whose intermediate values are larger).
// sgn: +1 forward, -1 inverse (conjugated in and out).
template <typename Tin, typename Tout, bool BLUE, int RM>
__global__ void __launch_bounds__(gen_max_threads<RM>())
    k_gen_cols(const cplx<Tin>* in, cplx<Tout>* out, GenCols v, int tilesB, double sgn,
               GenDev g) {
  using CL = cplx<typename std::conditional<BLUE, double, Tout>::type>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  CL* lds = reinterpret_cast<CL*>(smem_raw);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ag = tile / tilesB;
  const int b0 = (tile - ag * tilesB) * (int)blockDim.x;
  const int a = ag / v.G, gr = ag - a * v.G;
  const int c = threadIdx.x, j = threadIdx.y;
  const bool colok = b0 + c < v.B;
  // Columns past B read column b0 (discarded).
  const cplx<Tin>* src =
      in + (int64_t)a * v.inA + (int64_t)gr * v.inG + b0 + (colok ? c : 0) + (int64_t)j * v.inL;
  cplx<Tout>* dst = out + (int64_t)a * v.outA + (int64_t)gr * v.outG + b0 + c;
  cplx<Tout>* dstj = dst + (int64_t)j * v.outL;
  const bool whole = v.nout == g.L && v.offm == 0;
  // The elements come in order of r: running pointers, one 64-bit add each.
  const cplx<Tin>* sp = src;
  auto load = [&](int r, int u) {
    if (r > 0) sp += (int64_t)u * v.inL;
    const cplx<Tin> x = ld_stream(sp);
    return double2{(double)x.x, sgn * (double)x.y};
  };
  auto store = [&](int r, int u, double2 x) {
    if (!colok) return;
    const cplx<Tout> y{Tout(x.x), Tout(sgn * x.y)};
    if (whole) {
      if (r > 0) dstj += (int64_t)u * v.outL;
      st_stream(dstj, y);
      return;
    }
    int o = j + r * u + v.offm;
    if (o >= g.L) o -= g.L;
    for (; o < v.nout; o += g.L) st_stream(dst + (int64_t)o * v.outL, y);
  };
  const LayGenCol lay{blockDim.x};
  if constexpr (BLUE)
    gen_run_blue<RM>(lds, g.stg, g.ns, g.W, g.chirp, g.filt, g.L, c, j, lay, load, store, false);
  else
    gen_run<RM, 0>(lds, g.stg, g.ns, g.W, c, j, lay, load, NoMid{}, store, false);
}

}  // namespace

template <typename Tin, typename Tout>
void launch_gen_cols(const GenAxis& ax, const cplx<Tin>* in, cplx<Tout>* out, const GenCols& v,
                     int dir, hipStream_t s) {
  const size_t cl = ax.blue ? sizeof(double2) : sizeof(cplx<Tout>);
  const int tc = gen_col_tile(ax, cl, sizeof(cplx<Tout>), gen_axis_threads(ax));
  const int tilesB = (v.B + tc - 1) / tc;
  const int64_t nb = (int64_t)v.A * v.G * tilesB;
  if (nb > INT32_MAX) fail(FC_ERR_INVALID, "transform too large for one launch");
  if (nb == 0) return;
  const dim3 blk((unsigned)tc, (unsigned)ax.tcol);
  const size_t lds = (size_t)ax.N * tc * cl;
  const double sgn = dir < 0 ? 1.0 : -1.0;
  auto go = [&](auto blue, auto rm) {
    hipLaunchKernelGGL((k_gen_cols<Tin, Tout, decltype(blue)::value, decltype(rm)::value>),
                       dim3((unsigned)nb), blk, lds, s, in, out, v, tilesB, sgn, gen_dev(ax));
  };
  gen_dispatch(ax, go);
  FC_LAUNCH_CHECK();
}

template void launch_gen_cols<float, float>(const GenAxis&, const float2*, float2*,
                                            const GenCols&, int, hipStream_t);
template void launch_gen_cols<double, double>(const GenAxis&, const double2*, double2*,
                                              const GenCols&, int, hipStream_t);
template void launch_gen_cols<float, double>(const GenAxis&, const float2*, double2*,
                                             const GenCols&, int, hipStream_t);

// ---- host tables ------------------------------------------------------------
namespace {

constexpr int kGenRadices[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 15, 16};

// All nondecreasing factorisations of n into the radices, each compared with
// the best so far.
void search_radices(int n, int from, std::vector<int>& cur, std::vector<int>& best) {
  if (n == 1) {
    auto better = [](const std::vector<int>& a, const std::vector<int>& b) {
      if (a.size() != b.size()) return a.size() < b.size();
      if (a.front() != b.front()) return a.front() > b.front();
      return a.back() < b.back();
    };
    if (best.empty() || better(cur, best)) best = cur;
    return;
  }
  if (!best.empty() && cur.size() >= best.size()) return;
  for (int i = from; i < (int)(sizeof(kGenRadices) / sizeof(int)); ++i) {
    const int r = kGenRadices[i];
    if (r > n) break;
    if (n % r) continue;
    cur.push_back(r);
    search_radices(n / r, i, cur, best);
    cur.pop_back();
  }
}

// exp(-2 pi i m / N) in long double, reduced to the first octant's accuracy by
// exact integer reduction of m.
std::complex<long double> root(int64_t m, int64_t N) {
  m %= N;
  const long double a = 2.0L * 3.141592653589793238462643383279502884L * (long double)m / N;
  return {cosl(a), -sinl(a)};
}

// Plain recursive mixed-radix transform of the filter (host, once per length).
void host_fft(const std::complex<long double>* x, int64_t stride, int n,
              std::complex<long double>* out, const std::vector<std::complex<long double>>& w,
              int64_t wstride) {
  if (n == 1) {
    out[0] = x[0];
    return;
  }
  int p = 2;
  while (n % p) ++p;
  const int m = n / p;
  std::vector<std::complex<long double>> sub((size_t)n);
  for (int q = 0; q < p; ++q)
    host_fft(x + q * stride, stride * p, m, sub.data() + (size_t)q * m, w, wstride * p);
  const int64_t N = (int64_t)w.size();
  for (int k = 0; k < n; ++k) {
    std::complex<long double> s = 0;
    for (int q = 0; q < p; ++q) s += sub[(size_t)q * m + k % m] * w[((int64_t)q * k * wstride) % N];
    out[k] = s;
  }
}

template <typename V>
void put(DeviceBuffer& d, const std::vector<V>& h) {
  d.allocate(sizeof(V) * h.size());
  FC_HIP(hipMemcpy(d.as<void>(), h.data(), sizeof(V) * h.size(), hipMemcpyHostToDevice));
}

void add_stages(std::vector<GenStage>& st, const std::vector<int>& rad, int N, size_t from) {
  int NS = 1;
  for (size_t i = 0; i < rad.size(); ++i) {
    const FastDiv f((uint32_t)NS);
    if (i >= from)
      st.push_back(GenStage{rad[i], N / rad[i], NS, N / (NS * rad[i]), f.m, f.s, 0, 0});
    NS *= rad[i];
  }
}

}  // namespace

std::vector<int> gen_radices(int L) {
  std::vector<int> cur, best;
  if (L == 1) return {1};
  if (L >= 1 && L <= kGenMaxLen) search_radices(L, 0, cur, best);
  // A column's threads have to fit one workgroup (2 * 11^3 does not).
  if (!best.empty() &&
      L / best.front() > (best.back() <= kGenRadSmall ? gen_max_threads<kGenRadSmall>()
                                                      : gen_max_threads<16>()))
    best.clear();
  return best;
}

bool gen_len_ok(int L) {
  return L >= 1 && L <= kGenMaxLen && (L <= kGenMaxBlue || !gen_radices(L).empty());
}

GenAxis gen_axis_stages(int L) {
  GenAxis ax;
  if (!gen_len_ok(L)) return ax;
  ax.L = L;
  ax.radices = gen_radices(L);
  int N = L;
  if (ax.radices.empty()) {
    // The convolution length: among the lengths in [2 L - 1, 1.25 (2 L - 1)],
    // fewest stages, then shortest.
    ax.blue = true;
    for (int n = 2 * L - 1; n <= kGenMaxLen && n <= (2 * L - 1) * 5 / 4 + 1; ++n) {
      std::vector<int> r = gen_radices(n);
      if (r.empty()) continue;
      if (ax.radices.empty() || r.size() < ax.radices.size()) {
        ax.radices = r;
        N = n;
      }
    }
    if (ax.radices.empty()) return ax;
  }
  ax.N = N;
  ax.ns = (int)ax.radices.size();
  for (int r : ax.radices) {
    ax.tcol = std::max(ax.tcol, ax.N / r);
    ax.rmax = std::max(ax.rmax, r);
  }
  return ax;
}

std::shared_ptr<GenAxis> make_gen_axis(int L) {
  auto ax = std::make_shared<GenAxis>(gen_axis_stages(L));
  if (ax->N == 0) return nullptr;
  std::vector<GenStage> st;
  add_stages(st, ax->radices, ax->N, 0);
  std::vector<int> rev(ax->radices.rbegin(), ax->radices.rend());
  add_stages(st, rev, ax->N, 1);
  put(ax->stages, st);
  const int N = ax->N;
  std::vector<std::complex<long double>> w(N);
  std::vector<double2> hw(N);
  for (int m = 0; m < N; ++m) {
    w[m] = root(m, N);
    hw[m] = make_double2((double)w[m].real(), (double)w[m].imag());
  }
  put(ax->W, hw);
  if (ax->blue) {
    // chirp[e] = exp(-i pi e^2 / L) with e^2 reduced mod 2 L.
    std::vector<double2> ch(L), hf(N);
    std::vector<std::complex<long double>> f(N, 0), F(N);
    for (int e = 0; e < L; ++e) {
      const std::complex<long double> b = root((int64_t)e * e, 2 * (int64_t)L);
      ch[e] = make_double2((double)b.real(), (double)b.imag());
      f[e] = std::conj(b);
      if (e) f[N - e] = std::conj(b);
    }
    host_fft(f.data(), 1, N, F.data(), w, 1);
    for (int m = 0; m < N; ++m)
      hf[m] = make_double2((double)(F[m].real() / N), (double)(F[m].imag() / N));
    put(ax->chirp, ch);
    put(ax->filt, hf);
  }
  return ax;
}

}  // namespace fc
