// Deterministic mass assignment (MassAssignor, cc/particle_mesh/mass_assignor.h:30-234
// with the NGP/TSC stencils of cc/particle_mesh/distribution_functions.h:25-160,
// plus CIC).
//
// The reference buffers particles, merge-sorts them by cell and scatters each
// particle's 27 weights into the grid slab by slab.  Here:
//   1. k_ma_prepare   grid coordinates / skip test (config_space_grid.h:31-46),
//                     the key cell (the cell holding the particle; for CIC the
//                     lower corner of its 2x2x2 block of target cells) and FP64
//                     weight sums per block;
//   2. stable radix sort of (key, particle index) (radix_sort.h: passes of
//      at most 8 bits over the bits the largest key needs): within a key
//      cell the particles keep their input order;
//   3. k_records      records (offsets from the key cell, weight) in sorted
//                     order, from the particles again;
//   4. k_row_bounds   per grid row (x, y), the sorted particles at the borders
//                     of its z tiles (binary searches);
//   5. k_ma_tile      one wave per 8 x 32 tile of target cells of an x plane:
//                     the particles of every key cell whose stencil reaches
//                     the tile, an equal share per lane, summed in registers
//                     and then in an FP64 copy of the tile in LDS; each
//                     touched grid cell is read and written once.
// (The D12 wavelet's gather finds its particles per key cell instead, by
// k_cell_runs.)
// No floating-point atomics on memory and no order that depends on
// scheduling: repeated runs give identical bits.

#include <mutex>
#include <vector>

#include "fc_objects.h"
#include "philox.h"
#include "radix_sort.h"
#include "xcd.h"

namespace fc {
namespace {

constexpr int kPrepThreads = 256;
constexpr int TY = 8, TZ = 32;  // target tile of one wave of k_ma_tile, in one x plane
constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / kWave;  // consecutive x planes of a workgroup

struct GridGeom {
  int n0, n1, n2;
  double p0, p1, p2;
  double cell;
};

__device__ __forceinline__ bool to_grid(double p, double pmin, double cell, int n, bool wrap,
                                        double* x) {
#pragma clang fp contract(off)
  double v = (p - pmin) / cell;
  const double xmax = (double)n;
  if (v < 0 || v >= xmax) {
    if (!wrap) return false;
    v = fmod(v, xmax);
    if (v < 0) v += xmax;
    // fmod(-eps, n) + n can round up to n: that is the periodic image 0.
    if (v >= xmax) v = 0.0;
  }
  *x = v;
  return true;
}

// Orders a wave's LDS accesses across its lanes (they execute in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Key cell and offset along one axis: a = floor(x - anchor), wrapped into
// [0, n), and r = (x - anchor) - floor(x - anchor) in [0, 1).  anchor is 0
// (NGP, TSC, D12: the cell holding the particle) or 1/2 (CIC: the lower of the
// two cells whose centres bracket the particle).
__device__ __forceinline__ int key_axis(double x, double anchor, int n, double* r) {
#pragma clang fp contract(off)
  const double xa = x - anchor;
  const double fa = floor(xa);
  *r = xa - fa;
  int a = (int)fa;
  if (a < 0) a += n;
  return a;
}

// Where the particles come from: an array pos [n, ncol] (ncol 3 or 4) with
// weights [n] or null, or the random generator.  Each particle is asked for
// twice, for its key and, in sorted order, for its record: cheaper than
// keeping 32 bytes per particle in input order in between.
struct ArraySource {
  const double* pos;
  int ncol;
  const double* weights;
  double w_scalar;
  __device__ __forceinline__ double4 operator()(int64_t i) const {
    const double* p = pos + i * ncol;
    return make_double4(p[0], p[1], p[2],
                        ncol == 4 ? p[3] : (weights ? weights[i] : w_scalar));
  }
};
struct UniformSource {
  double3 lo, span;
  uint64_t seed, first;
  double weight;
  __device__ __forceinline__ double4 operator()(int64_t i) const {
    const double3 p = random_uniform(lo, span, seed, first + (uint64_t)i);
    return make_double4(p.x, p.y, p.z, weight);
  }
};

// Key and record (offsets from the key cell, weight) of particle p; false if
// it is skipped.  The record's z is the position itself unless cell_z (the
// key cell along z is found from it again).
struct Locator {
  GridGeom g;
  int wrap;
  double shift, anchor;
  bool cell_z;
  __device__ __forceinline__ bool operator()(const double4& p, uint32_t* key,
                                             double4* rec) const {
#pragma clang fp contract(off)
    double x, y, z;
    if (!(to_grid(p.x, g.p0, g.cell, g.n0, wrap, &x) &&
          to_grid(p.y, g.p1, g.cell, g.n1, wrap, &y) &&
          to_grid(p.z, g.p2, g.cell, g.n2, wrap, &z)))
      return false;
    if (shift != 0.0) {  // interlaced grid: displace by `shift` cells, wrap
      x += shift;
      y += shift;
      z += shift;
      if (x >= g.n0) x -= g.n0;
      if (y >= g.n1) y -= g.n1;
      if (z >= g.n2) z -= g.n2;
    }
    double rx, ry, rz;
    const int ix = key_axis(x, anchor, g.n0, &rx);
    const int iy = key_axis(y, anchor, g.n1, &ry);
    const int iz = key_axis(z, anchor, g.n2, &rz);
    *key = (uint32_t)(((uint64_t)ix * g.n1 + iy) * g.n2 + iz);
    *rec = make_double4(rx, ry, cell_z ? rz : z - anchor, p.w);
    return true;
  }
};

// Keys (skipped particles get `sentinel`, sorted after every cell) and the
// weight sums per block.
template <class Source>
__global__ void __launch_bounds__(kPrepThreads)
    k_ma_prepare(Source src, int64_t n, Locator loc, uint32_t sentinel,
                 uint32_t* __restrict__ keys, double* __restrict__ part_w,
                 unsigned long long* __restrict__ part_n) {
#pragma clang fp contract(off)
  __shared__ double sd[kPrepThreads / kWave];
  __shared__ unsigned long long su[kPrepThreads / kWave];
  const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
  const int64_t lo = (int64_t)blockIdx.x * chunk;
  const int64_t hi = lo + chunk < n ? lo + chunk : n;
  double tw = 0.0, tw2 = 0.0;
  unsigned long long added = 0;
  for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
    const double4 p = src(i);
    uint32_t key = sentinel;
    double4 rec;
    if (loc(p, &key, &rec)) {
      tw += p.w;
      tw2 += p.w * p.w;
      added += 1;
    }
    keys[i] = key;
  }
  tw = block_sum(tw, sd);
  tw2 = block_sum(tw2, sd);
  added = block_sum_u64(added, su);
  if (threadIdx.x == 0) {
    part_w[2 * blockIdx.x] = tw;
    part_w[2 * blockIdx.x + 1] = tw2;
    part_n[blockIdx.x] = added;
  }
}

// One block of kWave threads: lane l sums partials l, l + 64, ... in order,
// then the fixed butterfly of block_sum; the result does not depend on
// scheduling.
__global__ void __launch_bounds__(kWave)
    k_ma_finish_stats(const double* __restrict__ part_w,
                      const unsigned long long* __restrict__ part_n, int nb,
                      double* __restrict__ out_w, unsigned long long* out_n) {
#pragma clang fp contract(off)
  __shared__ double sd[1];
  __shared__ unsigned long long su[1];
  double a = 0.0, b = 0.0;
  unsigned long long c = 0;
  for (int i = threadIdx.x; i < nb; i += kWave) {
    a += part_w[2 * i];
    b += part_w[2 * i + 1];
    c += part_n[i];
  }
  a = block_sum(a, sd);
  b = block_sum(b, sd);
  c = block_sum_u64(c, su);
  if (threadIdx.x == 0) {
    out_w[0] = a;
    out_w[1] = b;
    out_n[0] = c;
  }
}

// The records of the particles on the grid, in sorted order.
template <class Source>
__global__ void k_records(const uint32_t* __restrict__ order, Source src, Locator loc,
                          const unsigned long long* __restrict__ nvalid_p,
                          double4* __restrict__ out) {
  const int64_t nvalid = (int64_t)*nvalid_p;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvalid;
       i += (int64_t)gridDim.x * blockDim.x) {
    uint32_t key;
    double4 rec = make_double4(0, 0, 0, 0);
    loc(src(order[i]), &key, &rec);
    out[i] = rec;
  }
}

__global__ void k_zero_i32(int32_t* __restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

// Runs of equal keys in the sorted keys[0, nvalid): the first particle of
// each run writes runs[key] = {its position, the run length}, the length
// found by an exponential then a binary search (a long run costs its first
// thread O(log length), not O(length)), and sets the key's occupancy bit.
__global__ void k_cell_runs(const uint32_t* __restrict__ keys,
                            const unsigned long long* __restrict__ nvalid_p,
                            int2* __restrict__ runs, uint32_t* __restrict__ occ) {
  const int64_t nvalid = (int64_t)*nvalid_p;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvalid;
       i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t k = keys[i];
    if (i > 0 && keys[i - 1] == k) continue;
    int64_t lo = i, hi = i + 1, step = 1;  // keys[lo] == k
    while (hi < nvalid && keys[hi] == k) {
      lo = hi;
      step <<= 1;
      hi = lo + step < nvalid ? lo + step : nvalid;
    }
    while (hi - lo > 1) {  // keys[lo] == k; hi == nvalid or keys[hi] != k
      const int64_t mid = lo + (hi - lo) / 2;
      if (keys[mid] == k)
        lo = mid;
      else
        hi = mid;
    }
    runs[k] = make_int2((int)i, (int)(lo + 1 - i));
    atomicOr(&occ[k >> 5], 1u << (k & 31));
  }
}

// Run {first, count} of key cell c: {0, 0} unless its occupancy bit is set.
__device__ __forceinline__ int2 cell_run(const uint32_t* __restrict__ occ,
                                         const int2* __restrict__ runs, int64_t c) {
  return ((occ[c >> 5] >> (c & 31)) & 1u) ? runs[c] : make_int2(0, 0);
}

// v mod n for the halo of a tile: one compare in the common case, the full
// modulo only on grids smaller than the halo.
__device__ __forceinline__ int wrap_index(int v, int n) {
  if ((unsigned)v < (unsigned)n) return v;
  if (v < 0 && v + n >= 0) return v + n;
  if (v >= n && v - n < n) return v - n;
  return ((v % n) + n) % n;
}

// Stencils: target cell = key cell + o, o in [OMIN, OMAX] per axis, with
// 1D weights wt[o - OMIN] of the offset r from the key cell.
template <int SCHEME>
struct Stencil;
template <>
struct Stencil<0> {  // NGP, distribution_functions.h:25-32
  static constexpr int OMIN = 0, OMAX = 0;
  static constexpr double anchor = 0.0;
  __device__ static void weights(double, double* wt) { wt[0] = 1.0; }
};
template <>
struct Stencil<1> {  // TSC, distribution_functions.h:59-67
  static constexpr int OMIN = -1, OMAX = 1;
  static constexpr double anchor = 0.0;
  __device__ static void weights(double r, double* wt) {
#pragma clang fp contract(off)
    wt[0] = 0.5 * (1 - r) * (1 - r);
    wt[1] = 0.5 + r - r * r;
    wt[2] = 0.5 * r * r;
  }
};
template <>
struct Stencil<3> {  // CIC about cell centres: key cell a <= x - 1/2 < a + 1
  static constexpr int OMIN = 0, OMAX = 1;
  static constexpr double anchor = 0.5;
  __device__ static void weights(double r, double* wt) {
#pragma clang fp contract(off)
    wt[0] = 1.0 - r;
    wt[1] = r;
  }
};

// First sorted particle at the z borders of the planes' tiles, per grid row
// (x, y): entries 2b and 2b + 1 bound the key cells that reach tile b from
// inside the row, entry 2 ntz starts the row's last key cell and entry
// 2 ntz + 1 ends its first one (the ranges that reach the row's other end
// through the periodic wrap).
__host__ __device__ inline int row_bounds(int n2) { return 2 * ((n2 + TZ - 1) / TZ) + 2; }

// The 64 entries of a wave lie close together: its two halves first search
// for the rows they begin and end with, 32 probes a step, and each lane then
// searches between the two (13 dependent loads instead of 24 at 20 million
// particles in 512^3; bound by that latency: 203 -> 117 us).
template <int SCHEME>
__global__ void k_row_bounds(const uint32_t* __restrict__ keys,
                             const unsigned long long* __restrict__ nvalid_p, int64_t nrows,
                             int n2, int32_t* __restrict__ bounds) {
  using S = Stencil<SCHEME>;
  const int nb = row_bounds(n2), ntz = nb / 2 - 1;
  const int nvalid = (int)*nvalid_p;
  const int lane = threadIdx.x % kWave;
  const int64_t entries = nrows * nb;
  for (int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; i0 < entries;
       i0 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i1 = i0 + kWave - 1 < entries ? i0 + kWave - 1 : entries - 1;
    // First particle at or after the start of the first row (lanes 0 .. 31)
    // and of the row after the last one (32 .. 63).
    const int64_t edge = (lane < 32 ? i0 / nb : i1 / nb + 1) * n2;  // at most ncells < 2^31
    const int sub = lane % 32;
    int lo = 0, hi = nvalid;  // keys[lo - 1] < edge <= keys[hi]
    while (__ballot(lo < hi) != 0ull) {
      // 32 probes part [lo, hi) into 33 pieces.
      const int step = (hi - lo) / 33 + 1;
      const int64_t at = lo + (int64_t)(sub + 1) * step - 1;
      const bool below = at < hi && (int64_t)keys[at] < edge;
      const uint32_t under = (uint32_t)(__ballot(below) >> (lane & 32));
      const int n = __popc(under);  // probes 0 .. n - 1 are below the edge
      const int64_t nlo = lo + (int64_t)n * step, nhi = nlo + step - 1;
      if (lo < hi) {
        lo = (int)nlo;
        hi = (int)(nhi < hi ? nhi : hi);
        if (lo > hi) lo = hi;
      }
    }
    const int first = __shfl(lo, 0, kWave), last = __shfl(lo, 32, kWave);
    const int64_t i = i0 + lane;
    if (i >= entries) continue;
    const int64_t row = i / nb;
    const int j = (int)(i - row * nb), b = j >> 1;
    int z;
    if (b < ntz)
      z = (j & 1) ? min(b * TZ + TZ - S::OMIN, n2) : max(b * TZ - S::OMAX, 0);
    else
      z = (j & 1) ? 1 : n2 - 1;
    const uint32_t key = (uint32_t)(row * n2 + z);
    lo = first;
    hi = last;  // keys[lo - 1] < key <= keys[hi]
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if (keys[mid] < key)
        lo = mid + 1;
      else
        hi = mid;
    }
    bounds[i] = lo;
  }
}

// One wave per TY x TZ tile of target cells of one x plane, without any
// barrier.  The key cells that reach the tile are W RY rows, each up to three
// ranges of the sorted particles (inside the row, and through the wrap from
// either end).  Lane l takes the l-th of 64 equal shares of the concatenated
// ranges and walks it in order, summing the W x W weights of one key cell in
// registers; when the key cell changes it adds them to the wave's FP64 copies
// of the tile in LDS, one per plane of key cells.  Two lanes never hit one
// address in one instruction: key cells of one plane differ in their targets
// for each of the W x W offsets, and a key cell spread over several lanes ends
// inside the share of one of them only, the others hold it at the end of their
// share and add it after the loop, one lane after the other.  So each target
// cell is summed in an order that the input alone decides.
//
// Bound by the latency of a tile's chain (bounds, records, LDS adds) and by
// the lanes a sparse tile leaves idle, not by memory: hence no barrier, grid
// cells requested first, and the wave order of the XCDs, which lets the tiles
// that share rows meet in one L2.  20 million particles CIC into 512^3 FP32
// 0.77 ms (2.06 ms with a workgroup per 4 x 4 x 32 tile and a segmented scan
// across lanes); 3 million clustered particles TSC into 256^3 FP64 0.21 ms
// (0.80 ms).  Four rows instead of eight: 0.79 and 0.24 ms.
template <typename Tg, int SCHEME>
__global__ void __launch_bounds__(kTileThreads)
    k_ma_tile(Tg* __restrict__ grid, GridGeom g, const int32_t* __restrict__ bounds,
              const double4* __restrict__ srec, int tiles_y, int tiles_z) {
#pragma clang fp contract(off)
  using S = Stencil<SCHEME>;
  constexpr int W = S::OMAX - S::OMIN + 1;
  constexpr int RY = TY + W - 1;                   // key rows that reach the tile, per key plane
  constexpr int PY = TY + 2 * (W - 1), PZ = TZ + 2 * (W - 1);  // tile with the stencils' margin
  constexpr int NROW = W * RY, NKIND = W, NQ = NROW * NKIND;
  constexpr int kChunks = (NQ + kWave - 1) / kWave;
  __shared__ double acc_s[kTileWaves][W * PY * PZ];  // one copy per key plane
  __shared__ int32_t first_s[kTileWaves][kChunks * kWave];    // first particle of each range
  __shared__ int32_t pre_s[kTileWaves][kChunks * kWave + 1];  // exclusive prefix of their lengths

  int b = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  const int bz = b % tiles_z;
  b /= tiles_z;
  const int by = b % tiles_y;
  const int bx = b / tiles_y;
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  const int x = bx * kTileWaves + wv, y0 = by * TY, z0 = bz * TZ;
  if (x >= g.n0) return;
  double* acc = acc_s[wv];
  int32_t* first = first_s[wv];
  int32_t* pre = pre_s[wv];
  const int nb = row_bounds(g.n2);

  int begin[kChunks], len[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int q = c * kWave + lane;
    const int kind = q / NROW, row = q % NROW;
    const int y = y0 - S::OMAX + row % RY;
    bool on = q < NQ && y < g.n1 - S::OMIN;
    int lo = 2 * bz, hi = 2 * bz + 1;
    if (kind == 1) {  // the last key cell of the row reaches its first target cell
      on = on && bz == 0;
      lo = nb - 2;
      hi = nb - 3;
    } else if (kind == 2) {  // the first key cell reaches the last target cell
      on = on && bz == tiles_z - 1;
      lo = 0;
      hi = nb - 1;
    }
    begin[c] = len[c] = 0;
    if (on) {
      const int gx = wrap_index(x - S::OMAX + row / RY, g.n0);
      const int32_t* t = bounds + ((int64_t)gx * g.n1 + wrap_index(y, g.n1)) * nb;
      begin[c] = t[lo];
      len[c] = t[hi] - begin[c];
    }
  }
  int total = 0;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    int incl = len[c];
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int t = __shfl_up(incl, d, kWave);
      if (lane >= d) incl += t;
    }
    first[c * kWave + lane] = begin[c];
    pre[c * kWave + lane] = total + incl - len[c];
    total += __shfl(incl, kWave - 1, kWave);
  }
  if (total == 0) return;  // no particle reaches this tile
  if (lane == 0) pre[kChunks * kWave] = total;
  for (int i = lane; i < W * PY * PZ; i += kWave) acc[i] = -0.0;  // -0 + v == v; see the store
  // The tile's own grid cells, requested before the particles.
  constexpr int kOut = TY * TZ / kWave;
  Tg old[kOut];
  Tg* dst[kOut];
#pragma unroll
  for (int q = 0; q < kOut; ++q) {
    const int tz = lane % TZ, ty = (lane + q * kWave) / TZ;
    dst[q] = y0 + ty < g.n1 && z0 + tz < g.n2
                 ? grid + ((int64_t)x * g.n1 + (y0 + ty)) * g.n2 + (z0 + tz)
                 : nullptr;
    old[q] = dst[q] ? *dst[q] : Tg(0);
  }
  wave_lds_fence();

  const int share = (total - 1) / kWave + 1;
  const int64_t p0 = (int64_t)lane * share;
  int left = (int)(p0 >= total ? 0 : total - p0 < share ? total - p0 : share);
  int q = 0, idx = 0, in_range = 0;
  double4 next = make_double4(0, 0, 0, 0);
  if (left > 0) {
    int hi = kChunks * kWave;  // pre[q] <= p0 < pre[hi]
    while (hi - q > 1) {
      const int mid = (q + hi) >> 1;
      if (pre[mid] <= p0)
        q = mid;
      else
        hi = mid;
    }
    idx = first[q] + (int)(p0 - pre[q]);
    in_range = pre[q + 1] - (int)p0;
    next = srec[idx];
  }
  const bool any = left > 0;
  double v[W][W];
#pragma unroll
  for (int bb = 0; bb < W; ++bb)
#pragma unroll
    for (int c = 0; c < W; ++c) v[bb][c] = 0.0;
  int held = -1;  // key cell of v: its corner target in its plane's copy
  auto flush = [&] {
    double* t = acc + held;
#pragma unroll
    for (int bb = 0; bb < W; ++bb)
#pragma unroll
      for (int c = 0; c < W; ++c)
        __hip_atomic_fetch_add(t + bb * PZ + c, v[bb][c], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  for (int j = 0; j < share; ++j) {
    if (left > 0) {
      const double4 p = next;
      const int kind = q / NROW, row = q % NROW, rx = row / RY, ry = row % RY;
      // Advance; the next record is on its way while this one is summed.
      ++idx;
      if (--left > 0) {
        if (--in_range == 0) {
          do {
            ++q;
            in_range = pre[q + 1] - pre[q];
          } while (in_range == 0);
          idx = first[q];
        }
        next = srec[idx];
      }
      const double fz = floor(p.z);
      int iz = (int)fz;
      if (iz < 0) iz += g.n2;
      const int rz = iz + S::OMAX - (kind == 0 ? z0 : kind == 1 ? g.n2 : z0 - g.n2);
      const int cell = (rx * PY + ry) * PZ + rz;
      double wx[W], wy[W], wz[W];
      S::weights(p.x, wx);
      S::weights(p.y, wy);
      S::weights(p.z - fz, wz);
      double wa = wx[W - 1];  // the key plane x - OMAX + rx adds with weight W - 1 - rx
#pragma unroll
      for (int o = 1; o < W; ++o) wa = rx == o ? wx[W - 1 - o] : wa;
      wa = wa * p.w;  // weight folded into x, as the reference
      if (cell != held) {
        if (held >= 0) flush();
        held = cell;
#pragma unroll
        for (int bb = 0; bb < W; ++bb)
#pragma unroll
          for (int c = 0; c < W; ++c) v[bb][c] = 0.0;
      }
#pragma unroll
      for (int bb = 0; bb < W; ++bb) {
        const double vxy = wa * wy[bb];
#pragma unroll
        for (int c = 0; c < W; ++c) v[bb][c] += vxy * wz[c];
      }
    }
  }
  // What each lane still holds: equal key cells sit in neighbouring lanes.
  const int prev = __shfl_up(held, 1, kWave);
  const unsigned long long heads = __ballot(lane == 0 || prev != held);
  const unsigned long long upto = heads & (~0ull >> (kWave - 1 - lane));
  const int rank = any ? lane - (kWave - 1 - __clzll((long long)upto)) : -1;
  for (int r = 0; __ballot(rank >= r) != 0ull; ++r)
    if (rank == r) flush();
  wave_lds_fence();
  // A sum that is still -0 had no particle: adding it would change nothing.
#pragma unroll
  for (int q = 0; q < kOut; ++q) {
    const int tz = lane % TZ, ty = (lane + q * kWave) / TZ;
    double add = acc[(ty + W - 1) * PZ + tz + W - 1];
#pragma unroll
    for (int c = 1; c < W; ++c) add += acc[(c * PY + ty + W - 1) * PZ + tz + W - 1];
    if (dst[q] && __double_as_longlong(add) != (long long)0x8000000000000000ull)
      *dst[q] = (Tg)((double)old[q] + add);
  }
}

// D12 wavelet (distribution_functions.h:162-217): a particle in cell s with
// sub-cell sample (sx, sy, sz) = floor(64 r) adds
// tab[ox][sx] w * tab[oy][sy] * tab[oz][sz] to cell s - 1 + o, o in [0, 8)^3,
// tab being the caller's 8 x 64 sample table (d12.h's wavesample order).
// Target t therefore gathers from source cells t - 6 .. t + 1 per axis.
constexpr int WC = 8, WS = 64;
constexpr int WTX = 2, WTY = 4, WTZ = 32;  // target tile (256 cells, one per thread)
constexpr int DX = WTX + WC - 1, DY = WTY + WC - 1, DZ = WTZ + WC - 1;

template <typename Tg>
__global__ void __launch_bounds__(WTX* WTY* WTZ)
    k_ma_gather_wavelet(Tg* __restrict__ grid, GridGeom g, const int2* __restrict__ runs,
                        const uint32_t* __restrict__ occ,
                        const double4* __restrict__ srec, const double* __restrict__ table,
                        int tiles_y, int tiles_z) {
#pragma clang fp contract(off)
  __shared__ int32_t cs[DX * DY * DZ];
  __shared__ int32_t ce[DX * DY * DZ];
  __shared__ double tab[WC * WS];
  int b = blockIdx.x;
  const int bz = b % tiles_z;
  b /= tiles_z;
  const int by = b % tiles_y;
  const int bx = b / tiles_y;
  const int x0 = bx * WTX, y0 = by * WTY, z0 = bz * WTZ;
  for (int i = threadIdx.x; i < WC * WS; i += blockDim.x) tab[i] = table[i];
  for (int h = threadIdx.x; h < DX * DY * DZ; h += blockDim.x) {
    const int hz = h % DZ, hy = (h / DZ) % DY, hx = h / (DZ * DY);
    const int gx = wrap_index(x0 + hx - (WC - 2), g.n0);
    const int gy = wrap_index(y0 + hy - (WC - 2), g.n1);
    const int gz = wrap_index(z0 + hz - (WC - 2), g.n2);
    const int64_t c = ((int64_t)gx * g.n1 + gy) * g.n2 + gz;
    const int2 r = cell_run(occ, runs, c);
    cs[h] = r.x;
    ce[h] = r.x + r.y;
  }
  __syncthreads();
  const int tz = threadIdx.x % WTZ, ty = (threadIdx.x / WTZ) % WTY, tx = threadIdx.x / (WTZ * WTY);
  const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
  if (x >= g.n0 || y >= g.n1 || z >= g.n2) return;
  double sum = 0.0;
  bool touched = false;
  for (int ox = 0; ox < WC; ++ox)
    for (int oy = 0; oy < WC; ++oy)
      for (int oz = 0; oz < WC; ++oz) {
        const int h = ((tx + WC - 1 - ox) * DY + (ty + WC - 1 - oy)) * DZ + (tz + WC - 1 - oz);
        touched |= cs[h] < ce[h];
        for (int p = cs[h]; p < ce[h]; ++p) {
          const double4 q = srec[p];
          const int sx = (int)floor(q.x * WS), sy = (int)floor(q.y * WS), sz = (int)floor(q.z * WS);
          const double dxw = tab[ox * WS + sx] * q.w;
          const double dxy = dxw * tab[oy * WS + sy];
          sum += tab[oz * WS + sz] * dxy;
        }
      }
  if (touched) {
    Tg* cell = grid + ((int64_t)x * g.n1 + y) * g.n2 + z;
    *cell = (Tg)((double)*cell + sum);
  }
}

// Process-wide D12 table (fc_set_wavelet_table), copied to each context's
// device on first use after a change.
std::mutex g_wavelet_mu;
std::vector<double> g_wavelet;
uint64_t g_wavelet_ver = 0;

const double* wavelet_on_device(fc_ctx* ctx) {
  std::lock_guard<std::mutex> lk(g_wavelet_mu);
  if (g_wavelet.empty())
    fail(FC_ERR_INVALID,
         "distribution scheme 2 (D12 wavelet) needs its sample table: call "
         "fc_set_wavelet_table first");
  if (ctx->wavelet_ver != g_wavelet_ver) {
    ctx->wavelet.reserve(sizeof(double) * g_wavelet.size());
    FC_HIP(hipMemcpyAsync(ctx->wavelet.as<void>(), g_wavelet.data(),
                          sizeof(double) * g_wavelet.size(), hipMemcpyHostToDevice, ctx->stream));
    FC_HIP(hipStreamSynchronize(ctx->stream));
    ctx->wavelet_ver = g_wavelet_ver;
  }
  return ctx->wavelet.as<double>();
}

template <typename Tg>
void launch_wavelet(Tg* grid, const GridGeom& gg, const int2* runs, const uint32_t* occ,
                    const double4* srec, hipStream_t s, const double* table) {
  const int tx = (gg.n0 + WTX - 1) / WTX, ty = (gg.n1 + WTY - 1) / WTY,
            tz = (gg.n2 + WTZ - 1) / WTZ;
  const uint64_t nb = (uint64_t)tx * ty * tz;
  if (nb > 0x7fffffffULL) fail(FC_ERR_INVALID, "grid too large for mass assignment");
  hipLaunchKernelGGL((k_ma_gather_wavelet<Tg>), dim3((unsigned)nb), dim3(WTX * WTY * WTZ), 0, s,
                     grid, gg, runs, occ, srec, table, ty, tz);
  FC_LAUNCH_CHECK();
}

template <int SCHEME>
void launch_tiles(fc_grid* grid, const GridGeom& gg, const uint32_t* skeys,
                  const unsigned long long* nvalid, int32_t* bounds, const double4* srec,
                  hipStream_t s, hipEvent_t sorted) {
  const int64_t nrows = (int64_t)gg.n0 * gg.n1;
  const int ty = (gg.n1 + TY - 1) / TY, tz = (gg.n2 + TZ - 1) / TZ;
  const uint64_t nb = (uint64_t)((gg.n0 + kTileWaves - 1) / kTileWaves) * ty * tz;
  if (nb > 0x7fffffffULL) fail(FC_ERR_INVALID, "grid too large for mass assignment");
  hipLaunchKernelGGL((k_row_bounds<SCHEME>), dim3(grid1d(nrows * row_bounds(gg.n2), 256)),
                     dim3(256), 0, s, skeys, nvalid, nrows, gg.n2, bounds);
  FC_LAUNCH_CHECK();
  FC_HIP(hipEventRecord(sorted, s));
  if (grid->prec == FC_FP64)
    hipLaunchKernelGGL((k_ma_tile<double, SCHEME>), dim3((unsigned)nb), dim3(kTileThreads), 0, s,
                       grid->data.as<double>(), gg, bounds, srec, ty, tz);
  else
    hipLaunchKernelGGL((k_ma_tile<float, SCHEME>), dim3((unsigned)nb), dim3(kTileThreads), 0, s,
                       grid->data.as<float>(), gg, bounds, srec, ty, tz);
  FC_LAUNCH_CHECK();
}

int key_bits(uint64_t sentinel) {
  int b = 1;
  while (b < 64 && (sentinel >> b) != 0) ++b;
  return b;
}

// Bytes of the table that finds the sorted particles of a key cell: row
// bounds, or (D12 wavelet) a run per cell and the occupancy bits.
struct RunScratch {
  size_t runs, occ = 0;
  RunScratch(const int* shape, bool wavelet) {
    const size_t rows = (size_t)shape[0] * shape[1], cells = rows * shape[2];
    runs = wavelet ? sizeof(int2) * cells : sizeof(int32_t) * rows * row_bounds(shape[2]);
    if (wavelet) occ = sizeof(uint32_t) * ((cells + 31) / 32);
  }
};

template <class Source>
void mass_assign(fc_grid* grid, const Source& src, int64_t n, int scheme, int wrap, double shift,
                 fc_ma_stats* stats) {
  if (scheme < 0 || scheme > 3)
    fail(FC_ERR_INVALID, "unknown distribution scheme " + std::to_string(scheme));
  if (n < 0) fail(FC_ERR_INVALID, "negative particle count");
  if (n > 0x7fffffffLL) fail(FC_ERR_INVALID, "more than 2^31-1 particles in one call");
  if (!(shift >= 0.0 && shift < 1.0)) fail(FC_ERR_INVALID, "shift must be in [0, 1)");
  fc_ctx* ctx = grid->ctx;
  hipStream_t s = ctx->stream;
  DeviceGuard dg(ctx->device);
  const uint64_t ncells = grid->size();
  const uint64_t sentinel = ncells;
  GridGeom gg{grid->shape[0], grid->shape[1], grid->shape[2], grid->posmin[0],
              grid->posmin[1], grid->posmin[2], grid->cell};
  const double* wtab = scheme == 2 ? wavelet_on_device(ctx) : nullptr;
  if (scheme == 2)
    for (int d = 0; d < 3; ++d)
      if (grid->shape[d] < WC)
        fail(FC_ERR_INVALID, "the D12 wavelet needs at least 8 cells per axis");
  if (n == 0) return;

  hipEvent_t ev[3];
  for (auto& e : ev) FC_HIP(hipEventCreate(&e));
  struct EvGuard {
    hipEvent_t* e;
    ~EvGuard() {
      for (int i = 0; i < 3; ++i) (void)hipEventDestroy(e[i]);
    }
  } evg{ev};

  if (ncells >= 0x7fffffffULL) fail(FC_ERR_INVALID, "grid too large for mass assignment");
  const int nbp = (int)std::min<int64_t>(1024, (n + kPrepThreads - 1) / kPrepThreads);
  // Work buffers live in the context and are reused by later calls.
  DeviceBuffer* sc = ctx->scratch;
  sc[1].reserve(sizeof(uint32_t) * n);
  sc[2].reserve(sizeof(uint32_t) * n);
  sc[3].reserve(sizeof(uint32_t) * n);
  sc[4].reserve(sizeof(uint32_t) * n);
  sc[6].reserve(sizeof(double4) * n);
  sc[7].reserve(sizeof(double) * 2 * (nbp + 2));
  sc[8].reserve(sizeof(unsigned long long) * (nbp + 1));
  const RunScratch rs(grid->shape, scheme == 2);
  sc[9].reserve(rs.runs);
  sc[11].reserve(rs.occ);
  DeviceBuffer &keys = sc[1], &keys2 = sc[2], &idx = sc[3], &idx2 = sc[4], &srec = sc[6],
               &partw = sc[7], &partn = sc[8], &runs = sc[9], &occ = sc[11];
  const double anchor = scheme == 3 ? 0.5 : 0.0;  // CIC keys by its 2x2x2 block

  const Locator loc{gg, wrap, shift, anchor, scheme == 2};
  hipLaunchKernelGGL(k_ma_prepare<Source>, dim3(nbp), dim3(kPrepThreads), 0, s, src, n, loc,
                     (uint32_t)sentinel, keys.as<uint32_t>(), partw.as<double>(),
                     partn.as<unsigned long long>());
  FC_LAUNCH_CHECK();
  // The sums of w and w^2 and the number of particles on the grid, read back as one.
  unsigned long long* nvalid =
      reinterpret_cast<unsigned long long*>(partw.as<double>() + 2 * nbp + 2);
  hipLaunchKernelGGL(k_ma_finish_stats, dim3(1), dim3(64), 0, s, partw.as<double>(),
                     partn.as<unsigned long long>(), nbp, partw.as<double>() + 2 * nbp, nvalid);
  FC_LAUNCH_CHECK();

  FC_HIP(hipEventRecord(ev[0], s));
  const int bits = key_bits(sentinel);
  ctx->scratch[0].reserve(radix_plan(n, bits).scratch_bytes());
  const bool second = radix_sort_pairs(keys.as<uint32_t>(), keys2.as<uint32_t>(),
                                       idx.as<uint32_t>(), idx2.as<uint32_t>(), n, bits,
                                       ctx->scratch[0].as<void>(), s);
  const uint32_t* skeys = second ? keys2.as<uint32_t>() : keys.as<uint32_t>();
  const uint32_t* sidx = second ? idx2.as<uint32_t>() : idx.as<uint32_t>();
  hipLaunchKernelGGL(k_records<Source>, dim3(grid1d(n, 256, 65536)), dim3(256), 0, s, sidx, src,
                     loc, nvalid, srec.as<double4>());
  FC_LAUNCH_CHECK();
  if (scheme == 2) {
    const int64_t nwords = (int64_t)(rs.occ / sizeof(uint32_t));
    hipLaunchKernelGGL(k_zero_i32, dim3(grid1d(nwords, 256, 65536)), dim3(256), 0, s,
                       occ.as<int32_t>(), nwords);
    FC_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_cell_runs, dim3(grid1d(n, 256, 65536)), dim3(256), 0, s, skeys, nvalid,
                       runs.as<int2>(), occ.as<uint32_t>());
    FC_LAUNCH_CHECK();
    FC_HIP(hipEventRecord(ev[1], s));
    if (grid->prec == FC_FP64)
      launch_wavelet(grid->data.as<double>(), gg, runs.as<int2>(), occ.as<uint32_t>(),
                     srec.as<double4>(), s, wtab);
    else
      launch_wavelet(grid->data.as<float>(), gg, runs.as<int2>(), occ.as<uint32_t>(),
                     srec.as<double4>(), s, wtab);
  } else {
    const auto launch = scheme == 0   ? launch_tiles<0>
                        : scheme == 1 ? launch_tiles<1>
                                      : launch_tiles<3>;
    launch(grid, gg, skeys, nvalid, runs.as<int32_t>(), srec.as<double4>(), s, ev[1]);
  }
  FC_HIP(hipEventRecord(ev[2], s));

  double wsum[2];
  unsigned long long nadd = 0;
  read_back(ctx, partw.as<double>() + 2 * nbp, sizeof(wsum) + sizeof(nadd), [&](const char* p) {
    std::memcpy(wsum, p, sizeof(wsum));
    std::memcpy(&nadd, p + sizeof(wsum), sizeof(nadd));
  });
  float t_sort = 0, t_win = 0;
  FC_HIP(hipEventElapsedTime(&t_sort, ev[0], ev[1]));
  FC_HIP(hipEventElapsedTime(&t_win, ev[1], ev[2]));
  if (stats) {
    stats->num_added += nadd;
    stats->num_skipped += (uint64_t)n - nadd;
    stats->totw += wsum[0];
    stats->totwsq += wsum[1];
    stats->sort_time += t_sort * 1e-3;
    stats->window_time += t_win * 1e-3;
  }
}

}  // namespace

void mass_assign_device(fc_grid* grid, const double* pos_dev, int64_t n, int ncol,
                        const double* w_dev, double w_scalar, int scheme, int wrap, double shift,
                        fc_ma_stats* stats) {
  if (ncol != 3 && ncol != 4) fail(FC_ERR_INVALID, "Rows must be 3D or 4D.");
  mass_assign(grid, ArraySource{pos_dev, ncol, w_dev, w_scalar}, n, scheme, wrap, shift, stats);
}

// n particles of the random generator, uniform in [lo, lo + span).
void mass_assign_uniform(fc_grid* grid, int64_t n, double3 lo, double3 span, uint64_t seed,
                         uint64_t first, double weight, int scheme, int wrap,
                         fc_ma_stats* stats) {
  mass_assign(grid, UniformSource{lo, span, seed, first, weight}, n, scheme, wrap, 0.0, stats);
}

}  // namespace fc

extern "C" {

int fc_set_wavelet_table(const double* table, int n) {
  return fc::guard([&] {
    if (table && n != fc::WC * fc::WS)
      fc::fail(FC_ERR_INVALID, "the D12 table has 8 x 64 = 512 samples");
    std::lock_guard<std::mutex> lk(fc::g_wavelet_mu);
    if (table)
      fc::g_wavelet.assign(table, table + n);
    else
      fc::g_wavelet.clear();
    ++fc::g_wavelet_ver;
  });
}

int fc_mass_assign_footprint(fc_grid* grid, int64_t n, int ncol, int has_weights,
                             int host_input, size_t* grow, size_t* transient) {
  return fc::guard([&] {
    fc::check_grid(grid);
    if (n < 0) fc::fail(FC_ERR_INVALID, "negative particle count");
    if (ncol != 3 && ncol != 4) fc::fail(FC_ERR_INVALID, "Rows must be 3D or 4D.");
    fc_ctx* ctx = grid->ctx;
    fc::DeviceGuard dg(ctx->device);
    size_t g = 0;
    if (n > 0) {
      const uint64_t ncells = grid->size();
      const int nbp = (int)std::min<int64_t>(1024, (n + fc::kPrepThreads - 1) / fc::kPrepThreads);
      const size_t temp = fc::radix_plan(n, fc::key_bits(ncells)).scratch_bytes();
      const fc::RunScratch tiles(grid->shape, false), wavelet(grid->shape, true);
      const size_t want[12] = {temp,
                               sizeof(uint32_t) * n,
                               sizeof(uint32_t) * n,
                               sizeof(uint32_t) * n,
                               sizeof(uint32_t) * n,
                               0,
                               sizeof(double4) * n,
                               sizeof(double) * 2 * (nbp + 2),
                               sizeof(unsigned long long) * (nbp + 1),
                               std::max(tiles.runs, wavelet.runs),
                               host_input ? sizeof(double) * n * (ncol + (has_weights ? 1 : 0)) : 0,
                               wavelet.occ};
      for (int i = 0; i < 12; ++i)
        if (want[i] > ctx->scratch[i].bytes()) g += want[i] - ctx->scratch[i].bytes();
    }
    if (grow) *grow = g;
    if (transient) *transient = 0;
  });
}

int fc_mass_assign_device(fc_grid* grid, const double* pos_dev, int64_t n, int ncol,
                          const double* weights_dev, double w_scalar, int scheme,
                          int periodic_wrap, double shift, fc_ma_stats* stats) {
  return fc::guard([&] {
    fc::check_grid(grid);
    if (n > 0 && !pos_dev) fc::fail(FC_ERR_INVALID, "null positions");
    fc::mass_assign_device(grid, pos_dev, n, ncol, weights_dev, w_scalar, scheme, periodic_wrap,
                           shift, stats);
  });
}

int fc_mass_assign(fc_grid* grid, const double* pos, int64_t n, int ncol,
                   const double* weights, double w_scalar, int scheme, int periodic_wrap,
                   double shift, fc_ma_stats* stats) {
  return fc::guard([&] {
    fc::check_grid(grid);
    if (n > 0 && !pos) fc::fail(FC_ERR_INVALID, "null positions");
    if (ncol != 3 && ncol != 4) fc::fail(FC_ERR_INVALID, "Rows must be 3D or 4D.");
    if (n <= 0) return;
    fc::DeviceGuard dg(grid->ctx->device);
    hipStream_t s = grid->ctx->stream;
    fc_ctx* ctx = grid->ctx;
    ctx->scratch[10].reserve(sizeof(double) * n * (ncol + (weights ? 1 : 0)));
    double* dpos = ctx->scratch[10].as<double>();
    double* dw = weights ? dpos + n * ncol : nullptr;
    // Staged copies from the length on that HostCopier takes them, which only
    // then is made (its page-locked slots, streams and events take 140 us).
    const bool staged = sizeof(double) * n * ncol >= fc::HostCopier::kMinBytes;
    if (staged && !ctx->copier) ctx->copier.reset(new fc::HostCopier(ctx->device));
    auto copy = [&](double* d, const double* h, size_t bytes) {
      FC_HIP(staged ? ctx->copier->copy(d, h, bytes, s)
                    : hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, s));
    };
    copy(dpos, pos, sizeof(double) * n * ncol);
    if (weights) copy(dw, weights, sizeof(double) * n);
    fc::mass_assign_device(grid, dpos, n, ncol, dw, w_scalar, scheme, periodic_wrap, shift, stats);
  });
}

}  // extern "C"
