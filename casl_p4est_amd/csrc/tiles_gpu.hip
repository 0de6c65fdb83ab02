// The tiled stencil encoding (tiles.hpp) built on the device from tables that
// are already there (a grid built by casl_device_grid_build), so a grid that
// changes every step does not travel to the host and back.  The result is the
// host builder's (tiles.cpp) byte for byte:
//
//   scales     the coarsest and the finest arm cell of every axis: one reduction
//   tables     one pass over the tables makes the stencil's own copy, checks
//              every index and distance and everything of a record that does
//              not depend on its tile, and leaves 32 bytes per node (NodeSum):
//              what the steps below read instead of the tables' 337
//   halos      a block per tile collects H1 and H2 in an LDS hash set and sorts
//              them there; a tile whose halo exceeds the LDS limits is halved
//              and its halves are tried in the next round, which gives the
//              tiles of the host's depth-first halving in order
//   records    a block per tile ranks its record positions by (group,
//              position), the host's emission order, looks the corners' slots
//              up and writes every record in place
//   check      the independent bounds check of validate_tile_host, per tile
// The stencil it fills keeps only device arrays; the few scalars the host
// needs (the scales, the record counts, which tiles were halved, the error
// flags) are the only values copied back.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "reinit_device.hpp"
#include "tiles_device.hpp"

using namespace casl;
using namespace casl::dev;

namespace {

constexpr int BLOCK = 256;
inline unsigned grid_for(int64_t n) {
  if (n >= (int64_t(1) << 31)) throw std::runtime_error("grid too large for one launch");
  return unsigned(std::max<int64_t>(1, (n + BLOCK - 1) / BLOCK));
}

// error bits raised by the kernels
enum : int {
  BAD_INDEX = 1,       // a stencil node index out of range
  BAD_ZERO = 2,        // a zero face distance
  BAD_INEXACT = 4,     // a distance not exact in FP32
  BAD_SCALE = 8,       // an arm cell that is not base * 2^-l, 0 <= l <= 15
  BAD_ENCODE = 16,     // a corner outside T u H1 u H2
  BAD_UNITS = 32,      // a transverse offset that is not a multiple of the finest cell
  BAD_VERIFY = 64,     // a decoded record differs from the tables
  BAD_BOUNDS = 128,    // the independent bounds check failed
  BAD_NODE = 512,      // a node the encoding cannot hold (no corner of nonzero weight, too many hanging faces)
  ODD_WEIGHT = 256,    // no error: a regular face whose transverse offsets are not base * 2^-l
};

// The flattened tables on the device (FP64 distances), as casl_flat_stencil.
template <int D>
struct DTab {
  static constexpr int F = 2 * D, C = 1 << (D - 1), T = 2 * (D - 1);
  const int32_t *__restrict__ nbr;
  const double *__restrict__ d;
  const double *__restrict__ dtr;
  const uint8_t *__restrict__ wall;
  int64_t N;
  __device__ int32_t nb(int f, int c, int64_t n) const { return nbr[(int64_t(f) * C + c) * N + n]; }
  __device__ double df(int f, int64_t n) const { return d[int64_t(f) * N + n]; }
  __device__ double dt(int f, int k, int64_t n) const { return dtr[(int64_t(f) * T + k) * N + n]; }
  // get_linear_interpolation_weights of a face's corners from its transverse offsets
  __device__ static void weights_of(const double *u, double *wt) {
    const double m0 = u[0], p0 = u[1];
    if constexpr (D == 2) {
      wt[0] = p0;
      wt[1] = m0;
    } else {
      const double zm = u[2], zp = u[3];
      wt[0] = p0 * zp;
      wt[1] = m0 * zp;
      wt[2] = p0 * zm;
      wt[3] = m0 * zm;
    }
  }
};

__device__ __forceinline__ void transverse(int D, int a, int &t1, int &t2) {
  if (D == 2) {
    t1 = 1 - a;
    t2 = -1;
  } else {
    t1 = (a == 0 ? 1 : 0);
    t2 = (a == 2 ? 1 : 2);
  }
}

// The scales of the encoding: per axis, the coarsest arm cell and the finest
// cell (a cell of level l spans base[a] * 2^-l along axis a).
struct Scales {
  double base[3], unit[3];
  int lmax;
};

__device__ __forceinline__ void flag(int *bad, int bit) { atomicOr(bad, bit); }

// What the host reads back between the steps, and the kernels' shared words.
struct BuildState {
  unsigned long long amax[3], amin[3];  // bits of the coarsest and finest arm cell per axis
  int bad;
  int pad;
  long long n_uni, n_rec, n_ext, n_halo;
};

// ---------------------------------------------------------------- scales
// Blocks of the scale reduction: each thread strides over the nodes, the block
// reduces through wave shuffles and LDS, and one atomic per block and axis
// reaches memory (one per node serialized on the few target words).
constexpr unsigned REDUCE_BLOCKS = 2048;
inline unsigned reduce_grid(int64_t n) { return std::max(1u, std::min(REDUCE_BLOCKS, grid_for(n))); }

template <class T>
__device__ __forceinline__ T block_max(T v) {
  __shared__ T part[BLOCK / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const T w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  __syncthreads();  // part[] may still be read by a previous call
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < BLOCK / 64; ++k) v = part[k] > v ? part[k] : v;
  return v;  // the block's maximum in thread 0
}

// the coarsest and the finest arm cell per axis (non-negative doubles order
// like their bit patterns)
template <int D>
__global__ void __launch_bounds__(BLOCK) k_arm_range(DTab<D> t, BuildState *__restrict__ out) {
  double mx[D], mn[D];
#pragma unroll
  for (int a = 0; a < D; ++a) {
    mx[a] = 0.0;
    mn[a] = HUGE_VAL;
  }
  bool bad = false;
  for (int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; n < t.N; n += int64_t(gridDim.x) * blockDim.x) {
    const uint8_t w = t.wall[n];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const double d0 = t.df(2 * a, n), d1 = t.df(2 * a + 1, n);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const double arm = ((w >> (2 * a + q)) & 1) ? (q ? -d1 - d0 : -d0 - d1) : (q ? d1 : d0);
        if (arm > 0) {
          mx[a] = fmax(mx[a], arm);
          mn[a] = fmin(mn[a], arm);
        } else {
          bad = true;
        }
      }
    }
  }
  if (bad) flag(&out->bad, BAD_SCALE);
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const unsigned long long x = block_max((unsigned long long)__double_as_longlong(mx[a]));
    const unsigned long long y = block_max(~(unsigned long long)__double_as_longlong(mn[a]));
    if (threadIdx.x == 0) {
      atomicMax(&out->amax[a], x);
      atomicMin(&out->amin[a], ~y);
    }
  }
}

// The level of an arm cell.  The host builder takes l = the nearest
// integer of log2(base / q) and requires base * 2^-l == q with 0 <= l <= 15;
// that accepts exactly the q with base's significand and a binary exponent l
// below base's, and returns that l, so the exponents are compared here
// without the logarithm.
__device__ __forceinline__ int level_of(double base, double q, int &bad) {
  int eb = 0, eq = 0;
  const double mb = frexp(base, &eb), mq = frexp(q, &eq);
  const int l = eb - eq;
  if (!(q > 0) || mb != mq || l < 0 || l > 15) {
    bad |= BAD_SCALE;
    return 0;
  }
  return l;
}

// The finest level: that of the finest arm cell, where every cell is a
// power-of-two fraction of the coarsest (else BAD_SCALE is raised per node).
// As the host builder: one scale per axis, axes past D keep the box edge 1.
template <int D>
CASL_HD inline Scales scales_of(const BuildState &b) {
  Scales sc;
  sc.lmax = 0;
  for (int a = 0; a < 3; ++a) sc.base[a] = 1.0;
  for (int a = 0; a < D; ++a) {
    double lo;
    __builtin_memcpy(&sc.base[a], &b.amax[a], sizeof(double));
    __builtin_memcpy(&lo, &b.amin[a], sizeof(double));
    int eb = 0, el = 0;
    (void)frexp(sc.base[a], &eb);
    (void)frexp(lo, &el);
    const int l = eb - el;
    if (l > sc.lmax && l < 16) sc.lmax = l;
  }
  for (int a = 0; a < 3; ++a) sc.unit[a] = ldexp(sc.base[a], -sc.lmax);
  return sc;
}

// ---------------------------------------------------------------- tables
// What the tiling needs of a node: per face its first corner of nonzero
// weight, the record's geometry word, and which faces hang on which corners.
struct alignas(32) NodeSum {
  int32_t prim[6];
  uint32_t geo;
  // bits 0-1: 0 uniform, 1 regular, 1 + k hanging on k faces; 2-4 and 5-7: the
  // hanging faces; 8-11 and 12-15: their corners of nonzero weight
  uint32_t hang;
  __device__ int kind() const { return int(hang & 3u); }
  __device__ int faces() const { return kind() - 1; }  // hanging faces (kind >= 2)
  __device__ int face(int q) const { return int((hang >> (2 + 3 * q)) & 7u); }
  __device__ uint32_t corners(int q) const { return (hang >> (8 + 4 * q)) & 15u; }
};
static_assert(sizeof(NodeSum) == 32, "NodeSum must be 32 bytes");

__device__ __forceinline__ NodeSum load_sum(const NodeSum *__restrict__ p, int64_t n) {
  const uint4 *q = reinterpret_cast<const uint4 *>(p + n);
  const uint4 a = q[0], b = q[1];
  NodeSum s;
  s.prim[0] = int32_t(a.x);
  s.prim[1] = int32_t(a.y);
  s.prim[2] = int32_t(a.z);
  s.prim[3] = int32_t(a.w);
  s.prim[4] = int32_t(b.x);
  s.prim[5] = int32_t(b.y);
  s.geo = b.z;
  s.hang = b.w;
  return s;
}

// v is 0 or base times a power of two
__device__ __forceinline__ bool scale_multiple(double b, double v) {
  int eb = 0, ev = 0;
  return v == 0.0 || frexp(b, &eb) == frexp(v, &ev);
}

// The one pass over the tables: indices checked, distances converted to FP32
// (exact, or the stencil cannot be made) and the stencil's copy written; the
// node's levels, walls and hanging faces taken, and checked as the host
// builder's verify() does: the decoded record reproduces the tables bit for
// bit.  SUM = false: the stencil's copy only.  Bound by the 337 bytes read and
// 249 written per node (3D): 8.1M nodes 1.01 ms (4.7 TB/s), where the
// conversion and the table copy (1.1 ms), a pass for the levels, and the
// tables read again by every step of the tiling took 4.4.
template <int D, bool SUM>
__global__ void __launch_bounds__(BLOCK) k_tables(DTab<D> t, int32_t *__restrict__ nbr, uint8_t *__restrict__ wall,
                                                  float *__restrict__ dist, NodeSum *__restrict__ sum,
                                                  BuildState *__restrict__ state) {
  constexpr int F = DTab<D>::F, C = DTab<D>::C, T = DTab<D>::T;
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= t.N) return;
  int bad = 0;
  const uint32_t w = t.wall[n];
  wall[n] = uint8_t(w);
  double d[F];
#pragma unroll
  for (int f = 0; f < F; ++f) {
    d[f] = t.df(f, n);
    if (!(d[f] != 0.0)) bad |= BAD_ZERO;
    const float v = float(d[f]);
    if (double(v) != d[f]) bad |= BAD_INEXACT;
    dist[int64_t(f) * t.N + n] = v;
  }
  Scales sc;
  NodeSum r;
  if constexpr (SUM) {
    sc = scales_of<D>(*state);
    r.prim[4] = r.prim[5] = 0;
    r.geo = (w & ((1u << F) - 1u)) << 24;
    r.hang = 0;
    double dd[F];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const double arm = ((w >> f) & 1u) ? (-d[f] - d[f ^ 1]) : d[f];
      const int l = level_of(sc.base[f >> 1], arm, bad);
      r.geo |= uint32_t(l) << (4 * f);
      dd[f] = ldexp(sc.base[f >> 1], -l);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      if ((w >> f) & 1u) dd[f] = -dd[f ^ 1] - ldexp(sc.base[f >> 1], -int((r.geo >> (4 * f)) & 15u));
      if (dd[f] != d[f]) bad |= BAD_VERIFY;
    }
  }
  int k = 0;  // hanging faces
#pragma unroll
  for (int f = 0; f < F; ++f) {
    int32_t g[C];
    double u[T];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      g[c] = t.nb(f, c, n);
      if (g[c] < 0 || g[c] >= t.N) bad |= BAD_INDEX;
      nbr[(int64_t(f) * C + c) * t.N + n] = g[c];
    }
#pragma unroll
    for (int q = 0; q < T; ++q) {
      u[q] = t.dt(f, q, n);
      const float v = float(u[q]);
      if (double(v) != u[q]) bad |= BAD_INEXACT;
      dist[(int64_t(F) + int64_t(f) * T + q) * t.N + n] = v;
    }
    if constexpr (SUM) {
      double wt[C];
      DTab<D>::weights_of(u, wt);
      uint32_t mask = 0;
#pragma unroll
      for (int c = 0; c < C; ++c) mask |= (wt[c] != 0.0) ? (1u << c) : 0u;
      int32_t first = g[0];
#pragma unroll
      for (int c = C - 1; c >= 0; --c)
        if ((mask >> c) & 1u) first = g[c];
      r.prim[f] = first;
      int t1, t2;
      transverse(D, f >> 1, t1, t2);
      if (mask == 0) {
        bad |= BAD_NODE;
      } else if ((mask & (mask - 1u)) == 0) {
#pragma unroll
        for (int q = 0; q < T; ++q)
          if (!scale_multiple(sc.base[q < 2 ? t1 : t2], u[q])) bad |= ODD_WEIGHT;
      } else {
        if (k == HangExt<D>::NH) {
          bad |= BAD_NODE;
        } else {
          r.hang |= (uint32_t(f) << (2 + 3 * k)) | (mask << (8 + 4 * k));
          ++k;
        }
        // the offsets in finest cells, and the arm cell's transverse extents
        // at the face's level
        const int l = int((r.geo >> (4 * f)) & 15u);
#pragma unroll
        for (int m = 0; m < D - 1; ++m) {
          const int ax = m == 0 ? t1 : t2;
          const double kk = u[2 * m] / sc.unit[ax];
          if (!(kk >= 0) || kk > 65535 || floor(kk) != kk || kk * sc.unit[ax] != u[2 * m])
            bad |= BAD_UNITS;
          else if (ldexp(sc.base[ax], -l) - u[2 * m] != u[2 * m + 1])
            bad |= BAD_VERIFY;
        }
      }
    }
  }
  if constexpr (SUM) {
    // uniform: regular, off the walls, all arms at one level
    constexpr uint32_t LEVELS = D == 2 ? 0x1111u : 0x111111u;
    const bool uniform = k == 0 && (r.geo >> 24) == 0 && r.geo == (r.geo & 15u) * LEVELS;
    r.hang |= uint32_t(k > 0 ? 1 + k : (uniform ? 0 : 1));
    if (k > 0) r.geo |= GEO_IRREGULAR;
    uint4 *q = reinterpret_cast<uint4 *>(sum + n);
    q[0] = make_uint4(uint32_t(r.prim[0]), uint32_t(r.prim[1]), uint32_t(r.prim[2]), uint32_t(r.prim[3]));
    q[1] = make_uint4(uint32_t(r.prim[4]), uint32_t(r.prim[5]), r.geo, r.hang);
  }
  if (bad) flag(&state->bad, bad);
}

// ---------------------------------------------------------------- halos
// A tile tried: its node range, and where its counts and its halo ids go.
struct TileItem {
  int32_t s, e;
};
// A tile kept: its counts (n1, n2, then the records of each group) and halo ids.
struct TileSrc {
  const int32_t *counts, *halo;
  int32_t s, pad;
};
constexpr int ITEM_COUNTS = 10;

// Block and LDS sizes of the tile kernels.
template <int D, bool SMALL>
struct TileBlock {
  static constexpr int LMAX = TileLimits<D, SMALL>::LMAX;
  static constexpr int HALO_THREADS = SMALL ? 256 : 1024;  // k_halos
  static constexpr int THREADS = SMALL ? 256 : 512;        // k_records
  static constexpr int TABLE = LMAX + LMAX / 2 - 64;  // hash set entries (two blocks of 80 KB per CU)
  static_assert(LMAX + HALO_THREADS < TABLE, "every probe of the hash set reaches an empty entry");
};

constexpr uint32_t NO_NODE = 0xffffffffu;

// Adds id to the set; true if it was not there.  The callers keep at least one
// entry empty, so every probe ends.
template <int TABLE>
__device__ __forceinline__ bool set_insert(uint32_t *set, uint32_t id) {
  uint32_t p = __umulhi(id * 2654435761u, uint32_t(TABLE));
  for (;;) {
    uint32_t cur = set[p];
    if (cur == NO_NODE) {
      cur = atomicCAS(&set[p], NO_NODE, id);
      if (cur == NO_NODE) return true;
    }
    if (cur == id) return false;
    if (++p == uint32_t(TABLE)) p = 0;
  }
}

// Ascending sort of v[0, n) in LDS by the whole block: the bitonic network
// with every comparison ascending (the first step of a merge mirrors its
// second half), so the entries past n count as largest and stay away.  Pairs
// up to 64 apart lie within the 128 entries of one wave's 64 pairs, whose
// steps need no barrier of the block.
template <int THREADS>
__device__ __forceinline__ void block_sort(int32_t *v, int n) {
  int half = 1;
  while (half < n) half <<= 1;
  half >>= 1;  // pairs
  bool far = true;
  for (int k = 2; k <= 2 * half; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (far || j > 64)
        __syncthreads();
      else
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      far = j > 64;
      for (int i = int(threadIdx.x); i < half; i += THREADS) {
        const int o = i & (j - 1), b = (i - o) << 1;
        const int l = b + o, r = j == (k >> 1) ? b + 2 * j - 1 - o : l + j;
        if (r < n) {
          const int32_t x = v[l], y = v[r];
          if (x > y) {
            v[l] = y;
            v[r] = x;
          }
        }
      }
    }
  }
  __syncthreads();
}

// Calls fn(id) for every corner of nonzero weight of node n.
template <int D, class Fn>
__device__ __forceinline__ void for_needed(const DTab<D> &t, const NodeSum &r, int64_t n, Fn fn) {
#pragma unroll
  for (int f = 0; f < DTab<D>::F; ++f) fn(r.prim[f]);
  for (int q = 0; q < r.faces(); ++q) {
    const uint32_t m = r.corners(q);
    for (uint32_t c = m & (m - 1u); c; c &= c - 1u) fn(t.nb(r.face(q), __ffs(int(c)) - 1, n));
  }
}

// H1 and H2 of one tile, each ascending, and the size of each of its record
// groups; counts[0] = -1 where the tile exceeds its LDS limits (the host's
// halo() test).  Bound by the latency of the set's probes and of the sorts'
// LDS steps; the tables are not touched but for hanging corners.  8.1M nodes
// 0.62 ms, where (tile, node) keys of every reference sorted by the whole grid
// (with their counting passes and scans) took 5.2.
template <int D, bool SMALL>
__global__ void __launch_bounds__((TileBlock<D, SMALL>::HALO_THREADS), (SMALL ? 4 : 8))
k_halos(DTab<D> t, const NodeSum *__restrict__ sum, const TileItem *__restrict__ items, int32_t *__restrict__ counts,
        int32_t *__restrict__ halos) {
  using B = TileBlock<D, SMALL>;
  using Lim = TileLimits<D, SMALL>;
  __shared__ uint32_t set[B::TABLE];
  __shared__ int32_t ids[B::LMAX];
  __shared__ int32_t found;
  __shared__ int32_t group[8];
  const int tid = int(threadIdx.x);
  const TileItem it = items[blockIdx.x];
  const int nT = it.e - it.s;
  int32_t *cnt = counts + int64_t(blockIdx.x) * ITEM_COUNTS;
  for (int i = tid; i < B::TABLE; i += B::HALO_THREADS) set[i] = NO_NODE;
  if (tid == 0) found = 0;
  if (tid < 8) group[tid] = 0;
  __syncthreads();
  // Once more than cap ids are there the tile does not fit: a thread that
  // sees it adds no more, so at most cap + THREADS ids enter the set.
  auto collect = [&](int32_t g, int cap) {
    if (g >= it.s && g < it.e) return;
    if (__hip_atomic_load(&found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > cap) return;
    if (!set_insert<B::TABLE>(set, uint32_t(g))) return;
    const int p = atomicAdd(&found, 1);
    if (p < B::LMAX) ids[p] = g;
  };
  auto count = [&](const int *c, int first) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int v = c[k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if ((tid & 63) == 0 && v) atomicAdd(&group[first + k], v);
    }
  };
  const int cap1 = Lim::DMAX - nT, cap2 = Lim::LMAX - nT;
  {
    int c[4] = {0, 0, 0, 0};
    for (int i = tid; i < nT; i += B::HALO_THREADS) {
      const NodeSum r = load_sum(sum, int64_t(it.s) + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) c[k] += r.kind() == k ? 1 : 0;
      for_needed<D>(t, r, int64_t(it.s) + i, [&](int32_t g) { collect(g, cap1); });
    }
    count(c, 0);
  }
  __syncthreads();
  const int n1 = found;
  if (n1 > cap1 || n1 > cap2) {
    if (tid == 0) cnt[0] = -1;
    return;
  }
  block_sort<B::HALO_THREADS>(ids, n1);
  {
    int c[4] = {0, 0, 0, 0};
    for (int i = tid; i < n1; i += B::HALO_THREADS) {
      const int32_t h = ids[i];
      const NodeSum r = load_sum(sum, h);
#pragma unroll
      for (int k = 0; k < 4; ++k) c[k] += r.kind() == k ? 1 : 0;
      for_needed<D>(t, r, h, [&](int32_t g) { collect(g, cap2); });
    }
    count(c, 4);
  }
  __syncthreads();
  const int n = found;
  if (n > cap2) {
    if (tid == 0) cnt[0] = -1;
    return;
  }
  block_sort<B::HALO_THREADS>(ids + n1, n - n1);
  int32_t *out = halos + int64_t(blockIdx.x) * Lim::LMAX;
  for (int i = tid; i < n; i += B::HALO_THREADS) out[i] = ids[i];
  if (tid == 0) {
    cnt[0] = n1;
    cnt[1] = n - n1;
  }
  if (tid < 8) cnt[2 + tid] = group[tid];
}

// The per-tile arrays: exclusive prefixes of the uniform, non-uniform and
// extension records and of the halo ids over the tiles, by one block.
constexpr int SCAN_THREADS = 1024;
struct TileStarts {
  int32_t *tile, *urec, *rec, *ext, *halo, *h1count;
  uint32_t *nreg, *nuni;
};
__global__ void __launch_bounds__(SCAN_THREADS) k_tile_starts(const TileSrc *__restrict__ src, int nt, int32_t N,
                                                              TileStarts o, BuildState *__restrict__ state) {
  __shared__ long long part[SCAN_THREADS / 64][4];
  const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
  long long base[4] = {0, 0, 0, 0};
  for (int t0 = 0; t0 < nt; t0 += SCAN_THREADS) {
    const int t = t0 + tid;
    long long v[4] = {0, 0, 0, 0}, x[4];
    if (t < nt) {
      const int32_t *c = src[t].counts;
      const int32_t *g = c + 2;
      v[0] = g[0] + g[4];
      v[1] = g[1] + g[2] + g[3] + g[5] + g[6] + g[7];
      v[2] = g[2] + g[3] + g[6] + g[7];
      v[3] = c[0] + c[1];
      o.tile[t] = src[t].s;
      o.nreg[t] = uint32_t(g[1]) | (uint32_t(g[5]) << 16);
      o.nuni[t] = uint32_t(g[0]) | (uint32_t(g[4]) << 16);
      o.h1count[t] = c[0];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = v[k];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const long long y = __shfl_up(x[k], unsigned(d), 64);
        if (lane >= d) x[k] += y;
      }
      if (lane == 63) part[wave][k] = x[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      long long before = base[k];
#pragma unroll 1
      for (int w = 0; w < SCAN_THREADS / 64; ++w) {
        if (w < wave) before += part[w][k];
        base[k] += part[w][k];
      }
      x[k] += before - v[k];
    }
    __syncthreads();
    if (t < nt) {
      o.urec[t] = int32_t(x[0]);
      o.rec[t] = int32_t(x[1]);
      o.ext[t] = int32_t(x[2]);
      o.halo[t] = int32_t(x[3]);
    }
  }
  if (tid == 0) {
    o.tile[nt] = N;
    o.urec[nt] = int32_t(base[0]);
    o.rec[nt] = int32_t(base[1]);
    o.ext[nt] = int32_t(base[2]);
    o.halo[nt] = int32_t(base[3]);
    state->n_uni = base[0];
    state->n_rec = base[1];
    state->n_ext = base[2];
    state->n_halo = base[3];
  }
}

// ---------------------------------------------------------------- records
// The output arrays of the encoding.
struct TileOut {
  TileRec *rec;
  uint16_t *rec_slot;
  uint32_t *urec;
  uint16_t *ext;
  int32_t *halo;
  const int32_t *urs, *rs, *xs, *hs;  // exclusive prefixes of the per-tile counts
};

// A tile handled by one block: its halo node ids, H1 then H2 (each in
// ascending order), staged in LDS with a hash set of their positions, and the
// LDS slot of a node of the tile.
template <int TABLE>
struct TileLocal {
  int32_t s, nT;  // the tile's nodes
  const int32_t *ids;
  uint32_t *set;
  __device__ static uint32_t start(int32_t g) { return __umulhi(uint32_t(g) * 2654435761u, uint32_t(TABLE)); }
  __device__ void insert(int j) const {
    uint32_t p = start(ids[j]);
    while (atomicCAS(&set[p], NO_NODE, uint32_t(j)) != NO_NODE)
      if (++p == uint32_t(TABLE)) p = 0;
  }
  // LDS slot of node g in T u H1 u H2, -1 if not there
  __device__ int32_t operator()(int32_t g) const {
    if (g >= s && g - s < nT) return g - s;
    uint32_t p = start(g);
    for (;;) {
      const uint32_t j = set[p];
      if (j == NO_NODE) return -1;
      if (ids[j] == g) return nT + int32_t(j);
      if (++p == uint32_t(TABLE)) p = 0;
    }
  }
};

// Every record of a tile at its place in the host builder's order, and the
// tile's halo ids.  A block takes its tile's positions a row at a time, T then
// H1: ballots rank a row's records within their groups.  Bound by the
// latency of the corners' look-ups, LDS hash probes: 8.1M nodes 0.57 ms, where the classification, the sort of
// its (tile, group) keys and an emission that encoded and checked every record
// from the tables took 5.6.
template <int D, bool SMALL>
__global__ void __launch_bounds__((TileBlock<D, SMALL>::THREADS))
k_records(DTab<D> t, const NodeSum *__restrict__ sum, const TileSrc *__restrict__ src, TileOut o,
          BuildState *__restrict__ state) {
  using B = TileBlock<D, SMALL>;
  constexpr int WAVES = B::THREADS / 64, F = DTab<D>::F, C = DTab<D>::C;
  constexpr int XW = HangExt<D>::WORDS, SW = HangExt<D>::SW;
  __shared__ int32_t ids[B::LMAX];
  __shared__ uint32_t set[B::TABLE];
  __shared__ uint8_t row[2][WAVES][4];
  const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6, tl = int(blockIdx.x);
  const TileSrc ts = src[tl];
  const int32_t *cnt = ts.counts;
  const int n1 = cnt[0], nh = cnt[0] + cnt[1];
  TileLocal<B::TABLE> loc;
  loc.s = ts.s;
  loc.nT = cnt[2] + cnt[3] + cnt[4] + cnt[5];
  loc.ids = ids;
  loc.set = set;
  if (nh > B::LMAX) {  // ruled out by the tile limits
    if (tid == 0) flag(&state->bad, BAD_BOUNDS);
    return;
  }
  for (int i = tid; i < B::TABLE; i += B::THREADS) set[i] = NO_NODE;
  for (int i = tid; i < nh; i += B::THREADS) {
    const int32_t g = ts.halo[i];
    ids[i] = g;
    o.halo[int64_t(o.hs[tl]) + i] = g;
  }
  __syncthreads();
  for (int i = tid; i < nh; i += B::THREADS) loc.insert(i);
  __syncthreads();
  const Scales sc = scales_of<D>(*state);
  int64_t ubase = o.urs[tl], rbase = o.rs[tl], xbase = o.xs[tl];
  int bad = 0, flip = 0;
  for (int part = 0; part < 2; ++part) {
    const int p0 = part == 0 ? 0 : loc.nT, p1 = part == 0 ? loc.nT : loc.nT + n1;
    const int32_t *g = cnt + 2 + 4 * part;
    const int gn[4] = {g[0], g[1], g[2], g[3]};
    int done[4] = {0, 0, 0, 0};  // records of each group in the rows before
    for (int r0 = p0; r0 < p1; r0 += B::THREADS, flip ^= 1) {
      const int i = r0 + tid;
      const bool live = i < p1;
      const int64_t n = !live ? 0 : part == 0 ? int64_t(loc.s) + i : int64_t(ids[i - loc.nT]);
      NodeSum r{};
      if (live) r = load_sum(sum, n);
      const int kind = live ? r.kind() : -1;
      int rank = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t m = __ballot(kind == k);
        if (kind == k) rank = __popcll(m & ((uint64_t(1) << lane) - 1));
        if (lane == 0) row[flip][wave][k] = uint8_t(__popcll(m));
      }
      __syncthreads();  // row[flip ^ 1] was read before this barrier: two sets are enough
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (kind == k) rank += done[k];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
          const int v = row[flip][w][k];
          if (kind == k && w < wave) rank += v;
          done[k] += v;
        }
      }
      if (!live) continue;
      TileRec rec;
      bool ok = true;
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        int32_t l = 0;
        if (f < F) l = loc(r.prim[f]);
        ok = ok && l >= 0 && l <= 65535;
        rec.idx[f] = uint16_t(l);
      }
      rec.geo = r.geo;
      if (kind == 0) {
        if (ok) uni_pack<D>(rec.idx, uint32_t(i), r.geo & 15u, o.urec + (ubase + rank) * UniRec<D>::WORDS);
      } else {
        const int64_t q = rbase + (kind > 1 ? gn[1] : 0) + (kind > 2 ? gn[2] : 0) + rank;
        if (ok) {
          o.rec[q] = rec;
          o.rec_slot[q] = uint16_t(i);
        }
        if (kind > 1 && ok) {
          uint16_t e[XW];
#pragma unroll
          for (int w = 0; w < XW; ++w) e[w] = 0;
          const int f0 = r.face(0), f1 = kind > 2 ? r.face(1) : int(HANG_NONE);
          e[0] = uint16_t(D == 2 ? f0 : (f0 | (f1 << 4)));
#pragma unroll
          for (int h = 0; h < HangExt<D>::NH; ++h) {
            if (h >= kind - 1) break;
            const int f = r.face(h);
            const uint32_t m = r.corners(h);
            const int first = __ffs(int(m)) - 1;
#pragma unroll
            for (int c = 0; c < C; ++c) {
              const int32_t l = loc(t.nb(f, ((m >> c) & 1u) ? c : first, n));
              ok = ok && l >= 0 && l <= 65535;
              e[1 + h * SW + c] = uint16_t(l);
            }
            int t1, t2;
            transverse(D, f >> 1, t1, t2);
#pragma unroll
            for (int a = 0; a < D - 1; ++a) {
              const int ax = a == 0 ? t1 : t2;
              const double u = ax == 0 ? sc.unit[0] : ax == 1 ? sc.unit[1] : sc.unit[2];
              e[1 + h * SW + C + a] = uint16_t(t.dt(f, 2 * a, n) / u);
            }
          }
          uint32_t *x = reinterpret_cast<uint32_t *>(o.ext + (xbase + (kind > 2 ? gn[2] : 0) + rank) * XW);
#pragma unroll
          for (int w = 0; w < XW / 2; ++w) x[w] = uint32_t(e[2 * w]) | (uint32_t(e[2 * w + 1]) << 16);
        }
      }
      if (!ok) bad |= BAD_ENCODE;
    }
    ubase += gn[0];
    rbase += gn[1] + gn[2] + gn[3];
    xbase += gn[2] + gn[3];
  }
  if (bad) flag(&state->bad, bad);
}

// The independent bounds check of validate_tile_host, one block per tile.
template <int D>
__global__ void k_validate(TileArgs<float> A, int64_t N, TileCaps caps, int *__restrict__ bad) {
  constexpr int F = 2 * D, C = 1 << (D - 1), DMAX = TileLimits<D>::DMAX;
  static_assert(TileLimits<D, true>::DMAX <= DMAX, "the bit set covers the larger tiles");
  constexpr int WORDS = HangExt<D>::WORDS, SW = HangExt<D>::SW;
  __shared__ uint32_t seen[(DMAX + 31) / 32];
  const int tile = int(blockIdx.x);
  TileCtx<D> c;
  c.load(A, tile);
  for (int w = int(threadIdx.x); w < (DMAX + 31) / 32; w += BLOCK) seen[w] = 0;
  __syncthreads();
  const int nTn = c.nT - c.nTu, nH1n = c.nH1 - c.nH1u;
  const int nTreg = int(c.nreg & 0xffffu), nH1reg = int(c.nreg >> 16);
  const int nR = A.rec_start[tile + 1] - c.rb, nU = A.urec_start[tile + 1] - c.ub;
  if (c.nT <= 0 || c.nH1 < 0 || c.nH1 > c.nH || c.nT + c.nH > caps.lmax || c.nT + c.nH1 > caps.dmax ||
      nR + nU != c.nT + c.nH1 || c.nTu > c.nT || c.nH1u > c.nH1 || c.nTu + c.nH1u != nU || nTreg > nTn ||
      nH1reg > nH1n || A.ext_start[tile + 1] - c.ext0 != (nTn - nTreg) + (nH1n - nH1reg)) {
    if (threadIdx.x == 0) flag(bad, BAD_BOUNDS);
    return;
  }
  for (int k = int(threadIdx.x); k < c.nH; k += BLOCK) {
    const int32_t g = A.halo[c.hb + k];
    if (g < 0 || g >= N) flag(bad, BAD_BOUNDS);
  }
  for (int i = int(threadIdx.x); i < c.nT + c.nH1; i += BLOCK) {
    RecRegs r;
    const int js = fetch_record<D>(A, c, i, r);
    int slot = js;
    const TileRec rec = record_at<D>(c, i, r, slot);
    const bool own = i < c.nT;
    if (own ? (slot < 0 || slot >= c.nT) : (slot < c.nT || slot >= c.nT + c.nH1)) {
      flag(bad, BAD_BOUNDS);
      continue;
    }
    if (atomicOr(&seen[slot >> 5], 1u << (slot & 31)) & (1u << (slot & 31))) flag(bad, BAD_BOUNDS);
    const int bound = own ? c.nT + c.nH1 : c.nT + c.nH;
    for (int f = 0; f < F; ++f)
      if (rec.idx[f] >= bound) flag(bad, BAD_BOUNDS);
    if (!c.uniform(i)) {
      const int j = c.npos(i);
      const bool irregular = (rec.geo & GEO_IRREGULAR) != 0;
      if (irregular != (own ? (j >= nTreg) : (j >= nTn + nH1reg))) flag(bad, BAD_BOUNDS);
      if (irregular) {
        const uint16_t *e = c.ext_of(A.ext, i);
        const int h0 = D == 2 ? e[0] : (e[0] & 15), h1 = D == 2 ? int(HANG_NONE) : ((e[0] >> 4) & 15);
        if (h0 >= F || (h1 != HANG_NONE && (h1 >= F || h1 <= h0))) flag(bad, BAD_BOUNDS);
        for (int q = 0; q < (h1 == HANG_NONE ? 1 : 2); ++q)
          for (int cc = 0; cc < C; ++cc)
            if (e[1 + q * SW + cc] >= bound) flag(bad, BAD_BOUNDS);
      }
    }
  }
  (void)WORDS;
}

// ------------------------------------------------------------ host side
std::string bad_reason(int b) {
  if (b & BAD_SCALE) return "arm cell size is not a power-of-two fraction of the coarsest cell";
  if (b & BAD_UNITS) return "transverse offset is not a multiple of the finest cell";
  if (b & (BAD_NODE | BAD_ENCODE))
    return "a record the encoding cannot hold (corner outside the tile's halo or too many hanging faces)";
  if (b & BAD_VERIFY) return "tile record does not reproduce the tables";
  if (b & BAD_BOUNDS) return "tiled encoding failed its bounds check";
  return "tiled encoding failed";
}

void read_state(const DevBuf<BuildState> &d, BuildState &h, hipStream_t s) {
  HIP_CHECK(hipMemcpyAsync(&h, d.p, sizeof(BuildState), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
}

// The tiles of one round of trials: the nodes of each, and what came of it.
struct Round {
  DevBuf<TileItem> items;
  DevBuf<int32_t> counts, halos;
};

// A tile: its nodes, and where what came of its trial lies.
struct Tile {
  int32_t s, e, round, item;
};

// The tiles of a grid, in order: candidates of the tile size; those whose halo
// does not fit give way to their halves, which are tried in the next round.
template <int D, bool SMALL>
std::vector<Tile> cut_tiles(const DTab<D> &tab, const DevBuf<NodeSum> &sum,
                            std::vector<std::unique_ptr<Round>> &rounds, hipStream_t s) {
  using B = TileBlock<D, SMALL>;
  using Lim = TileLimits<D, SMALL>;
  const int64_t N = tab.N;
  std::vector<Tile> tiles;
  for (int64_t x = 0; x < N; x += Lim::TMAX)
    tiles.push_back({int32_t(x), int32_t(std::min<int64_t>(N, x + Lim::TMAX)), 0, int32_t(tiles.size())});
  std::vector<TileItem> items;
  for (const Tile &t : tiles) items.push_back({t.s, t.e});
  std::vector<int32_t> counts;
  while (!items.empty()) {
    if (rounds.size() > 40) throw std::runtime_error("tile splitting did not converge");
    rounds.push_back(std::make_unique<Round>());
    Round &r = *rounds.back();
    const size_t ni = items.size();
    r.items.ensure(ni);
    r.counts.ensure(ni * ITEM_COUNTS);
    r.halos.ensure(ni * size_t(Lim::LMAX));
    HIP_CHECK(hipMemcpyAsync(r.items.p, items.data(), ni * sizeof(TileItem), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL((k_halos<D, SMALL>), dim3(unsigned(ni)), dim3(B::HALO_THREADS), 0, s, tab, sum.p, r.items.p,
                       r.counts.p, r.halos.p);
    HIP_CHECK(hipGetLastError());
    counts.resize(ni * ITEM_COUNTS);
    HIP_CHECK(hipMemcpyAsync(counts.data(), r.counts.p, counts.size() * sizeof(int32_t), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    items.clear();
    const int32_t cur = int32_t(rounds.size()) - 1;
    bool any = false;
    for (size_t i = 0; i < ni && !any; ++i) any = counts[i * ITEM_COUNTS] < 0;
    if (!any) break;
    std::vector<Tile> next;
    next.reserve(tiles.size() + 16);
    for (const Tile &t : tiles) {
      if (t.round != cur || counts[size_t(t.item) * ITEM_COUNTS] >= 0) {
        next.push_back(t);
        continue;
      }
      if (t.e - t.s <= 1) throw std::runtime_error("a single node exceeds the tile limits");
      const int32_t m = t.s + (t.e - t.s) / 2;
      for (const TileItem &h : {TileItem{t.s, m}, TileItem{m, t.e}}) {
        next.push_back({h.s, h.e, cur + 1, int32_t(items.size())});
        items.push_back(h);
      }
    }
    tiles.swap(next);
  }
  return tiles;
}

template <int D, bool SMALL>
void build_tiles_of(const DTab<D> &tab, const DevBuf<NodeSum> &sum, DevBuf<BuildState> &dstate, BuildState &state,
                    casl_stencil *st, hipStream_t s) {
  using B = TileBlock<D, SMALL>;
  using Lim = TileLimits<D, SMALL>;
  const int64_t N = tab.N;
  const int flags = state.bad;
  std::vector<std::unique_ptr<Round>> rounds;
  const std::vector<Tile> tiles = cut_tiles<D, SMALL>(tab, sum, rounds, s);
  if (flags & BAD_NODE) throw std::runtime_error(bad_reason(BAD_NODE));

  // per-tile arrays and record counts
  const int nt = int(tiles.size());
  std::vector<TileSrc> srcs;
  srcs.reserve(tiles.size());
  for (const Tile &t : tiles) {
    const Round &r = *rounds[size_t(t.round)];
    srcs.push_back({r.counts.p + size_t(t.item) * ITEM_COUNTS, r.halos.p + size_t(t.item) * Lim::LMAX, t.s, 0});
  }
  DevBuf<TileSrc> src;
  src.ensure(size_t(nt));
  HIP_CHECK(hipMemcpyAsync(src.p, srcs.data(), size_t(nt) * sizeof(TileSrc), hipMemcpyHostToDevice, s));
  for (auto *x : {&st->t_tile_start, &st->t_urec_start, &st->t_rec_start, &st->t_ext_start, &st->t_halo_start})
    x->ensure(size_t(nt) + 1);
  st->t_nreg.ensure(size_t(nt));
  st->t_nuni.ensure(size_t(nt));
  st->t_h1count.ensure(size_t(nt));
  hipLaunchKernelGGL(k_tile_starts, dim3(1), dim3(SCAN_THREADS), 0, s, src.p, nt, int32_t(N),
                     TileStarts{st->t_tile_start.p, st->t_urec_start.p, st->t_rec_start.p, st->t_ext_start.p,
                                st->t_halo_start.p, st->t_h1count.p, st->t_nreg.p, st->t_nuni.p},
                     dstate.p);
  HIP_CHECK(hipGetLastError());
  read_state(dstate, state, s);
  const int64_t n_uni = state.n_uni, n_rec = state.n_rec, n_ext = state.n_ext, n_halo = state.n_halo;
  if (n_uni + n_rec >= int64_t(INT32_MAX) || n_halo >= int64_t(INT32_MAX))
    throw std::runtime_error("tile tables too large for int32 offsets");

  // records, and the independent bounds check before any other kernel reads them
  constexpr int UW = UniRec<D>::WORDS, XW = HangExt<D>::WORDS;
  st->t_rec.ensure(size_t(std::max<int64_t>(n_rec, 1)));
  st->t_rec_slot.ensure(size_t(std::max<int64_t>(n_rec, 1)));
  st->t_urec.ensure(size_t(std::max<int64_t>(n_uni * UW, 4)));
  st->t_ext.ensure(size_t(std::max<int64_t>(n_ext * XW, 16)));
  st->t_halo.ensure(size_t(std::max<int64_t>(n_halo, 1)));
  TileOut o{reinterpret_cast<TileRec *>(st->t_rec.p),
            st->t_rec_slot.p,
            st->t_urec.p,
            st->t_ext.p,
            st->t_halo.p,
            st->t_urec_start.p,
            st->t_rec_start.p,
            st->t_ext_start.p,
            st->t_halo_start.p};
  hipLaunchKernelGGL((k_records<D, SMALL>), dim3(unsigned(nt)), dim3(B::THREADS), 0, s, tab, sum.p, src.p, o,
                     dstate.p);
  HIP_CHECK(hipGetLastError());
  st->n_tiles = nt;
  st->n_halo = n_halo;
  st->n_records = n_uni + n_rec;
  st->n_uniform = n_uni;
  st->n_irregular = n_ext;
  st->small = SMALL;
  const Scales sc = scales_of<D>(state);
  for (int a = 0; a < 3; ++a) {
    st->geom_base[a] = sc.base[a];
    st->geom_unit[a] = sc.unit[a];
  }
  st->tiled = true;
  hipLaunchKernelGGL(k_validate<D>, dim3(unsigned(nt)), dim3(BLOCK), 0, s, tile_args<float>(st), N,
                     tile_caps(D, SMALL), &dstate.p->bad);
  HIP_CHECK(hipGetLastError());
  read_state(dstate, state, s);
  st->tiled = false;
  if (state.bad & ~ODD_WEIGHT) throw std::runtime_error(bad_reason(state.bad));
  st->regular_weights = (state.bad & ODD_WEIGHT) == 0;
  st->full_tiles = nt;
  if (SMALL && !st->dyadic_geometry()) {
    rounds.clear();
    st->full_tiles = int64_t(cut_tiles<D, false>(tab, sum, rounds, s).size());
  }
  st->tiled = true;
}

template <int D>
void make_stencil(const DTab<D> &t, casl_stencil *st, hipStream_t s) {
  const int64_t N = t.N;
  DevBuf<BuildState> dstate;
  DevBuf<NodeSum> sum;
  dstate.ensure(1);
  std::string no_room;
  try {
    sum.ensure(size_t(N));
  } catch (const std::bad_alloc &e) {  // the grid-wide tables alone
    no_room = e.what();
  }
  BuildState state{};
  for (auto &x : state.amin) x = 0x7ff0000000000000ull;  // +infinity
  HIP_CHECK(hipMemcpyAsync(dstate.p, &state, sizeof(BuildState), hipMemcpyHostToDevice, s));
  if (sum.p) {
    hipLaunchKernelGGL(k_arm_range<D>, dim3(reduce_grid(N)), dim3(BLOCK), 0, s, t, dstate.p);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((k_tables<D, true>), dim3(grid_for(N)), dim3(BLOCK), 0, s, t, st->nbr.p, st->wall.p,
                       st->dist.p, sum.p, dstate.p);
  } else {
    hipLaunchKernelGGL((k_tables<D, false>), dim3(grid_for(N)), dim3(BLOCK), 0, s, t, st->nbr.p, st->wall.p,
                       st->dist.p, nullptr, dstate.p);
  }
  HIP_CHECK(hipGetLastError());
  read_state(dstate, state, s);
  if (state.bad & BAD_INDEX) throw std::runtime_error("stencil node index out of range");
  if (state.bad & BAD_ZERO) throw std::runtime_error("zero face distance");
  if (state.bad & BAD_INEXACT) throw std::domain_error("stencil distance not exact in FP32");
  // the tiled encoding; where there is none the stencil keeps its grid-wide
  // tables and records why
  try {
    if (!sum.p) throw std::runtime_error(no_room);
    const Scales sc = scales_of<D>(state);
    if (!tile_scales_supported(sc.base, D))
      throw std::runtime_error("cells that are not cubes on a box whose edges are not dyadic");
    if (state.bad & BAD_SCALE) throw std::runtime_error(bad_reason(state.bad));
    if (small_tiles(D, N))
      build_tiles_of<D, true>(t, sum, dstate, state, st, s);
    else
      build_tiles_of<D, false>(t, sum, dstate, state, st, s);
  } catch (const hip_error &) {
    throw;
  } catch (const std::exception &e) {
    st->tiled = false;
    st->tile_error = e.what();
    return;
  }
  st->default_path();
}

}  // namespace

namespace casl {

void stencil_from_device_tables(const casl_flat_stencil &dtab, casl_stencil *st, hipStream_t s) {
  const int D = dtab.dim;
  if (D != 2 && D != 3) throw std::invalid_argument("dim must be 2 or 3");
  if (dtab.n_nodes <= 0 || dtab.n_nodes >= int64_t(INT32_MAX)) throw std::invalid_argument("bad n_nodes");
  const int64_t N = dtab.n_nodes;
  const int F = 2 * D, C = 1 << (D - 1), T = 2 * (D - 1);
  st->dim = D;
  st->N = N;
  st->zdt = dtab.zero_distance_threshold;
  HIP_CHECK(hipGetDevice(&st->device));
  st->tiled = false;
  st->nbr.ensure(size_t(F) * C * N);
  st->dist.ensure(size_t(F) * (1 + T) * N);
  st->wall.ensure(size_t(N));
  if (D == 2)
    make_stencil<2>(DTab<2>{dtab.nbr, dtab.d, dtab.d_tr, dtab.wall, N}, st, s);
  else
    make_stencil<3>(DTab<3>{dtab.nbr, dtab.d, dtab.d_tr, dtab.wall, N}, st, s);
}

}  // namespace casl
