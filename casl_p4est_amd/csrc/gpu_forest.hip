// Grid construction on the GPU: the single-tree forest refined by
// refine_levelset_cf, p4est's node numbering and construct_neighbors, so a
// changed level set does not send the grid through the host.
//
//   refinement      refine_levelset_cf applied level by level
//                   (src/my_p4est_refine_coarsen.cpp:17-89): one decision per
//                   quadrant, an exclusive scan of the refined counts, children
//                   written in place of their parent -- the leaves stay in
//                   Morton order, the order p4est's refine leaves them in
//   node numbering  my_p4est_nodes_new for one tree (src/my_p4est_nodes.c:
//                   383-446, 614-671): clamped corner keys; a node's index is
//                   its rank in their Morton order.  A corner that is some
//                   leaf's first corner has that leaf's key, and those keys are
//                   in order as they stand; only the others (hanging and upper
//                   wall nodes) are sorted, and the two lists merged by rank
//   neighbours      construct_neighbors (src/my_p4est_node_neighbors.cpp:114-1201):
//                   the cells around every node (leaf-corner scatter, else point
//                   location by binary search over the leaf keys), the finest
//                   cell per face, corner ids, distances, wall arms
// The arithmetic is that of the host construction (csrc/forest.cpp), so the
// tables are the same (the level-set values may differ in the last unit in
// the last place where they use sin, cos or atan2).
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include <cmath>
#include <memory>
#include <vector>

#include "reinit_device.hpp"

using namespace casl;

namespace {

constexpr int BLOCK = 256;
// One thread per item; a launch holds fewer than 2^32 work-items.
inline unsigned grid_for(int64_t n) {
  if (n >= (int64_t(1) << 32) - BLOCK) throw std::runtime_error("grid too large for one launch");
  return unsigned((n + BLOCK - 1) / BLOCK);
}

struct DQuad {
  int32_t c[3];
  int32_t level;
};

struct DevLS {
  int kind;
  int n_items;
  const double *p;  // device parameters
};

// The level sets of casl_levelset_eval, evaluated on the device.
__device__ double dev_levelset(const DevLS &ls, int dim, const double *x) {
  const double *p = ls.p;
  switch (ls.kind) {
    case CASL_LS_STAR: {
      double dx = x[0] - p[0], dy = x[1] - p[1];
      double r2 = dx * dx + dy * dy;
      double th = atan2(dy, dx);
      double r = p[2] + p[3] * cos(p[4] * th);
      return (sqrt(r2) - r) * (1.0 + p[5] * r2);
    }
    case CASL_LS_SPHERES: {
      double m = p[0];
      double best = HUGE_VAL;
      for (int i = 0; i < ls.n_items; ++i) {
        const double *s = p + 1 + 4 * i;
        double dx = x[0] - s[0], dy = x[1] - s[1], dz = x[2] - s[2];
        const double d2 = dx * dx + dy * dy + dz * dz;
        // Rounding is monotonic: where the root is at least best + r, v is
        // not below best and the root need not be taken.  The margin covers
        // the roundings of t * t and of the root; everything else (t not
        // positive, infinities, NaN) takes it.  k_sample on 64 spheres, 8.1M
        // nodes: 0.53 ms with every root, 0.34 without.
        const double t = best + s[3];
        if (t > 1e-100 && d2 > t * t * (1.0 + 0x1p-48)) continue;
        double v = sqrt(d2) - s[3];
        if (v < best) best = v;
      }
      return best * (1.0 + m * sin(2.0 * M_PI * x[0]) * cos(2.0 * M_PI * x[1]));
    }
    case CASL_LS_GYROID: {
      double w = p[0];
      double g = sin(w * x[0]) * cos(w * x[1]) + sin(w * x[1]) * cos(w * x[2]) + sin(w * x[2]) * cos(w * x[0]) - p[1];
      return g * (1.0 + p[2] * x[0] * x[1] * x[2]);
    }
    case CASL_LS_SPHERE: {
      double r2 = 0.0;
      for (int a = 0; a < dim; ++a) r2 += (x[a] - p[a]) * (x[a] - p[a]);
      return sqrt(r2) - p[dim];
    }
    case CASL_LS_PLANE: {
      double v = 0.0;
      for (int a = 0; a < dim; ++a) v += p[a] * x[a];
      return v + p[dim];
    }
    case CASL_LS_MODULATED: {
      double dx = x[0] - p[0], dy = x[1] - p[1];
      double e = sqrt(dx * dx + dy * dy) - p[2];
      return e * (1.0 + p[3] * sin(5.0 * x[0]) * cos(4.0 * x[1]));
    }
  }
  return 0.0;
}

template <int D>
struct Geo {
  static constexpr int MAXLEVEL = (D == 2 ? 30 : 19);
  static constexpr int32_t ROOT_LEN = int32_t(1) << MAXLEVEL;
  static constexpr int CH = 1 << D, F = 2 * D, C = 1 << (D - 1), T = 2 * (D - 1);
  double bmin[3], bmax[3];
  __host__ __device__ static int32_t qlen(int level) { return int32_t(1) << (MAXLEVEL - level); }
  __host__ __device__ double size(int a) const { return bmax[a] - bmin[a]; }
};

__device__ __forceinline__ uint64_t dspread2(uint32_t v) {
  uint64_t x = v;
  x = (x | (x << 16)) & 0x0000FFFF0000FFFFull;
  x = (x | (x << 8)) & 0x00FF00FF00FF00FFull;
  x = (x | (x << 4)) & 0x0F0F0F0F0F0F0F0Full;
  x = (x | (x << 2)) & 0x3333333333333333ull;
  x = (x | (x << 1)) & 0x5555555555555555ull;
  return x;
}
__device__ __forceinline__ uint32_t dcompact2(uint64_t x) {
  x &= 0x5555555555555555ull;
  x = (x | (x >> 1)) & 0x3333333333333333ull;
  x = (x | (x >> 2)) & 0x0F0F0F0F0F0F0F0Full;
  x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
  x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
  x = (x | (x >> 16)) & 0x00000000FFFFFFFFull;
  return uint32_t(x);
}
__device__ __forceinline__ uint64_t dspread3(uint32_t v) {
  uint64_t x = v & 0x1FFFFF;
  x = (x | (x << 32)) & 0x001F00000000FFFFull;
  x = (x | (x << 16)) & 0x001F0000FF0000FFull;
  x = (x | (x << 8)) & 0x100F00F00F00F00Full;
  x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
  x = (x | (x << 2)) & 0x1249249249249249ull;
  return x;
}
__device__ __forceinline__ uint32_t dcompact3(uint64_t x) {
  x &= 0x1249249249249249ull;
  x = (x | (x >> 2)) & 0x10C30C30C30C30C3ull;
  x = (x | (x >> 4)) & 0x100F00F00F00F00Full;
  x = (x | (x >> 8)) & 0x001F0000FF0000FFull;
  x = (x | (x >> 16)) & 0x001F00000000FFFFull;
  x = (x | (x >> 32)) & 0x00000000001FFFFFull;
  return uint32_t(x);
}
// bit b of axis a -> bit D*b + a (z outranks y outranks x at equal b)
template <int D>
__device__ __forceinline__ uint64_t dmorton(const int32_t *c) {
  if constexpr (D == 2)
    return dspread2(uint32_t(c[0])) | (dspread2(uint32_t(c[1])) << 1);
  else
    return dspread3(uint32_t(c[0])) | (dspread3(uint32_t(c[1])) << 1) | (dspread3(uint32_t(c[2])) << 2);
}
template <int D>
__device__ __forceinline__ void ddemorton(uint64_t k, int32_t *c) {
  if constexpr (D == 2) {
    c[0] = int32_t(dcompact2(k));
    c[1] = int32_t(dcompact2(k >> 1));
  } else {
    c[0] = int32_t(dcompact3(k));
    c[1] = int32_t(dcompact3(k >> 1));
    c[2] = int32_t(dcompact3(k >> 2));
  }
}

// The level set at the corners of a quadrant, x + (bit ? dx : 0).  Spheres: the
// same values as dev_levelset's, from the spheres that can be the nearest at
// some corner.  With B the least distance at the quadrant's middle and h its
// half diagonal, a sphere whose distance there exceeds B + 2 h is not below
// the least one at any corner; the margins are far above the roundings of
// these distances and of the middle, and whatever does not compare (NaN,
// infinities) is evaluated.  The modulation's factors are those of the
// quadrant's two abscissae and ordinates.  64 spheres, 8.1M nodes: k_decide
// 1.53 ms with all spheres at all corners, 0.56 so.
template <int D>
__device__ __forceinline__ void corner_values(const DevLS &ls, const double *x, const double *dx, double *f) {
  constexpr int CH = 1 << D;
  if constexpr (D == 3) {
    if (ls.kind == CASL_LS_SPHERES) {
      const double *p = ls.p;
      double c[3], h = 0.0, off = 0.0;
      for (int a = 0; a < 3; ++a) {
        c[a] = x[a] + 0.5 * dx[a];
        h += 0.25 * dx[a] * dx[a];
        off += fabs(c[a]);
      }
      h = sqrt(h) * (1.0 + 1e-6) + 1e-15 * off;
      auto dist2 = [](const double *q, const double *s) {
        const double ex = q[0] - s[0], ey = q[1] - s[1], ez = q[2] - s[2];
        return ex * ex + ey * ey + ez * ez;
      };
      double B = HUGE_VAL;
      for (int i = 0; i < ls.n_items; ++i) {
        const double *s = p + 1 + 4 * i;
        const double d2 = dist2(c, s), t = B + s[3];
        if (t > 1e-100 && d2 > t * t * (1.0 + 0x1p-48)) continue;
        const double v = sqrt(d2) - s[3];
        if (v < B) B = v;
      }
      double best[CH];
#pragma unroll
      for (int k = 0; k < CH; ++k) best[k] = HUGE_VAL;
      for (int i = 0; i < ls.n_items; ++i) {
        const double *s = p + 1 + 4 * i;
        const double t = B + s[3] + 2.0 * h + 1e-14 * (fabs(B) + fabs(s[3]));
        if (t > 1e-100 && dist2(c, s) > t * t * (1.0 + 1e-9)) continue;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
          double q[3];
          for (int a = 0; a < 3; ++a) q[a] = x[a] + ((k >> a) & 1) * dx[a];
          const double v = sqrt(dist2(q, s)) - s[3];
          if (v < best[k]) best[k] = v;
        }
      }
      const double m = p[0];
      double sn[2], cs[2];
      for (int b = 0; b < 2; ++b) {
        sn[b] = sin(2.0 * M_PI * (x[0] + b * dx[0]));
        cs[b] = cos(2.0 * M_PI * (x[1] + b * dx[1]));
      }
#pragma unroll
      for (int k = 0; k < CH; ++k) f[k] = best[k] * (1.0 + m * sn[k & 1] * cs[(k >> 1) & 1]);
      return;
    }
  }
  for (int k = 0; k < CH; ++k) {
    double xc[3];
    for (int a = 0; a < D; ++a) xc[a] = x[a] + ((k >> a) & 1) * dx[a];
    f[k] = dev_levelset(ls, D, xc);
  }
}

// ---------------------------------------------------------------- refinement
// refine_levelset_cf's decision (csrc/forest.cpp decide(), same arithmetic)
template <int D>
__device__ bool decide(const Geo<D> &G, const DQuad &q, int min_lvl, int max_lvl, double lip, double band_factor,
                       const DevLS &ls) {
  using GG = Geo<D>;
  if (q.level < min_lvl) return true;
  if (q.level >= max_lvl) return false;
  double dmin = (double)GG::qlen(q.level) / (double)GG::ROOT_LEN;
  double dx[3], x[3];
  for (int a = 0; a < D; ++a) dx[a] = G.size(a) * dmin;
  double smallest = fmax(G.size(0), G.size(1)) * ((double)GG::qlen(max_lvl)) / ((double)GG::ROOT_LEN);
  if (D == 3) smallest = fmax(smallest, G.size(2) * ((double)GG::qlen(max_lvl)) / ((double)GG::ROOT_LEN));
  double d2 = dx[0] * dx[0] + dx[1] * dx[1];
  if (D == 3) d2 = d2 + dx[2] * dx[2];
  double d = sqrt(d2);
  for (int a = 0; a < D; ++a) x[a] = G.size(a) * (double)q.c[a] / (double)GG::ROOT_LEN + G.bmin[a];
  double band = band_factor * smallest;
  double f[8];
  corner_values<D>(ls, x, dx, f);
  for (int k = 0; k < GG::CH; ++k)
    if (fabs(f[k]) - band <= 0.5 * lip * d) return true;
  if (D == 3) {
    if (f[0] * f[1] < 0 || f[0] * f[2] < 0 || f[1] * f[3] < 0 || f[2] * f[3] < 0 || f[3] * f[4] < 0 ||
        f[4] * f[5] < 0 || f[5] * f[6] < 0 || f[6] * f[7] < 0)
      return true;
  } else {
    if (f[0] * f[1] < 0 || f[0] * f[2] < 0 || f[1] * f[3] < 0 || f[2] * f[3] < 0) return true;
  }
  return false;
}

// Exclusive rank of the block's set flags (one per thread) and their count.
__device__ __forceinline__ int block_rank(bool set, int *count) {
  __shared__ int part[BLOCK / 64];
  const uint64_t m = __ballot(set);
  const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
  if (lane == 0) part[wave] = __popcll(m);
  __syncthreads();
  int r = __popcll(m & ((uint64_t(1) << lane) - 1)), c = 0;
#pragma unroll
  for (int w = 0; w < BLOCK / 64; ++w) {
    if (w < wave) r += part[w];
    c += part[w];
  }
  *count = c;
  return r;
}

// Pass p decides the quadrants of level p: a coarser leaf was decided in an
// earlier pass, and the decision depends on the quadrant alone.
template <int D>
__global__ void __launch_bounds__(BLOCK) k_decide(Geo<D> G, const DQuad *__restrict__ q, int64_t L, int pass,
                                                  int min_lvl, int max_lvl, double lip, double band, DevLS ls,
                                                  uint8_t *__restrict__ refine, int32_t *__restrict__ blk) {
  const int64_t l = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  const bool r = l < L && q[l].level == pass && q[l].level < Geo<D>::MAXLEVEL - 1 &&
                 decide<D>(G, q[l], min_lvl, max_lvl, lip, band, ls);
  if (l < L) refine[l] = r ? 1 : 0;
  int c = 0;
  (void)block_rank(r, &c);
  if (threadIdx.x == 0) blk[blockIdx.x] = c;
}

// Exclusive prefix of n counts in place by one block, and their total.
constexpr int SCAN_THREADS = 1024, SCAN_ITEMS = 4;
__global__ void __launch_bounds__(SCAN_THREADS) k_scan(int32_t *__restrict__ v, int64_t n,
                                                       int64_t *__restrict__ total) {
  __shared__ int64_t part[SCAN_THREADS / 64];
  const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
  int64_t base = 0;
  for (int64_t i0 = 0; i0 < n; i0 += SCAN_THREADS * SCAN_ITEMS) {
    const int64_t i = i0 + int64_t(threadIdx.x) * SCAN_ITEMS;
    int32_t x[SCAN_ITEMS];
    int64_t own = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
      x[k] = i + k < n ? v[i + k] : 0;
      own += x[k];
    }
    int64_t sum = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t y = __shfl_up(sum, unsigned(d), 64);
      if (lane >= d) sum += y;
    }
    __syncthreads();  // part[] was read by the row before
    if (lane == 63) part[wave] = sum;
    __syncthreads();
    int64_t at = base + sum - own;
#pragma unroll
    for (int w = 0; w < SCAN_THREADS / 64; ++w) {
      if (w < wave) at += part[w];
      base += part[w];
    }
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
      if (i + k < n) v[i + k] = int32_t(at);
      at += x[k];
    }
  }
  if (threadIdx.x == 0) *total = base;
}

template <int D>
__global__ void __launch_bounds__(BLOCK) k_emit(const DQuad *__restrict__ q, int64_t L,
                                                const uint8_t *__restrict__ refine, const int32_t *__restrict__ blk,
                                                DQuad *__restrict__ out) {
  const int64_t l = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  const bool r = l < L && refine[l] != 0;
  int c = 0;
  const int rank = block_rank(r, &c);
  if (l >= L) return;
  const DQuad p = q[l];
  const int64_t o = l + int64_t(Geo<D>::CH - 1) * (int64_t(blk[blockIdx.x]) + rank);
  if (!r) {
    out[o] = p;
    return;
  }
  const int32_t h = Geo<D>::qlen(p.level + 1);
  for (int k = 0; k < Geo<D>::CH; ++k) {
    DQuad n = p;
    n.level = p.level + 1;
    for (int a = 0; a < D; ++a) n.c[a] = p.c[a] + ((k >> a) & 1) * h;
    out[o + k] = n;
  }
}

// the uniform grid of one level, in Morton order
template <int D>
__global__ void k_uniform(int level, int64_t L, DQuad *__restrict__ q) {
  const int64_t l = int64_t(blockIdx.x) * BLOCK + threadIdx.x;
  if (l >= L) return;
  DQuad n{};
  n.level = level;
  ddemorton<D>(uint64_t(l) << (D * (Geo<D>::MAXLEVEL - level)), n.c);
  q[l] = n;
}

// ------------------------------------------------------------------ nodes
// the clamped key (p4est_node_clamp_inside) of corner k of a leaf
template <int D>
__device__ __forceinline__ uint64_t corner_key(const DQuad &q, int k) {
  const int32_t h = Geo<D>::qlen(q.level);
  int32_t p[3];
  for (int a = 0; a < D; ++a) {
    p[a] = q.c[a] + ((k >> a) & 1) * h;
    if (p[a] == Geo<D>::ROOT_LEN) p[a] = Geo<D>::ROOT_LEN - 1;
  }
  return dmorton<D>(p);
}

// first index in the ascending a[lo, hi) whose value is not below v
__device__ __forceinline__ int32_t lower_bound_u64(const uint64_t *__restrict__ a, int32_t lo, int32_t hi,
                                                   uint64_t v) {
  while (lo < hi) {
    const int32_t mid = int32_t((uint32_t(lo) + uint32_t(hi)) >> 1);
    if (a[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Ascending keys with the first of every prefix of TOP bits, so that a search
// spans the keys of one cell of level TOP / D: at most D (finest - TOP / D)
// steps, 9 on an octree of level 9, where a search of its 7.3M leaf keys takes
// 23.  Every leaf corner looked up: 0.55 ms, 1.18 among the 8.1M node keys
// without the prefixes.
template <int D>
struct KeyTable {
  static constexpr int TOP = 18, SHIFT = D * Geo<D>::MAXLEVEL - TOP;
  static constexpr int64_t ENTRIES = (int64_t(1) << TOP) + 2;  // v + 1 may pass the last key
  const uint64_t *__restrict__ key;
  const int32_t *__restrict__ top;  // [ENTRIES]
  int32_t n;
  // first index whose key is not below v
  __device__ int32_t lower(uint64_t v) const {
    const int64_t p = int64_t(v >> SHIFT);
    return lower_bound_u64(key, top[p], top[p + 1], v);
  }
  // the last key not above v (the leaf that holds point v)
  __device__ int32_t holding(uint64_t v) const { return lower(v + 1) - 1; }
};

template <int D>
__global__ void k_leaf_keys(const DQuad *__restrict__ q, int64_t L, uint64_t *__restrict__ keys,
                            uint8_t *__restrict__ level) {
  const int64_t l = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (l >= L) return;
  keys[l] = dmorton<D>(q[l].c);
  level[l] = uint8_t(q[l].level);
}

template <int D>
__global__ void k_top(const uint64_t *__restrict__ keys, int32_t n, int32_t *__restrict__ top) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < KeyTable<D>::ENTRIES) top[i] = lower_bound_u64(keys, 0, n, uint64_t(i) << KeyTable<D>::SHIFT);
}

// Which leaf's first corner every leaf corner is (-1: none), and how many are
// none per block.  The blocks stride over the corners, so their counts are few.
constexpr unsigned STRIDE_BLOCKS = 2048;
inline unsigned stride_grid(int64_t n) { return std::min(STRIDE_BLOCKS, grid_for(n)); }
template <int D>
__global__ void __launch_bounds__(BLOCK) k_owners(const DQuad *__restrict__ q, KeyTable<D> lk, int64_t K,
                                                  int32_t *__restrict__ local, int32_t *__restrict__ blk) {
  constexpr int CH = Geo<D>::CH;
  __shared__ int32_t none;
  if (threadIdx.x == 0) none = 0;
  __syncthreads();
  int32_t c = 0;
  for (int64_t i = int64_t(blockIdx.x) * BLOCK + threadIdx.x; i < K; i += int64_t(gridDim.x) * BLOCK) {
    const int32_t l = int32_t(i / CH);
    const int k = int(i % CH);
    int32_t m = l;
    if (k != 0) {
      const uint64_t v = corner_key<D>(q[l], k);
      m = lk.lower(v);
      if (m >= lk.n || lk.key[m] != v) {
        m = -1;
        ++c;
      }
    }
    local[i] = m;
  }
  if (c) atomicAdd(&none, c);
  __syncthreads();
  if (threadIdx.x == 0) blk[blockIdx.x] = none;
}

// The keys of the corners that are no leaf's first corner, in any order within
// the block's range.
template <int D>
__global__ void __launch_bounds__(BLOCK) k_extra_keys(const DQuad *__restrict__ q, int64_t K,
                                                      const int32_t *__restrict__ local,
                                                      const int32_t *__restrict__ blk, uint64_t *__restrict__ keys) {
  constexpr int CH = Geo<D>::CH;
  __shared__ int32_t next;
  if (threadIdx.x == 0) next = blk[blockIdx.x];
  __syncthreads();
  for (int64_t i = int64_t(blockIdx.x) * BLOCK + threadIdx.x; i < K; i += int64_t(gridDim.x) * BLOCK) {
    if (local[i] >= 0) continue;
    keys[atomicAdd(&next, 1)] = corner_key<D>(q[i / CH], int(i % CH));
  }
}

template <int D>
__device__ __forceinline__ void put_ixyz(int32_t *__restrict__ ixyz, int64_t n, const int32_t *c) {
  for (int a = 0; a < D; ++a) ixyz[n * D + a] = (c[a] == Geo<D>::ROOT_LEN - 1 ? Geo<D>::ROOT_LEN : c[a]);
}

// node index and coordinates of every leaf's first corner
template <int D>
__global__ void k_rank_leaves(const DQuad *__restrict__ q, KeyTable<D> lk, KeyTable<D> ek,
                              int32_t *__restrict__ node, int32_t *__restrict__ ixyz) {
  const int64_t l = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (l >= lk.n) return;
  const int32_t n = int32_t(l) + ek.lower(lk.key[l]);
  node[l] = n;
  put_ixyz<D>(ixyz, n, q[l].c);
}

// and of every other node
template <int D>
__global__ void k_rank_extra(KeyTable<D> lk, KeyTable<D> ek, int32_t *__restrict__ node,
                             int32_t *__restrict__ ixyz) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= ek.n) return;
  const int32_t n = int32_t(e) + lk.lower(ek.key[e]);
  node[e] = n;
  int32_t c[3];
  ddemorton<D>(ek.key[e], c);
  put_ixyz<D>(ixyz, n, c);
}

// each leaf corner's node, and the cell at that corner: leaf l is the cell in
// direction k ^ (CH - 1) of its corner k's node
template <int D>
__global__ void k_local_nodes(const DQuad *__restrict__ q, int64_t K, const int32_t *__restrict__ leaf_node,
                              KeyTable<D> ek, const int32_t *__restrict__ extra_node, int32_t *__restrict__ local,
                              int32_t *__restrict__ cell) {
  constexpr int CH = Geo<D>::CH;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= K) return;
  const int32_t l = int32_t(i / CH), m = local[i];
  const int k = int(i % CH);
  const int32_t n = m >= 0 ? leaf_node[m] : extra_node[ek.lower(corner_key<D>(q[l], k))];
  local[i] = n;
  cell[int64_t(n) * CH + (k ^ (CH - 1))] = l;
}

// ------------------------------------------------------------- neighbours
__global__ void k_fill_i32(int32_t *p, int64_t n, int32_t v) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

constexpr int32_t CELL_NONE = -1, CELL_UNSET = -2;  // outside the tree; not at a corner of its leaf

// the leaf in direction dir of a node at c whose slot is not set
template <int D>
__device__ __forceinline__ int32_t locate(const KeyTable<D> &lk, const int32_t *c, int dir) {
  int32_t p[3];
  for (int a = 0; a < D; ++a) {
    p[a] = c[a] + (((dir >> a) & 1) ? 1 : -1);
    if (p[a] < 0 || p[a] >= Geo<D>::ROOT_LEN) return CELL_NONE;
  }
  return lk.holding(dmorton<D>(p));
}

template <int D>
struct NbrOut {
  int32_t *nbr;
  double *dface, *dtr;
  uint8_t *wall;
  int *bad;
};

// The corners of the cell a face's arm ends at, and the node's offsets in it.
template <int D>
__device__ __forceinline__ void fill_from_cell(const Geo<D> &G, const DQuad &Q, const int32_t *__restrict__ corners,
                                               const int32_t *x, int64_t N, int64_t n, int f, int side,
                                               const NbrOut<D> &o) {
  using GG = Geo<D>;
  const int a = f >> 1;
  int t1, t2;
  if (D == 2) {
    t1 = 1 - a;
    t2 = -1;
  } else {
    t1 = (a == 0 ? 1 : 0);
    t2 = (a == 2 ? 1 : 2);
  }
#pragma unroll
  for (int c = 0; c < GG::C; ++c) {
    int corner = (side << a) | ((c & 1) << t1);
    if (D == 3) corner |= ((c >> 1) & 1) << t2;
    o.nbr[(int64_t(f) * GG::C + c) * N + n] = corners[corner];
  }
  const double qh = GG::qlen(Q.level) / (double)GG::ROOT_LEN;
#pragma unroll
  for (int t = 0; t < D - 1; ++t) {
    const int ax = (t == 0 ? t1 : t2);
    const double thr = G.size(ax) * ((double)1) / ((double)GG::ROOT_LEN);
    const double X = G.size(ax) * (x[ax] / (double)GG::ROOT_LEN) + G.bmin[ax];
    const double QX = G.size(ax) * (Q.c[ax] / (double)GG::ROOT_LEN) + G.bmin[ax];
    const double m0 = (fabs(X - QX) > thr) ? (X - QX) : 0.0;
    const double p0 = (fabs(G.size(ax) * qh - m0) > thr) ? (G.size(ax) * qh - m0) : 0.0;
    o.dtr[(int64_t(f) * GG::T + 2 * t + 0) * N + n] = m0;
    o.dtr[(int64_t(f) * GG::T + 2 * t + 1) * N + n] = p0;
  }
}

// One thread per node: its cells and their levels stay in registers, the
// finest cell of every face is picked from them, and each face reads one leaf
// and its row of corners.  337 bytes are written per node (3D) and about 80
// gathered: 8.1M nodes 1.33 ms (2.5 TB/s; 1.47 with 8 waves per SIMD instead of
// 4, whose gathers push each other out of the caches); with the cells read
// again for every face 1.91, and 0.82 more for a pass that located those not at
// a corner of their leaf one by one.
template <int D>
__global__ void __launch_bounds__(BLOCK) k_construct(Geo<D> G, const DQuad *__restrict__ leaves, KeyTable<D> lk,
                                                     const uint8_t *__restrict__ level,
                                                     const int32_t *__restrict__ local,
                                                     const int32_t *__restrict__ ixyz,
                                                     const int32_t *__restrict__ cell, int64_t N, NbrOut<D> o) {
  using GG = Geo<D>;
  constexpr int F = GG::F, CH = GG::CH;
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= N) return;
  int32_t x[D];
#pragma unroll
  for (int a = 0; a < D; ++a) x[a] = ixyz[n * D + a];
  int32_t cn[CH];
  int lv[CH];
#pragma unroll
  for (int dir = 0; dir < CH; ++dir) cn[dir] = cell[n * CH + dir];
  // the slots not set: outside the tree, or in a coarser leaf that often
  // holds several of them
  uint32_t unset = 0;
#pragma unroll
  for (int dir = 0; dir < CH; ++dir) {
    if (cn[dir] != CELL_UNSET) continue;
    bool inside = true;
#pragma unroll
    for (int a = 0; a < D; ++a) inside = inside && (((dir >> a) & 1) ? x[a] < GG::ROOT_LEN - 1 : x[a] > 0);
    if (inside)
      unset |= 1u << dir;
    else
      cn[dir] = CELL_NONE;
  }
  while (unset) {
    const int first = __ffs(int(unset)) - 1;
    const int32_t l = locate<D>(lk, x, first);
    const DQuad Q = leaves[l];
    const int32_t h = GG::qlen(Q.level);
#pragma unroll
    for (int dir = 0; dir < CH; ++dir) {
      bool in = ((unset >> dir) & 1u) != 0;
#pragma unroll
      for (int a = 0; a < D; ++a) {
        const int32_t v = x[a] + (((dir >> a) & 1) ? 1 : -1) - Q.c[a];
        in = in && v >= 0 && v < h;
      }
      if (in || dir == first) {
        cn[dir] = l;
        unset &= ~(1u << dir);
      }
    }
  }
#pragma unroll
  for (int dir = 0; dir < CH; ++dir) lv[dir] = cn[dir] < 0 ? -1 : int(level[cn[dir]]);
  double df[F];
  uint32_t walls = 0;  // faces without a cell
#pragma unroll
  for (int f = 0; f < F; ++f) {
    const int a = f >> 1, s = f & 1;
    int best = -2;
    int32_t qi = -1;
#pragma unroll
    for (int dir = 0; dir < CH; ++dir) {
      if (((dir >> a) & 1) != s) continue;
      if (lv[dir] > best) {  // finest cell, first wins on ties
        best = lv[dir];
        qi = cn[dir];
      }
    }
    df[f] = 0.0;
    if (qi < 0) {
      walls |= 1u << f;
      continue;
    }
    df[f] = G.size(a) * (GG::qlen(best) / (double)GG::ROOT_LEN);
    o.dface[int64_t(f) * N + n] = df[f];
    fill_from_cell<D>(G, leaves[qi], local + int64_t(qi) * CH, x, N, n, f, s == 0 ? 0 : 1, o);
  }
  if (walls) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      if (!((walls >> f) & 1u)) continue;
      const int a = f >> 1, s = f & 1, so = 1 - s;
      int dmin = -1, lbest = -1;
      int32_t qmin = -1;
#pragma unroll
      for (int dir = 0; dir < CH; ++dir) {
        if (((dir >> a) & 1) != so) continue;
        if (lbest < lv[dir]) {
          lbest = lv[dir];
          dmin = dir;
          qmin = cn[dir];
        }
      }
      if (dmin < 0) {
        *o.bad = 1;
        return;
      }
      int corner = so << a;
      for (int b = 0; b < D; ++b)
        if (b != a) corner |= (((dmin >> b) & 1) ? 0 : 1) << b;
      const int32_t ntmp = local[int64_t(qmin) * CH + corner];
      int32_t qtmp = cell[int64_t(ntmp) * CH + dmin];
      if (qtmp == CELL_UNSET) {
        int32_t y[D];
        for (int b = 0; b < D; ++b) y[b] = ixyz[int64_t(ntmp) * D + b];
        qtmp = locate<D>(lk, y, dmin);
      }
      if (qtmp < 0) {
        *o.bad = 1;
        return;
      }
      df[f] = -df[f ^ 1] - G.size(a) * (GG::qlen(level[qtmp]) / (double)GG::ROOT_LEN);
      o.dface[int64_t(f) * N + n] = df[f];
      fill_from_cell<D>(G, leaves[qtmp], local + int64_t(qtmp) * CH, x, N, n, f, so, o);
    }
  }
  uint8_t w = 0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    if (x[a] == 0) w |= uint8_t(1u << (2 * a));
    if (x[a] == GG::ROOT_LEN - 1 || x[a] == GG::ROOT_LEN) w |= uint8_t(1u << (2 * a + 1));
  }
  o.wall[n] = w;
}

template <int D>
__global__ void k_sample(Geo<D> G, const int32_t *__restrict__ ixyz, int64_t N, DevLS ls, double *__restrict__ out) {
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= N) return;
  double x[3];
  for (int a = 0; a < D; ++a) x[a] = G.size(a) * (ixyz[n * D + a] / (double)Geo<D>::ROOT_LEN) + G.bmin[a];
  out[n] = dev_levelset(ls, D, x);
}

int ls_param_count(const casl_levelset &ls, int dim) {
  switch (ls.kind) {
    case CASL_LS_STAR:
      if (dim != 2) throw std::invalid_argument("star level set is 2D");
      return 6;
    case CASL_LS_SPHERES:
      if (dim != 3) throw std::invalid_argument("spheres level set is 3D");
      if (ls.n_items < 0) throw std::invalid_argument("negative sphere count");
      return 1 + 4 * ls.n_items;
    case CASL_LS_GYROID:
      if (dim != 3) throw std::invalid_argument("gyroid level set is 3D");
      return 3;
    case CASL_LS_SPHERE:
    case CASL_LS_PLANE:
      return dim + 1;
    case CASL_LS_MODULATED:
      if (dim != 2) throw std::invalid_argument("modulated level set is 2D");
      return 4;
    case CASL_LS_CALLBACK:
      throw std::invalid_argument("host callbacks cannot be evaluated on the device");
  }
  throw std::invalid_argument("unknown level-set kind");
}

// device copy of a level set's parameters
struct DevLSHolder {
  casl::DevBuf<double> p;
  DevLS ls{};
  DevLSHolder(const casl_levelset *src, int dim) {
    if (!src || !src->params) throw std::invalid_argument("null level set");
    const int np = ls_param_count(*src, dim);
    p.ensure(size_t(np));
    HIP_CHECK(hipMemcpy(p.p, src->params, size_t(np) * sizeof(double), hipMemcpyHostToDevice));
    ls.kind = src->kind;
    ls.n_items = src->n_items;
    ls.p = p.p;
  }
};

}  // namespace

struct casl_device_grid {
  int dim = 0;
  int64_t L = 0, N = 0;
  int max_level = 0;
  double bmin[3] = {0, 0, 0}, bmax[3] = {1, 1, 1};
  double zdt = 0;
  casl::DevBuf<DQuad> leaves;
  casl::DevBuf<int32_t> ixyz, nbr;
  casl::DevBuf<double> dface, dtr;
  casl::DevBuf<uint8_t> wall;
};

namespace {

// A hipCUB device-wide call with its own temporary storage, which stays
// allocated until the call has finished on the stream.
template <class Fn>
void cub_call(hipStream_t s, Fn fn) {
  size_t bytes = 0;
  HIP_CHECK(fn(nullptr, bytes));
  casl::DevBuf<unsigned char> tmp;
  tmp.ensure(std::max<size_t>(bytes, 1));
  HIP_CHECK(fn(tmp.p, bytes));
  HIP_CHECK(hipStreamSynchronize(s));
}

int64_t read_total(const casl::DevBuf<int64_t> &total, hipStream_t s) {
  int64_t v = 0;
  HIP_CHECK(hipMemcpyAsync(&v, total.p, sizeof(v), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  return v;
}

template <int D>
void build_grid(casl_device_grid *g, int min_lvl, int max_lvl, double lip, double band, const DevLS &ls,
                hipStream_t s) {
  using GG = Geo<D>;
  constexpr int CH = GG::CH;
  if (max_lvl >= GG::MAXLEVEL - 1) throw std::invalid_argument("max_lvl too large for this dimension");
  if (min_lvl < 0 || max_lvl < 0) throw std::invalid_argument("negative levels");
  Geo<D> G;
  for (int a = 0; a < 3; ++a) {
    G.bmin[a] = g->bmin[a];
    G.bmax[a] = g->bmax[a];
  }
  // refinement: every quadrant coarser than min_lvl is refined, then level by level
  casl::DevBuf<DQuad> q, q2;
  casl::DevBuf<uint8_t> refine;
  casl::DevBuf<int32_t> blk;
  casl::DevBuf<int64_t> total;
  total.ensure(1);
  const int first = std::min(min_lvl, GG::MAXLEVEL - 1);
  if (D * first >= 31) throw std::runtime_error("too many leaves for int32 indices");
  int64_t L = int64_t(1) << (D * first);
  int finest = first;
  q.ensure(size_t(L));
  hipLaunchKernelGGL(k_uniform<D>, dim3(grid_for(L)), dim3(BLOCK), 0, s, first, L, q.p);
  HIP_CHECK(hipGetLastError());
  for (int pass = first; pass < GG::MAXLEVEL; ++pass) {
    refine.ensure(size_t(L));
    blk.ensure(std::max<size_t>(grid_for(L), STRIDE_BLOCKS));
    hipLaunchKernelGGL(k_decide<D>, dim3(grid_for(L)), dim3(BLOCK), 0, s, G, q.p, L, pass, min_lvl, max_lvl, lip, band,
                       ls, refine.p, blk.p);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(SCAN_THREADS), 0, s, blk.p, int64_t(grid_for(L)), total.p);
    HIP_CHECK(hipGetLastError());
    const int64_t refined = read_total(total, s);
    if (refined == 0) break;  // done
    const int64_t L2 = L + int64_t(CH - 1) * refined;
    if (L2 >= int64_t(INT32_MAX)) throw std::runtime_error("too many leaves for int32 indices");
    q2.ensure(size_t(L2));
    hipLaunchKernelGGL(k_emit<D>, dim3(grid_for(L)), dim3(BLOCK), 0, s, q.p, L, refine.p, blk.p, q2.p);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s));  // the next pass may release what the emission reads
    q.swap(q2);
    L = L2;
    finest = pass + 1;
  }
  q2.release();
  refine.release();
  // node numbering
  const int64_t K = L * CH;  // may exceed 2^31
  casl::DevBuf<uint64_t> leaf_keys;
  casl::DevBuf<uint8_t> level;
  casl::DevBuf<int32_t> top, local;
  leaf_keys.ensure(size_t(L));
  level.ensure(size_t(L));
  top.ensure(size_t(KeyTable<D>::ENTRIES));
  local.ensure(size_t(K));
  hipLaunchKernelGGL(k_leaf_keys<D>, dim3(grid_for(L)), dim3(BLOCK), 0, s, q.p, L, leaf_keys.p, level.p);
  hipLaunchKernelGGL(k_top<D>, dim3(grid_for(KeyTable<D>::ENTRIES)), dim3(BLOCK), 0, s, leaf_keys.p, int32_t(L),
                     top.p);
  const KeyTable<D> lk{leaf_keys.p, top.p, int32_t(L)};
  const unsigned sb = stride_grid(K);
  hipLaunchKernelGGL(k_owners<D>, dim3(sb), dim3(BLOCK), 0, s, q.p, lk, K, local.p, blk.p);
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(SCAN_THREADS), 0, s, blk.p, int64_t(sb), total.p);
  HIP_CHECK(hipGetLastError());
  const int64_t raw = read_total(total, s);
  if (raw >= int64_t(INT32_MAX)) throw std::runtime_error("too many hanging nodes for int32 indices");
  int64_t E = 0;
  casl::DevBuf<uint64_t> ka, kb;
  ka.ensure(size_t(std::max<int64_t>(raw, 1)));
  kb.ensure(size_t(std::max<int64_t>(raw, 1)));
  hipLaunchKernelGGL(k_extra_keys<D>, dim3(sb), dim3(BLOCK), 0, s, q.p, K, local.p, blk.p, ka.p);
  HIP_CHECK(hipGetLastError());
  // Every corner coordinate is a multiple of 2^z, z = MAXLEVEL - finest,
  // or ROOT_LEN - 1 (clamped): its low z bits are all 0 or all 1, so bit
  // z - 1 fixes the z - 1 bits below it.  Keys that agree from bit
  // D (z - 1) up are equal, and the sort can start there.
  const int end_bit = D * GG::MAXLEVEL, begin_bit = D * (GG::MAXLEVEL - finest - 1);
  hipcub::DoubleBuffer<uint64_t> db;
  cub_call(s, [&](void *t, size_t &b) {
    db = hipcub::DoubleBuffer<uint64_t>(ka.p, kb.p);  // the size query and the sort both start from ka
    return hipcub::DeviceRadixSort::SortKeys(t, b, db, raw, begin_bit, end_bit, s);
  });
  uint64_t *extra = db.Alternate();
  cub_call(s, [&](void *t, size_t &b) {
    return hipcub::DeviceSelect::Unique(t, b, db.Current(), extra, total.p, raw, s);
  });
  E = read_total(total, s);
  const int64_t N = L + E;
  if (N >= int64_t(INT32_MAX)) throw std::runtime_error("too many nodes for int32 indices");
  casl::DevBuf<int32_t> leaf_node, extra_node, cell, extra_top;
  casl::DevBuf<int> bad;
  leaf_node.ensure(size_t(L));
  extra_node.ensure(size_t(E));
  g->ixyz.ensure(size_t(N) * D);
  cell.ensure(size_t(N) * CH);
  bad.ensure(1);
  extra_top.ensure(size_t(KeyTable<D>::ENTRIES));
  hipLaunchKernelGGL(k_top<D>, dim3(grid_for(KeyTable<D>::ENTRIES)), dim3(BLOCK), 0, s, extra, int32_t(E),
                     extra_top.p);
  const KeyTable<D> ek{extra, extra_top.p, int32_t(E)};
  hipLaunchKernelGGL(k_rank_leaves<D>, dim3(grid_for(L)), dim3(BLOCK), 0, s, q.p, lk, ek, leaf_node.p, g->ixyz.p);
  hipLaunchKernelGGL(k_rank_extra<D>, dim3(grid_for(E)), dim3(BLOCK), 0, s, lk, ek, extra_node.p, g->ixyz.p);
  hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(N * CH)), dim3(BLOCK), 0, s, cell.p, N * CH, CELL_UNSET);
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(1), 0, s, reinterpret_cast<int32_t *>(bad.p), int64_t(1), 0);
  hipLaunchKernelGGL(k_local_nodes<D>, dim3(grid_for(K)), dim3(BLOCK), 0, s, q.p, K, leaf_node.p, ek, extra_node.p,
                     local.p, cell.p);
  HIP_CHECK(hipGetLastError());
  ka.release();
  kb.release();
  leaf_node.release();
  extra_node.release();
  // neighbours
  g->nbr.ensure(size_t(GG::F) * GG::C * N);
  g->dface.ensure(size_t(GG::F) * N);
  g->dtr.ensure(size_t(GG::F) * GG::T * N);
  g->wall.ensure(size_t(N));
  NbrOut<D> o{g->nbr.p, g->dface.p, g->dtr.p, g->wall.p, bad.p};
  hipLaunchKernelGGL(k_construct<D>, dim3(grid_for(N)), dim3(BLOCK), 0, s, G, q.p, lk, level.p, local.p, g->ixyz.p,
                     cell.p, N, o);
  HIP_CHECK(hipGetLastError());
  int hbad = 0;
  HIP_CHECK(hipMemcpyAsync(&hbad, bad.p, sizeof(int), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  if (hbad) throw std::runtime_error("construct_neighbors: a wall arm has no second-degree cell");
  // keep the leaves (the refinement's buffer, handed over); the finest level present
  g->leaves.release();
  g->leaves.swap(q);
  g->L = L;
  g->N = N;
  g->max_level = finest;
}

}  // namespace

extern "C" {

int casl_device_grid_build(int dim, const double *box_min, const double *box_max, int min_lvl, int max_lvl,
                           double lip, double band, const casl_levelset *ls, void *stream,
                           casl_device_grid_t **out) {
  return guarded([&]() {
    if (!out) throw std::invalid_argument("null output");
    *out = nullptr;
    if (dim != 2 && dim != 3) throw std::invalid_argument("dim must be 2 or 3");
    auto g = std::make_unique<casl_device_grid>();
    g->dim = dim;
    double m = 0;
    for (int a = 0; a < dim; ++a) {
      g->bmin[a] = box_min ? box_min[a] : 0.0;
      g->bmax[a] = box_max ? box_max[a] : 1.0;
      if (!(g->bmax[a] > g->bmin[a])) throw std::invalid_argument("empty box");
      const double sz = g->bmax[a] - g->bmin[a];
      m = (a == 0) ? sz : std::min(m, sz);
    }
    g->zdt = 1e-13 * m;
    DevLSHolder h(ls, dim);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dim == 2)
      build_grid<2>(g.get(), min_lvl, max_lvl, lip, band, h.ls, s);
    else
      build_grid<3>(g.get(), min_lvl, max_lvl, lip, band, h.ls, s);
    *out = g.release();
  });
}

int casl_device_grid_destroy(casl_device_grid_t *g) {
  delete g;
  return CASL_OK;
}

int casl_device_grid_sizes(const casl_device_grid_t *g, int64_t *n_leaves, int64_t *n_nodes, int32_t *max_level) {
  return guarded([&]() {
    if (!g) throw std::invalid_argument("null grid");
    if (n_leaves) *n_leaves = g->L;
    if (n_nodes) *n_nodes = g->N;
    if (max_level) *max_level = g->max_level;
  });
}

int casl_device_grid_tables(const casl_device_grid_t *g, casl_flat_stencil *out) {
  return guarded([&]() {
    if (!g || !out) throw std::invalid_argument("null argument");
    out->dim = g->dim;
    out->n_nodes = g->N;
    out->nbr = g->nbr.p;
    out->d = g->dface.p;
    out->d_tr = g->dtr.p;
    out->wall = g->wall.p;
    out->zero_distance_threshold = g->zdt;
  });
}

int casl_device_grid_download(const casl_device_grid_t *g, int32_t *nbr, double *d, double *d_tr, uint8_t *wall,
                              int32_t *ixyz) {
  return guarded([&]() {
    if (!g) throw std::invalid_argument("null grid");
    const int D = g->dim, F = 2 * D, C = 1 << (D - 1), T = 2 * (D - 1);
    const size_t N = size_t(g->N);
    if (nbr) HIP_CHECK(hipMemcpy(nbr, g->nbr.p, size_t(F) * C * N * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (d) HIP_CHECK(hipMemcpy(d, g->dface.p, size_t(F) * N * sizeof(double), hipMemcpyDeviceToHost));
    if (d_tr) HIP_CHECK(hipMemcpy(d_tr, g->dtr.p, size_t(F) * T * N * sizeof(double), hipMemcpyDeviceToHost));
    if (wall) HIP_CHECK(hipMemcpy(wall, g->wall.p, N, hipMemcpyDeviceToHost));
    if (ixyz) HIP_CHECK(hipMemcpy(ixyz, g->ixyz.p, size_t(D) * N * sizeof(int32_t), hipMemcpyDeviceToHost));
  });
}

int casl_device_grid_sample(const casl_device_grid_t *g, const casl_levelset *ls, double *phi, void *stream) {
  return guarded([&]() {
    if (!g || !phi) throw std::invalid_argument("null argument");
    DevLSHolder h(ls, g->dim);
    Geo<2> G2;
    Geo<3> G3;
    for (int a = 0; a < 3; ++a) {
      G2.bmin[a] = G3.bmin[a] = g->bmin[a];
      G2.bmax[a] = G3.bmax[a] = g->bmax[a];
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (g->dim == 2)
      hipLaunchKernelGGL(k_sample<2>, dim3(grid_for(g->N)), dim3(BLOCK), 0, s, G2, g->ixyz.p, g->N, h.ls, phi);
    else
      hipLaunchKernelGGL(k_sample<3>, dim3(grid_for(g->N)), dim3(BLOCK), 0, s, G3, g->ixyz.p, g->N, h.ls, phi);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(s));  // the parameter copy lives until here
  });
}

int casl_device_grid_stencil(const casl_device_grid_t *g, casl_stencil_t **out) {
  return guarded([&]() {
    if (!g || !out) throw std::invalid_argument("null argument");
    *out = nullptr;
    // the grid-wide tables and the tiled encoding, both from the grid's device
    // tables: nothing travels to the host but a few counts
    casl_flat_stencil tab{};
    tab.dim = g->dim;
    tab.n_nodes = g->N;
    tab.nbr = g->nbr.p;
    tab.d = g->dface.p;
    tab.d_tr = g->dtr.p;
    tab.wall = g->wall.p;
    tab.zero_distance_threshold = g->zdt;
    auto st = std::make_unique<casl_stencil>();
    stencil_from_device_tables(tab, st.get(), nullptr);
    HIP_CHECK(hipStreamSynchronize(nullptr));
    *out = st.release();
  });
}

}  // extern "C"
