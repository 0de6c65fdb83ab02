// Learned-curvature inputs on the adaptive grid, for 2D and 3D trees.
//
// The reference's learned curvature (kml::Curvature, src/my_p4est_curvature_ml.cpp)
// is 2D and reads 3x3 phi stencils of uniform-grid nodes next to the
// interface.  Here the same inputs come from any grid, through the
// construct_neighbors tables: for every node with |phi| < band, the block of
// 3^dim nodes at spacing h around it is found by walking face neighbours
// (x, then y, then z), every arm on the way being exactly h long and ending
// on a node (a zero transverse distance along every transverse axis).  A
// node without such a block keeps the numerical value; it is counted, not
// sampled.
//
//   features  phi/h over the block (x slowest, z fastest: the 2D order of
//             src/my_p4est_curvature_ml.h:49-60 extended by one axis), then
//             h*kappa interpolated (bi/trilinearly, inside the block) at the
//             projection x - phi n of the node onto the interface ("ihk",
//             src/my_p4est_curvature_ml.cpp:414-480), kappa being
//             compute_mean_curvature's div(n) and n compute_normals' output
//   3D normalisation  negate when ihk > 0; reflect every axis along which the
//             centred difference of phi is negative; order the axes by
//             decreasing difference.  Every one of the 48 symmetries of the
//             cube maps a stencil to the same input: the 3D counterpart of the
//             2D rotation to the first quadrant plus y = x reflection
//             (:327-398), with one row per sample instead of two.  The 27
//             values then go to a basis that BF16 inputs resolve: the centre
//             value, the half centred differences, and the deviations from
//             the plane through the centre with those slopes.
//   3D hybrid  as the 2D one (:483-556): numerical value where |ihk| < lo,
//             blend towards it up to hi, sign of ihk; a residual network's
//             corrections at most `deadband` in size are dropped.
#include <hip/hip_runtime.h>

#include <cmath>

#include "curv_device.hpp"
#include "reinit_device.hpp"
#include "tiles_device.hpp"

using namespace casl;
using namespace casl::dev;

namespace {

constexpr int BLOCK = 256;

inline unsigned grid_for(int64_t n) { return unsigned((n + BLOCK - 1) / BLOCK); }

template <int D>
struct Block {
  static constexpr int Q = (D == 2 ? 9 : 27);
  static constexpr int NF = Q + 1;
  // position of offsets (i, j[, k]) in {-1, 0, 1}^D, x slowest
  __host__ __device__ static constexpr int q(int i, int j, int k = 0) {
    return D == 2 ? 3 * (i + 1) + (j + 1) : 9 * (i + 1) + 3 * (j + 1) + (k + 1);
  }
};

// the arm of node n through face f if it is exactly h long and ends on a
// node (else -1): along every transverse axis one of the two transverse
// distances is zero, and the face corner on that side is the node
template <int D>
__device__ __forceinline__ int32_t arm(const Tables<D> &t, int f, int64_t n, float h) {
  if (t.d(f, n) != h) return -1;
  int c = 0;
#pragma unroll
  for (int k = 0; k < D - 1; ++k) {
    if (t.dt(f, 2 * k, n) == 0.f) {
      // corner bit 0 along this axis
    } else if (t.dt(f, 2 * k + 1, n) == 0.f) {
      c |= 1 << k;
    } else {
      return -1;
    }
  }
  return t.idx(f, c, n);
}

// Samples are found and written through one table of arms, arms[f][n]: the
// walk over a block takes 26 of them in 3D, and reading each from the
// stencil tables costs five scattered loads.  k_arms reads the grid-wide
// tables once in order (216 bytes a node in 3D); k_tile_arms reads the tile
// records instead (16 bytes a node), where a face's arm is h long when its
// level is h's, it is no wall arm, and it does not hang.
template <int D>
__global__ void __launch_bounds__(BLOCK) k_arms(Tables<D> t, float h, int32_t *__restrict__ arms) {
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= t.N) return;
#pragma unroll
  for (int f = 0; f < 2 * D; ++f) arms[int64_t(f) * t.N + n] = arm<D>(t, f, n, h);
}

struct AxisLevels {
  int l[3];  // the level whose arm cells are h long, per axis; -1: none
};

template <int D>
__global__ void __launch_bounds__(BLOCK)
    k_tile_arms(TileArgs<float> A, AxisLevels lv, int32_t *__restrict__ arms) {
  constexpr int F = 2 * D;
  TileCtx<D> c;
  c.load(A, xcd_tile(int(blockIdx.x), int(gridDim.x)));
  for (int i = int(threadIdx.x); i < c.nT; i += BLOCK) {
    RecRegs r;
    int j = fetch_record<D>(A, c, i, r);
    const TileRec rec = record_at<D>(c, i, r, j);
    int h0 = F, h1 = F;  // the faces that hang
    if (rec.geo & GEO_IRREGULAR) {
      const uint16_t *e = c.ext_of(A.ext, i);
      h0 = D == 2 ? int(e[0]) : int(e[0] & 15);
      if (D == 3) h1 = int((e[0] >> 4) & 15);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const bool ok = int((rec.geo >> (4 * f)) & 15u) == lv.l[f >> 1] && !((rec.geo >> (24 + f)) & 1u) && f != h0 &&
                      f != h1;
      const int q = rec.idx[f];
      arms[int64_t(f) * A.N + c.s + j] = !ok ? -1 : (q < c.nT ? c.s + q : A.halo[c.hb + (q - c.nT)]);
    }
  }
}

// The block of node n by its arms (x, then y, then z); false where an arm is
// missing.
template <int D>
__device__ __forceinline__ bool gather_block(const int32_t *__restrict__ arms, int64_t N, int64_t n, int32_t *blk) {
  using B = Block<D>;
  bool ok = true;
  auto step = [&](int from, int f, int to) {
    const int32_t b = blk[from];
    blk[to] = (ok && b >= 0) ? arms[int64_t(f) * N + b] : -1;
  };
  auto check = [&](int q) { ok = ok && blk[q] >= 0; };
  blk[B::q(0, 0, 0)] = int32_t(n);
  step(B::q(0, 0, 0), 0, B::q(-1, 0, 0));
  step(B::q(0, 0, 0), 1, B::q(1, 0, 0));
  check(B::q(-1, 0, 0));
  check(B::q(1, 0, 0));
#pragma unroll
  for (int i = -1; i <= 1; ++i) {
    step(B::q(i, 0, 0), 2, B::q(i, -1, 0));
    step(B::q(i, 0, 0), 3, B::q(i, 1, 0));
  }
#pragma unroll
  for (int i = -1; i <= 1; ++i) {
    check(B::q(i, -1, 0));
    check(B::q(i, 1, 0));
  }
  if constexpr (D == 3) {
#pragma unroll
    for (int i = -1; i <= 1; ++i)
#pragma unroll
      for (int j = -1; j <= 1; ++j) {
        step(B::q(i, j, 0), 4, B::q(i, j, -1));
        step(B::q(i, j, 0), 5, B::q(i, j, 1));
      }
#pragma unroll
    for (int i = -1; i <= 1; ++i)
#pragma unroll
      for (int j = -1; j <= 1; ++j) {
        check(B::q(i, j, -1));
        check(B::q(i, j, 1));
      }
  }
  return ok;
}

// nodes a block of k_find / k_emit covers, BLOCK at a time
constexpr int SPAN = 4 * BLOCK;

__device__ __forceinline__ int wave_rank(uint64_t mask) {
  return __popcll(mask & ((uint64_t(1) << (threadIdx.x & 63)) - 1));
}

// Every node's state -- 0: outside the band, 1: no block, 2: a sample -- and
// the number of samples and of band nodes without a block per SPAN nodes.
template <int D>
__global__ void __launch_bounds__(BLOCK)
    k_find(const int32_t *__restrict__ arms, int64_t N, const double *__restrict__ phi, double band,
           uint8_t *__restrict__ state, uint32_t *__restrict__ counts) {
  __shared__ uint32_t part[2][BLOCK / 64];
  uint32_t hit = 0, miss = 0;
#pragma unroll 1
  for (int k = 0; k < SPAN / BLOCK; ++k) {
    const int64_t n = int64_t(blockIdx.x) * SPAN + k * BLOCK + threadIdx.x;
    if (n >= N) break;
    int s = 0;
    if (fabs(phi[n]) < band) {
      int32_t blk[Block<D>::Q];
      s = gather_block<D>(arms, N, n, blk) ? 2 : 1;
    }
    state[n] = uint8_t(s);
    hit += s == 2;
    miss += s == 1;
  }
  for (int o = 32; o > 0; o >>= 1) {
    hit += __shfl_xor(hit, o);
    miss += __shfl_xor(miss, o);
  }
  if ((threadIdx.x & 63) == 0) {
    part[0][threadIdx.x >> 6] = hit;
    part[1][threadIdx.x >> 6] = miss;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLOCK / 64; ++w) {
      hit += part[0][w];
      miss += part[1][w];
    }
    counts[2 * blockIdx.x] = hit;
    counts[2 * blockIdx.x + 1] = miss;
  }
}

// first[b]: the samples before block b; total: {samples, band nodes without a
// block}.  One block walks over the counts, SCAN of them at a time.
constexpr int SCAN = 1024;
__global__ void __launch_bounds__(SCAN) k_scan(const uint32_t *__restrict__ counts, int64_t nb,
                                               int64_t *__restrict__ first, unsigned long long *__restrict__ total) {
  __shared__ int64_t wsum[SCAN / 64], wmiss[SCAN / 64];
  int64_t run = 0, missed = 0;
  const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
  for (int64_t b0 = 0; b0 < nb; b0 += SCAN) {
    const int64_t b = b0 + threadIdx.x;
    const int64_t own = b < nb ? int64_t(counts[2 * b]) : 0;
    int64_t v = own, m = b < nb ? int64_t(counts[2 * b + 1]) : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t u = __shfl_up(v, o);
      if (lane >= o) v += u;
      m += __shfl_xor(m, o);
    }
    if (lane == 63) wsum[wave] = v;
    if (lane == 0) wmiss[wave] = m;
    __syncthreads();
    int64_t before = 0, all = 0;
    for (int w = 0; w < SCAN / 64; ++w) {
      before += w < wave ? wsum[w] : 0;
      all += wsum[w];
      missed += wmiss[w];
    }
    if (b < nb) first[b] = run + before + v - own;
    run += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    total[0] = (unsigned long long)run;
    total[1] = (unsigned long long)missed;
  }
}

// The samples in node order: each BLOCK nodes' features are laid out in LDS at
// their rank and leave as one contiguous run.
template <int D>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
    k_emit(const int32_t *__restrict__ arms, int64_t N, const double *__restrict__ phi,
           const double *__restrict__ nrm, const double *__restrict__ kap, double h, double inv_h,
           const uint8_t *__restrict__ state, const int64_t *__restrict__ first, int64_t cap,
           float *__restrict__ feat, double *__restrict__ offset, int64_t *__restrict__ node) {
  using B = Block<D>;
  constexpr int LS = B::NF | 1;  // odd row stride
  __shared__ float rows[BLOCK * LS];
  __shared__ int wcount[BLOCK / 64];
  int64_t base = first[blockIdx.x];
#pragma unroll 1
  for (int chunk = 0; chunk < SPAN / BLOCK; ++chunk) {
    const int64_t n = int64_t(blockIdx.x) * SPAN + chunk * BLOCK + threadIdx.x;
    const bool ok = n < N && state[n] == 2;
    const uint64_t mask = __ballot(ok);
    if ((threadIdx.x & 63) == 0) wcount[threadIdx.x >> 6] = __popcll(mask);
    __syncthreads();
    int rank = wave_rank(mask), cnt = 0;
    for (int w = 0; w < BLOCK / 64; ++w) {
      rank += w < int(threadIdx.x >> 6) ? wcount[w] : 0;
      cnt += wcount[w];
    }
    if (ok && base + rank < cap) {
      const int64_t s = base + rank;
      float *o = rows + rank * LS;
      int32_t blk[B::Q];
      gather_block<D>(arms, N, n, blk);
      const double f0 = phi[n];
      if (inv_h != 0.0) {  // h is a power of two: the product is the quotient
#pragma unroll
        for (int q = 0; q < B::Q; ++q) o[q] = float(phi[blk[q]] * inv_h);
      } else {
#pragma unroll
        for (int q = 0; q < B::Q; ++q) o[q] = float(phi[blk[q]] / h);
      }
      // the projection's offset, in units of h clamped to the block, and the
      // cell of the block that holds it
      double w[D];
      bool low[D];  // the cell lies on the negative side
#pragma unroll
      for (int a = 0; a < D; ++a) {
        const double off = -f0 * nrm[int64_t(a) * N + n];
        double u = off / h;
        u = u < -1.0 ? -1.0 : (u > 1.0 ? 1.0 : u);
        low[a] = u < 0.0;
        w[a] = low[a] ? u + 1.0 : u;
        offset[s * D + a] = off;
      }
      // kappa at the cell's corners: corner bit 1 is the node's side where the
      // cell is on the negative side, else the far side
      double v[1 << D];
#pragma unroll
      for (int e = 0; e < (1 << D); ++e) {  // e: the axes along which the corner is not the node's
        int32_t id = int32_t(n);
        if (D == 2) {
          const int32_t x = low[0] ? blk[B::q(-1, 0)] : blk[B::q(1, 0)];
          const int32_t y = low[1] ? blk[B::q(0, -1)] : blk[B::q(0, 1)];
          const int32_t xm = low[1] ? blk[B::q(-1, -1)] : blk[B::q(-1, 1)];
          const int32_t xp = low[1] ? blk[B::q(1, -1)] : blk[B::q(1, 1)];
          id = e == 0 ? id : e == 1 ? x : e == 2 ? y : (low[0] ? xm : xp);
        } else {
          auto at = [&](int i, int j, int k) {  // signs already chosen where nonzero
            const int32_t zp = blk[B::q(i, j, k)];
            const int32_t zm = blk[B::q(i, j, -k)];
            return k == 0 ? blk[B::q(i, j, 0)] : (low[D - 1] ? zm : zp);
          };
          auto aty = [&](int i, int j, int k) {
            return j == 0 ? at(i, 0, k) : (low[1] ? at(i, -1, k) : at(i, 1, k));
          };
          auto atx = [&](int i, int j, int k) {
            return i == 0 ? aty(0, j, k) : (low[0] ? aty(-1, j, k) : aty(1, j, k));
          };
          id = atx(e & 1, (e >> 1) & 1, (e >> 2) & 1);
        }
        v[e] = kap[id];
      }
      // corner c (bit a: the cell's upper side along a) is e = c, with the bits
      // of the negative axes flipped
#pragma unroll
      for (int a = 0; a < D; ++a)
#pragma unroll
        for (int e = 0; e < (1 << D); ++e)
          if (!((e >> a) & 1)) {
            const int g = e | (1 << a);
            const double x = v[e], y = v[g];
            v[e] = low[a] ? y : x;
            v[g] = low[a] ? x : y;
          }
      double k = 0.0;
#pragma unroll
      for (int c = 0; c < (1 << D); ++c) {
        double wt = 1.0;
#pragma unroll
        for (int a = 0; a < D; ++a) wt = wt * (((c >> a) & 1) ? w[a] : 1.0 - w[a]);
        k = k + wt * v[c];
      }
      o[B::Q] = float(h * k);
      node[s] = n;
    }
    __syncthreads();
    const int64_t room = cap - base;
    const int out = int(room < 0 ? 0 : (room < cnt ? room : cnt)) * B::NF;
    for (int e = int(threadIdx.x); e < out; e += BLOCK)
      feat[base * B::NF + e] = rows[(e / B::NF) * LS + e % B::NF];
    base += cnt;
    __syncthreads();
  }
}

// [n][28] samples -> [n][28] network inputs (one canonical orientation)
__global__ void __launch_bounds__(BLOCK) k_normalize3(const float *__restrict__ feat, int64_t n,
                                                      float *__restrict__ out) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  curv_normalize3(feat + 28 * s, out + 28 * s);
}

// Hybrid h*kappa of 3D samples: one network output per sample.  With a
// residual network, corrections no larger than `dead` are dropped: on a
// well-resolved surface the numerical value is more accurate than the
// network's noise floor.
__global__ void __launch_bounds__(BLOCK) k_hybrid3(const float *__restrict__ feat, const float *__restrict__ pred,
                                                   int64_t n, float lo, float hi, int residual, float dead,
                                                   float *__restrict__ hk) {
  const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  hk[s] = curv_hybrid3(feat[28 * s + 27], pred[s], lo, hi, residual, dead);
}

// The samples of a call, in node order.  8.1M-node octree: 2.56
// ms with one thread per node walking the stencil tables and an atomic per
// sample (plus a sort and three gathers for the order, 0.9 ms), here arms 0.13,
// find 0.12 and emit 0.29 ms.
template <int D>
void grid_samples(casl_stencil *st, const double *phi, const double *nrm, const double *kap, double h, double band,
                  float *feat, double *offset, int64_t *node, int64_t cap, hipStream_t s) {
  const int64_t N = st->N, nb = (N + SPAN - 1) / SPAN;
  st->arms.ensure(size_t(2 * D) * N);
  st->sample_state.ensure(size_t(N));
  st->sample_counts.ensure(size_t(2 * nb));
  st->sample_first.ensure(size_t(nb));
  if (st->tiled && st->path == CASL_PATH_TILED) {
    AxisLevels lv;
    for (int a = 0; a < 3; ++a) {
      lv.l[a] = -1;
      for (int l = 0; l < 16; ++l)
        if (float(st->geom_base[a] * std::ldexp(1.0, -l)) == float(h)) lv.l[a] = l;
    }
    hipLaunchKernelGGL(k_tile_arms<D>, dim3(unsigned(st->n_tiles)), dim3(BLOCK), 0, s, tile_args<float>(st), lv,
                       st->arms.p);
  } else {
    hipLaunchKernelGGL(k_arms<D>, dim3(grid_for(N)), dim3(BLOCK), 0, s, st->tables<D>(), float(h), st->arms.p);
  }
  hipLaunchKernelGGL(k_find<D>, dim3(unsigned(nb)), dim3(BLOCK), 0, s, st->arms.p, N, phi, band, st->sample_state.p,
                     st->sample_counts.p);
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(SCAN), 0, s, st->sample_counts.p, nb, st->sample_first.p, st->red.p);
  int e = 0;
  const double inv_h = std::frexp(h, &e) == 0.5 ? 1.0 / h : 0.0;
  if (cap > 0)
    hipLaunchKernelGGL(k_emit<D>, dim3(unsigned(nb)), dim3(BLOCK), 0, s, st->arms.p, N, phi, nrm, kap, h, inv_h,
                       st->sample_state.p, st->sample_first.p, cap, feat, offset, node);
  HIP_CHECK(hipGetLastError());
}

}  // namespace

extern "C" {

int casl_curvature_grid_samples(casl_stencil_t *st, const double *phi, const double *normals, const double *kappa,
                                double h, double band, float *feat, double *offset, int64_t *node,
                                int64_t max_samples, int64_t *n_samples, int64_t *n_skipped, void *stream) {
  return guarded([&]() {
    if (!st || !phi || !normals || !kappa || !n_samples || !(h > 0) || !(band > 0) || max_samples < 0)
      throw std::invalid_argument("bad arguments");
    if (max_samples > 0 && (!feat || !offset || !node)) throw std::invalid_argument("null output arrays");
    if (double(float(h)) != h) throw std::invalid_argument("h must be exact in FP32 (a grid spacing)");
    hipStream_t s = static_cast<hipStream_t>(stream);
    st->red.ensure(2);
    if (st->dim == 2)
      grid_samples<2>(st, phi, normals, kappa, h, band, feat, offset, node, max_samples, s);
    else
      grid_samples<3>(st, phi, normals, kappa, h, band, feat, offset, node, max_samples, s);
    unsigned long long c[2] = {0, 0};
    HIP_CHECK(hipMemcpyAsync(c, st->red.p, sizeof(c), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    *n_samples = int64_t(c[0]);
    if (n_skipped) *n_skipped = int64_t(c[1]);
  });
}

int casl_curvature_normalize_3d(const float *feat, int64_t n, float *out, void *stream) {
  return guarded([&]() {
    if (n < 0 || (n > 0 && (!feat || !out))) throw std::invalid_argument("bad arguments");
    if (n == 0) return;
    hipLaunchKernelGGL(k_normalize3, dim3(grid_for(n)), dim3(BLOCK), 0, static_cast<hipStream_t>(stream), feat, n,
                       out);
    HIP_CHECK(hipGetLastError());
  });
}

int casl_curvature_hybrid_3d(const float *feat, const float *pred, int64_t n, float lo, float hi, int residual,
                             float deadband, float *hk, void *stream) {
  return guarded([&]() {
    if (n < 0 || (n > 0 && (!feat || !pred || !hk)) || !(hi > lo) || !(lo >= 0.f) || !(deadband >= 0.f))
      throw std::invalid_argument("bad arguments");
    if (n == 0) return;
    hipLaunchKernelGGL(k_hybrid3, dim3(grid_for(n)), dim3(BLOCK), 0, static_cast<hipStream_t>(stream), feat, pred, n,
                       lo, hi, residual, deadband, hk);
    HIP_CHECK(hipGetLastError());
  });
}

}  // extern "C"
