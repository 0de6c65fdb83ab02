// First derivatives, normals and mean curvature on the flattened stencils
// (the numerical curvature chain of the reference), FP64:
//   casl_first_derivatives  my_p4est_node_neighbors_t::first_derivatives_central
//                           (src/my_p4est_node_neighbors.h:568-600), per node
//                           dx/dy/dz_central (src/my_p4est_quad_neighbor_nodes_of_node.cpp:638-760)
//   casl_normals            compute_normals (src/my_p4est_utils.cpp:1720-1740):
//                           gradient / |gradient|, 0 where |gradient| < EPS
//   casl_mean_curvature     compute_mean_curvature(neighbors, normals, kappa)
//                           (src/my_p4est_utils.cpp:1648-1690) with
//                           qnnn::get_curvature(normals) (src/my_p4est_quad_neighbor_nodes_of_node.h:2167-2171):
//                           dx_central(n_x) + dy_central(n_y) [+ dz_central(n_z)]
// Every call is one pass.  Normals and mean curvature run on the tiled encoding
// where it holds power-of-two cells (one block per tile, the field of T u H1
// in LDS, 16-byte records in place of 216 bytes of tables a node); everything
// else, and first derivatives, run one thread per node on the grid-wide tables.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "reinit_device.hpp"
#include "tiles_device.hpp"

using namespace casl;
using namespace casl::dev;

namespace {

constexpr int BLOCK = 256;

template <int D, class TB>
__global__ void __launch_bounds__(BLOCK) k_gradient(TB t, const double *__restrict__ f, double *__restrict__ fd) {
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= t.N) return;
  double g[D];
  gradient_central<D>(t, n, f, g);
#pragma unroll
  for (int a = 0; a < D; ++a) fd[int64_t(a) * t.N + n] = g[a];
}

template <int D, class TB>
__global__ void __launch_bounds__(BLOCK) k_normals(TB t, const double *__restrict__ phi, double *__restrict__ nrm) {
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= t.N) return;
  double g[D];
  gradient_central<D>(t, n, phi, g);
  double s = g[0] * g[0] + g[1] * g[1];
  if constexpr (D == 3) s = s + g[2] * g[2];
  const double a = sqrt(s);
#pragma unroll
  for (int k = 0; k < D; ++k) nrm[int64_t(k) * t.N + n] = (a < EPS) ? 0.0 : g[k] / a;
}

// kappa = sum_a d(n_a)/dx_a, each with its own transverse corrections
template <int D, class TB>
__global__ void __launch_bounds__(BLOCK) k_curvature(TB t, const double *__restrict__ nrm, double *__restrict__ kap) {
  const int64_t n = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (n >= t.N) return;
  double k = 0.0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    double g[D];
    gradient_central<D>(t, n, nrm + int64_t(a) * t.N, g);
    k = (a == 0) ? g[0] : k + g[a];
  }
  kap[n] = k;
}

// gradient_central of a tile node from the field in LDS, in the same operation
// order.  Regular nodes have no correction (their transverse products are 0,
// so every weight is 0); equal power-of-two arms make every division exact.
// tab, n: the grid-wide tables and the node, read for hanging nodes of cells
// that are not CUBES.
template <int D, bool CUBES, class TB>
__device__ __forceinline__ void tile_gradient(const TB &t, int j, const double *__restrict__ f, const Tables<D> &tab,
                                              int64_t n, double *grad) {
  constexpr int F = 2 * D;
  const double f000 = f[j];
  if constexpr (TB::UNIFORM) {
#pragma unroll
    for (int a = 0; a < D; ++a)
      grad[a] = ((f[t.id[2 * a + 1]] - f000) + (f000 - f[t.id[2 * a]])) * (0.5 * t.iq[0]);
  } else if constexpr (TB::REGULAR) {
#pragma unroll
    for (int a = 0; a < D; ++a)
      grad[a] = central_derivative(f[t.id[2 * a + 1]], f000, f[t.id[2 * a]], t.dist[2 * a + 1], t.dist[2 * a]);
  } else {
    double fnb[F], vq[TB::NH], f0, dd[D];
    hang_laplace<D, double>(t, j, f, f0, fnb, dd, vq);
#pragma unroll
    for (int a = 0; a < D; ++a)
      grad[a] = central_derivative(fnb[2 * a + 1], f000, fnb[2 * a], t.dist[2 * a + 1], t.dist[2 * a]);
    // the hanging faces' transverse products, and inverse_d_max over arms and
    // transverse distances.  In cubes a regular face has its arm cell's size
    // among them; in other cells its extents are those of the other axes, and
    // which of them the list holds is known to the tables alone.
    double P[F][2] = {}, m = 0.0;
    const int h0 = t.hface(0), h1 = TB::NH > 1 ? t.hface(TB::NH - 1) : h0;
#pragma unroll
    for (int q = 0; q < F; ++q) m = max2(m, max2(t.dist[q], (q == h0 || q == h1) ? 0.0 : t.q[q]));
#pragma unroll
    for (int q = 0; q < TB::NH; ++q) {
      const int fq = t.hface(q);
      if (q == 0 || fq < F) {
        const auto sg = t.slot_geom(fq);
        const double m0 = t.hdt(q, 0, sg), p0 = t.hdt(q, 1, sg);
        m = max2(max2(m, m0), p0);
        double z0 = 0.0, z1 = 0.0;
        if constexpr (D == 3) {
          z0 = t.hdt(q, 2, sg);
          z1 = t.hdt(q, 3, sg);
          m = max2(max2(m, z0), fq == 4 ? 0.0 : z1);  // the reference's list leaves d_00m_0p out
        }
#pragma unroll
        for (int k = 0; k < F; ++k) {
          P[k][0] = (k == fq) ? m0 * p0 : P[k][0];
          P[k][1] = (k == fq) ? z0 * z1 : P[k][1];
        }
      }
    }
    double idm;
    if constexpr (CUBES)
      idm = 1.0 / m;
    else
      idm = inverse_d_max<D>(tab, n);
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int k = 0; k < D - 1; ++k) {
        const double dm = t.dist[2 * a], dp = t.dist[2 * a + 1];
        // dd_correction_weight with the products at hand
        const double w = 0.5 * (P[2 * a + 1][k] * dm / dp - P[2 * a][k] * dp / dm) / (dm + dp);
        const int ta = (k == 0) ? (a == 0 ? 1 : 0) : (a == 2 ? 1 : 2);
        if (!check_if_zero(w * idm)) grad[a] -= dd[ta] * w;
      }
  }
}

// fn(stencil, LDS slot) for the record at position i of a tile
template <int D, class Fn>
__device__ __forceinline__ void with_record(const TileArgs<double> &A, const TileCtx<D> &c, bool ufast, int i,
                                            const RecRegs &r, int fetched, Fn &&fn) {
  int j = fetched;
  if (ufast && c.uniform(i)) {
    UniStencil<D, double> st;
    j = st.load(r.w, A.geom);
    fn(st, j);
    return;
  }
  const TileRec rec = record_at<D>(c, i, r, j);
  if (!(rec.geo & GEO_IRREGULAR)) {
    RegStencil<D, double> st;
    st.load(rec, A.geom);
    fn(st, j);
  } else {
    HangStencil<D, double> st;
    st.load(rec, c.ext_of(A.ext, i), A.geom);
    fn(st, j);
  }
}

// 512 threads, four tile nodes each: 32 KB of LDS and at most 128 VGPRs let
// two blocks share a compute unit, one loading while the other computes.
constexpr int TBLOCK = 512;

// the field of T u H1 into LDS; the caller puts barriers around it
template <int D>
__device__ __forceinline__ void load_field(const TileArgs<double> &A, const TileCtx<D> &c,
                                           const double *__restrict__ f, double *__restrict__ lds) {
  for (int j = int(threadIdx.x); j < c.nT; j += TBLOCK) lds[j] = f[c.s + j];
  for (int j = int(threadIdx.x); j < c.nH1; j += TBLOCK) lds[c.nT + j] = f[A.halo[c.hb + j]];
}

// compute_normals, one block per tile.  8.4M-node octree: 0.76 ms on the
// grid-wide tables, 0.17 ms here.
template <int D, bool CUBES>
__global__ void __launch_bounds__(TBLOCK) __attribute__((amdgpu_waves_per_eu(4)))
    k_tile_normals(TileArgs<double> A, Tables<D> tab, const double *__restrict__ phi, double *__restrict__ nrm) {
  __shared__ double f[TileLimits<D>::DMAX];
  TileCtx<D> c;
  c.load(A, xcd_tile(int(blockIdx.x), int(gridDim.x)));
  const bool ufast = A.geom.template uni_fast<ANY_CELLS>();
  load_field<D>(A, c, phi, f);
  __syncthreads();
  for (int i = int(threadIdx.x); i < c.nT; i += TBLOCK) {
    RecRegs r;
    const int js = fetch_record<D>(A, c, i, r);
    with_record<D>(A, c, ufast, i, r, js, [&](const auto &st, int j) {
      double g[D];
      tile_gradient<D, CUBES>(st, j, f, tab, c.s + j, g);
      double s = g[0] * g[0] + g[1] * g[1];
      if constexpr (D == 3) s = s + g[2] * g[2];
      const double a = sqrt(s);
#pragma unroll
      for (int k = 0; k < D; ++k) nrm[int64_t(k) * A.N + c.s + j] = (a < EPS) ? 0.0 : g[k] / a;
    });
  }
}

// One axis of k_tile_curvature: d(n_a)/dx_a added to the partial sums in LDS,
// or (the last axis) the sum written out.
template <int D, bool CUBES, int AX>
__device__ __forceinline__ void curvature_axis(const TileArgs<double> &A, const Tables<D> &tab, const TileCtx<D> &c,
                                               bool ufast, const double *__restrict__ nrm, double *__restrict__ f,
                                               double *__restrict__ sum, double *__restrict__ kap) {
  load_field<D>(A, c, nrm + int64_t(AX) * A.N, f);
  __syncthreads();
  for (int i = int(threadIdx.x); i < c.nT; i += TBLOCK) {
    RecRegs r;
    const int js = fetch_record<D>(A, c, i, r);
    with_record<D>(A, c, ufast, i, r, js, [&](const auto &st, int j) {
      double g[D];
      tile_gradient<D, CUBES>(st, j, f, tab, c.s + j, g);  // the other axes' parts drop out at compile time
      const double k = (AX == 0) ? g[0] : sum[i] + g[AX];
      if constexpr (AX == D - 1)
        kap[c.s + j] = k;
      else
        sum[i] = k;
    });
  }
  __syncthreads();  // the component has been read
}

// compute_mean_curvature, one block per tile, one component of the normals in
// LDS at a time (the sum over the axes stays in LDS, each thread its own
// entries: 48 KB, so that blocks share a compute unit).  8.4M-node octree:
// 1.64 ms on the grid-wide tables, 0.29 ms here.
template <int D, bool CUBES>
__global__ void __launch_bounds__(TBLOCK) __attribute__((amdgpu_waves_per_eu(4)))
    k_tile_curvature(TileArgs<double> A, Tables<D> tab, const double *__restrict__ nrm, double *__restrict__ kap) {
  __shared__ double f[TileLimits<D>::DMAX];
  __shared__ double sum[TileLimits<D>::TMAX];
  TileCtx<D> c;
  c.load(A, xcd_tile(int(blockIdx.x), int(gridDim.x)));
  const bool ufast = A.geom.template uni_fast<ANY_CELLS>();
  curvature_axis<D, CUBES, 0>(A, tab, c, ufast, nrm, f, sum, kap);
  curvature_axis<D, CUBES, 1>(A, tab, c, ufast, nrm, f, sum, kap);
  if constexpr (D == 3) curvature_axis<D, CUBES, 2>(A, tab, c, ufast, nrm, f, sum, kap);
}

inline unsigned grid_for(int64_t n) { return unsigned((n + BLOCK - 1) / BLOCK); }

// The tiles take a call when they are the stencil's path and hold cells of
// power-of-two edges (the shortcuts above are exact there).
inline bool on_tiles(const casl_stencil *st) { return st->use_tiles(true) && !st->weighted_tiles(); }

// fn(integral_constant<bool, cubes>) for the tiles of a call on_tiles().
template <class Fn>
void with_cubes(const casl_stencil *st, Fn &&fn) {
  if (tile_cells(st, true) == DYADIC_CUBES)
    fn(std::true_type{});
  else
    fn(std::false_type{});
}

void check_stencil(const casl_stencil *st, const void *a, const void *b) {
  if (!st || !a || !b) throw std::invalid_argument("null argument");
}

}  // namespace

extern "C" {

int casl_first_derivatives(casl_stencil_t *st, const double *f, double *fd, void *stream) {
  return guarded([&]() {
    check_stencil(st, f, fd);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (st->dim == 2)
      st->with_tables<2>(true, [&](auto t) {
        hipLaunchKernelGGL((k_gradient<2, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, f, fd);
      });
    else
      st->with_tables<3>(true, [&](auto t) {
        hipLaunchKernelGGL((k_gradient<3, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, f, fd);
      });
    HIP_CHECK(hipGetLastError());
  });
}

int casl_normals(casl_stencil_t *st, const double *phi, double *normals, void *stream) {
  return guarded([&]() {
    check_stencil(st, phi, normals);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (on_tiles(st)) {
      const dim3 g(unsigned(st->n_tiles)), b(TBLOCK);
      with_cubes(st, [&](auto cubes) {
        constexpr bool CUBES = decltype(cubes)::value;
        if (st->dim == 2)
          hipLaunchKernelGGL((k_tile_normals<2, CUBES>), g, b, 0, s, tile_args<double>(st), st->tables<2>(), phi, normals);
        else
          hipLaunchKernelGGL((k_tile_normals<3, CUBES>), g, b, 0, s, tile_args<double>(st), st->tables<3>(), phi, normals);
      });
    } else if (st->dim == 2)
      st->with_tables<2>(true, [&](auto t) {
        hipLaunchKernelGGL((k_normals<2, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, phi, normals);
      });
    else
      st->with_tables<3>(true, [&](auto t) {
        hipLaunchKernelGGL((k_normals<3, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, phi, normals);
      });
    HIP_CHECK(hipGetLastError());
  });
}

int casl_mean_curvature(casl_stencil_t *st, const double *normals, double *kappa, void *stream) {
  return guarded([&]() {
    check_stencil(st, normals, kappa);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (on_tiles(st)) {
      const dim3 g(unsigned(st->n_tiles)), b(TBLOCK);
      with_cubes(st, [&](auto cubes) {
        constexpr bool CUBES = decltype(cubes)::value;
        if (st->dim == 2)
          hipLaunchKernelGGL((k_tile_curvature<2, CUBES>), g, b, 0, s, tile_args<double>(st), st->tables<2>(), normals, kappa);
        else
          hipLaunchKernelGGL((k_tile_curvature<3, CUBES>), g, b, 0, s, tile_args<double>(st), st->tables<3>(), normals, kappa);
      });
    } else if (st->dim == 2)
      st->with_tables<2>(true, [&](auto t) {
        hipLaunchKernelGGL((k_curvature<2, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, normals, kappa);
      });
    else
      st->with_tables<3>(true, [&](auto t) {
        hipLaunchKernelGGL((k_curvature<3, decltype(t)>), dim3(grid_for(st->N)), dim3(BLOCK), 0, s, t, normals, kappa);
      });
    HIP_CHECK(hipGetLastError());
  });
}

}  // extern "C"
