// Small fully-connected ReLU network (h*kappa regressor) trained and run on
// the GPU with hand-written BF16 MFMA kernels (FP32 accumulation).
//
// The reference runs a comparable network for inference only, on the CPU
// with OpenBLAS sgemm (src/my_p4est_curvature_ml.cpp:214-286), and ships no
// training code; this is the MI355X-native counterpart with training.
//
// Layer l: Z_l = A_{l-1} W_l + b_l, A_l = relu(Z_l) (last layer: no ReLU);
// A_0 = bf16((x - mean)/std).  Weights are FP32 masters [in][out] with BF16
// copies for the GEMMs; activations are stored in BF16; every GEMM
// accumulates in FP32.  Loss: mean squared error.
//
// GEMM: one wavefront computes a 32x32 tile with
// v_mfma_f32_32x32x16_bf16 (A lanes hold rows i = lane%32, k = 8*(lane/32)+v;
// B lanes hold columns j = lane%32, same k; the 16 accumulators of a lane are
// rows 8*(r/4) + 4*(lane/32) + r%4 of column lane%32); a 256-thread block
// covers 64x64.  Every operand load is bounds checked, so any M, N, K work.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "curv_device.hpp"
#include "mlp_chain.hpp"
#include "reinit_device.hpp"

using namespace casl;
using casl::dev::curv_hybrid2;
using casl::dev::curv_hybrid3;
using casl::dev::curv_normalize2;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__host__ __device__ inline uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return 0x7fc0;  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t h) {
  uint32_t u = uint32_t(h) << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// The GEMM epilogue of one 32x32 wave tile at (tm, tn): bias, ReLU or the
// ReLU'-mask, FP32 and/or BF16 stores.
__device__ __forceinline__ void gemm_store(const f32x16 &acc, int M, int N, int tm, int tn, int lane,
                                           const float *__restrict__ bias, const uint16_t *__restrict__ mask, int ldm,
                                           int relu, float *__restrict__ C, uint16_t *__restrict__ C16, int ldc) {
  const int li = lane & 31;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = tm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    const int col = tn + li;
    if (row < M && col < N) {
      float v = acc[r];
      if (bias) v += bias[col];
      if (relu) v = v > 0.f ? v : 0.f;
      if (mask && !(bf2f(mask[size_t(row) * ldm + col]) > 0.f)) v = 0.f;
      if (C) C[size_t(row) * ldc + col] = v;
      if (C16) C16[size_t(row) * ldc + col] = f2bf(v);
    }
  }
}

// C[M x N] = op(A)[M x K] op(B)[K x N] (+ bias[N]) then ReLU or ReLU'-mask.
//   op(A)(i, k) = TA ? A[k*lda + i] : A[i*lda + k]
//   op(B)(k, j) = TB ? B[j*ldb + k] : B[k*ldb + j]
//   mask: multiply by (mask[i*ldm + j] > 0), the ReLU derivative of a stored activation
// Split K: block z covers k in [z*kc, (z+1)*kc) and writes its FP32 partial
// to C32 + z*M*ldc (k_sum_splits adds the partials in a fixed order).
template <bool TA, bool TB>
__global__ void __launch_bounds__(256)
    k_gemm(int M, int N, int K, int kc, const uint16_t *__restrict__ A, int lda, const uint16_t *__restrict__ B,
           int ldb, const float *__restrict__ bias, const uint16_t *__restrict__ mask, int ldm, int relu,
           float *__restrict__ C32, uint16_t *__restrict__ C16, int ldc) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tm = blockIdx.y * 64 + (wave >> 1) * 32;
  const int tn = blockIdx.x * 64 + (wave & 1) * 32;
  const int li = lane & 31, lk = (lane >> 5) * 8;
  const int i = tm + li, j = tn + li;
  const int kb = int(blockIdx.z) * kc, ke = min(K, kb + kc);
  // rows of op(A) / columns of op(B) that are contiguous in k can be read 16 bytes at a time
  const bool avec = !TA && (lda & 7) == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;
  const bool bvec = TB && (ldb & 7) == 0 && (reinterpret_cast<uintptr_t>(B) & 15) == 0;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int k0 = kb; k0 < ke; k0 += 16) {
    const int kk = k0 + lk;
    union {
      uint4 q;
      uint16_t h[8];
    } ua, ub;
    if (avec && i < M && kk + 8 <= ke) {
      ua.q = *reinterpret_cast<const uint4 *>(A + size_t(i) * lda + kk);
    } else {
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const int k = kk + v;
        ua.h[v] = (i < M && k < ke) ? (TA ? A[size_t(k) * lda + i] : A[size_t(i) * lda + k]) : uint16_t(0);
      }
    }
    if (bvec && j < N && kk + 8 <= ke) {
      ub.q = *reinterpret_cast<const uint4 *>(B + size_t(j) * ldb + kk);
    } else {
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const int k = kk + v;
        ub.h[v] = (j < N && k < ke) ? (TB ? B[size_t(j) * ldb + k] : B[size_t(k) * ldb + j]) : uint16_t(0);
      }
    }
    bf16x8 a, b;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      a[v] = __builtin_bit_cast(__bf16, ua.h[v]);
      b[v] = __builtin_bit_cast(__bf16, ub.h[v]);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
  }
  float *C = C32 ? C32 + size_t(blockIdx.z) * M * ldc : nullptr;
  gemm_store(acc, M, N, tm, tn, lane, bias, mask, ldm, relu, C, C16, ldc);
}

// k_gemm with LDS-staged panels, for M and N multiples of 64 and K ranges
// (K and kc) multiples of 64 with 16-byte aligned operands: per K chunk of
// 64 the block's op(A) panel [64 x 64] and op(B) panel [64 x 64] are loaded
// with 16-byte vectors, all of a thread's loads in flight together, into
// LDS (k contiguous per row of op(A) and per column of op(B); transposed
// layouts are transposed on the way in), double-buffered so the next
// chunk's loads overlap this chunk's MFMAs.  Each wave then reads its
// operands from LDS.  The MFMA sequence (k ascending by 16) and the operand
// layout are k_gemm's, so the results are the same bits.
template <bool TA, bool TB>
__global__ void __launch_bounds__(256)
    k_gemm_lds(int M, int N, int K, int kc, const uint16_t *__restrict__ A, int lda, const uint16_t *__restrict__ B,
               int ldb, const float *__restrict__ bias, const uint16_t *__restrict__ mask, int ldm, int relu,
               float *__restrict__ C32, uint16_t *__restrict__ C16, int ldc) {
  constexpr int KC = 64, LS = KC + 8;  // chunk, LDS row stride in bf16 (144 bytes: 16-byte aligned rows)
  __shared__ __align__(16) uint16_t sa[2][64 * LS], sb[2][64 * LS];
  const int tid = int(threadIdx.x), wave = tid >> 6, lane = tid & 63;
  const int bm = int(blockIdx.y) * 64, bn = int(blockIdx.x) * 64;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int li = lane & 31, lk = (lane >> 5) * 8;
  const int kb = int(blockIdx.z) * kc, ke = min(K, kb + kc);
  const int nch = (ke - kb) / KC;
  // vector v of a panel (2 per thread): row v / 8 (of op(A), of op(B)^T, or
  // of the stored k-major matrix when transposed), 8 elements at (v % 8) * 8
  uint4 ra[2], rb[2];
  auto gload = [&](int k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int v = tid + 256 * h, r = v >> 3, c = (v & 7) * 8;
      ra[h] = TA ? *reinterpret_cast<const uint4 *>(A + size_t(k0 + r) * lda + bm + c)
                 : *reinterpret_cast<const uint4 *>(A + size_t(bm + r) * lda + k0 + c);
      rb[h] = TB ? *reinterpret_cast<const uint4 *>(B + size_t(bn + r) * ldb + k0 + c)
                 : *reinterpret_cast<const uint4 *>(B + size_t(k0 + r) * ldb + bn + c);
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int v = tid + 256 * h, r = v >> 3, c = (v & 7) * 8;
      if (TA) {
        const uint16_t *e = reinterpret_cast<const uint16_t *>(&ra[h]);
#pragma unroll
        for (int t = 0; t < 8; ++t) sa[buf][(c + t) * LS + r] = e[t];
      } else {
        *reinterpret_cast<uint4 *>(&sa[buf][r * LS + c]) = ra[h];
      }
      if (TB) {
        *reinterpret_cast<uint4 *>(&sb[buf][r * LS + c]) = rb[h];
      } else {
        const uint16_t *e = reinterpret_cast<const uint16_t *>(&rb[h]);
#pragma unroll
        for (int t = 0; t < 8; ++t) sb[buf][(c + t) * LS + r] = e[t];
      }
    }
  };
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  if (nch > 0) {
    gload(kb);
    lstore(0);
  }
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const int buf = ch & 1;
    if (ch + 1 < nch) gload(kb + (ch + 1) * KC);
#pragma unroll
    for (int ks = 0; ks < KC / 16; ++ks) {
      const uint4 ua = *reinterpret_cast<const uint4 *>(&sa[buf][(wm + li) * LS + ks * 16 + lk]);
      const uint4 ub = *reinterpret_cast<const uint4 *>(&sb[buf][(wn + li) * LS + ks * 16 + lk]);
      const bf16x8 a = __builtin_bit_cast(bf16x8, ua), b = __builtin_bit_cast(bf16x8, ub);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    if (ch + 1 < nch) lstore(buf ^ 1);
    __syncthreads();
  }
  float *C = C32 ? C32 + size_t(blockIdx.z) * M * ldc : nullptr;
  gemm_store(acc, M, N, bm + wm, bn + wn, lane, bias, mask, ldm, relu, C, C16, ldc);
}

// out[e] = sum_z part[z*n + e], z = 0 .. splits-1 in order; eight loads are
// issued ahead of their additions, so the chain waits on memory once per
// eight splits (64-thread blocks spread the elements over every CU)
__global__ void k_sum_splits(const float *__restrict__ part, int splits, int64_t n, float *__restrict__ out) {
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= n) return;
  float s = part[e];
  int z = 1;
  for (; z + 8 <= splits; z += 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = part[size_t(z + k) * n + e];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k];
  }
  for (; z < splits; ++z) s += part[size_t(z) * n + e];
  out[e] = s;
}

// A_0 = bf16((x - mean) / std)
__global__ void k_pack_input(const float *__restrict__ x, const float *__restrict__ mean,
                             const float *__restrict__ inv_std, int n, int d, uint16_t *__restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(n) * d) return;
  const int c = int(t % d);
  out[t] = f2bf((x[t] - mean[c]) * inv_std[c]);
}

// dY = 2 (y - t) / n (MSE gradient), as FP32 and BF16; loss accumulates sum (y - t)^2
__global__ void k_mse_seed(const float *__restrict__ y, const float *__restrict__ t, int n, float scale,
                           float *__restrict__ dy32, uint16_t *__restrict__ dy16, float *__restrict__ loss) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  float e = 0.f;
  if (i < n) {
    e = y[i] - t[i];
    const float g = 2.f * e * scale;
    dy32[i] = g;
    dy16[i] = f2bf(g);
  }
  float s = e * e;
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) atomicAdd(loss, s);
}

// Bias gradients, out[c] = sum over rows of x[r * m + c], in a fixed order.
// k_colsum_part: block b sums rows [b * COLSUM_ROWS, ...) per column with
// coalesced row reads (consecutive threads take consecutive columns; 256 / m
// row lanes when m < 256, added in lane order) into part[b * m + c].
// k_colsum_fin: one block per column; thread t adds partials t, t + 256, ...
// in ascending order, then a fixed tree over the threads in LDS.  Short rows
// per block and a tree at the end keep every dependent chain short.
constexpr int COLSUM_ROWS = 32;
__global__ void __launch_bounds__(256)
    k_colsum_part(const float *__restrict__ x, int n, int m, float *__restrict__ part) {
  __shared__ float red[256];
  const int t = int(threadIdx.x), b = int(blockIdx.x);
  const int r0 = b * COLSUM_ROWS, r1 = min(n, r0 + COLSUM_ROWS);
  for (int c0 = 0; c0 < m; c0 += 256) {
    const int cw = min(m - c0, 256), lanes = 256 / cw, lane = t / cw, c = c0 + t % cw;
    float s = 0.f;
    if (lane < lanes)
      for (int r = r0 + lane; r < r1; r += lanes) s += x[size_t(r) * m + c];
    red[t] = s;
    __syncthreads();
    if (t < cw) {
      float tot = red[t];
      for (int l = 1; l < lanes; ++l) tot += red[l * cw + t];
      part[size_t(b) * m + c0 + t] = tot;
    }
    __syncthreads();
  }
}
__global__ void __launch_bounds__(256) k_colsum_fin(const float *__restrict__ part, int nb, int m,
                                                    float *__restrict__ out) {
  __shared__ float red[256];
  const int c = int(blockIdx.x), t = int(threadIdx.x);
  float s = 0.f;
  for (int b = t; b < nb; b += 256) s += part[size_t(b) * m + c];
  red[t] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) red[t] += red[t + w];
    __syncthreads();
  }
  if (t == 0) out[c] = red[0];
}

// Adam on FP32 masters, weights then biases in one launch; refreshes the BF16
// copy of the weights and its transposed copy (in: the input width, 0: none)
struct AdamVec {
  float *p;
  const float *g;
  float *m, *v;
};
__global__ void k_adam(AdamVec W, int nw, AdamVec B, int nb, uint16_t *__restrict__ p16, uint16_t *__restrict__ p16t,
                       int in, float lr, float b1, float b2, float eps, float c1, float c2) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nw + nb) return;
  const bool weight = i < nw;
  if (!weight) i -= nw;
  float *__restrict__ p = weight ? W.p : B.p;
  const float *__restrict__ g = weight ? W.g : B.g;
  float *__restrict__ m = weight ? W.m : B.m;
  float *__restrict__ v = weight ? W.v : B.v;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  p[i] = pi;
  if (weight) {
    const uint16_t h = f2bf(pi);
    p16[i] = h;
    if (in > 0) {
      const int64_t t = chain::transposed_index(in, i);
      if (t >= 0) p16t[t] = h;
    }
  }
}

__global__ void k_to_bf16(const float *__restrict__ a, uint16_t *__restrict__ b, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = f2bf(a[i]);
}

__global__ void k_zero_f(float *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

inline unsigned blocks(int64_t n, int b = 256) { return unsigned((n + b - 1) / b); }

template <bool TA, bool TB>
void gemm(int M, int N, int K, const uint16_t *A, int lda, const uint16_t *B, int ldb, const float *bias,
          const uint16_t *mask, int ldm, int relu, float *C32, uint16_t *C16, int ldc, hipStream_t s,
          int splits = 1) {
  const int kc = splits > 1 ? ((K + splits - 1) / splits + 15) / 16 * 16 : K;
  dim3 grid(unsigned((N + 63) / 64), unsigned((M + 63) / 64), unsigned(splits));
  const bool staged = M % 64 == 0 && N % 64 == 0 && K % 64 == 0 && kc % 64 == 0 && lda % 8 == 0 && ldb % 8 == 0 &&
                      (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (reinterpret_cast<uintptr_t>(B) & 15) == 0;
  prof_begin("k_gemm", s);
  if (staged)
    hipLaunchKernelGGL((k_gemm_lds<TA, TB>), grid, dim3(256), 0, s, M, N, K, kc, A, lda, B, ldb, bias, mask, ldm,
                       relu, C32, C16, ldc);
  else
    hipLaunchKernelGGL((k_gemm<TA, TB>), grid, dim3(256), 0, s, M, N, K, kc, A, lda, B, ldb, bias, mask, ldm, relu,
                       C32, C16, ldc);
  prof_end("k_gemm", s);
  HIP_CHECK(hipGetLastError());
}

// number of K splits that gives a small output tile grid enough blocks
inline int k_splits(int M, int N, int K) {
  const int tiles = ((M + 63) / 64) * ((N + 63) / 64);
  int s = 1;
  while (s < 64 && tiles * s < 512 && K / (2 * s) >= 256) s *= 2;
  return s;
}

}  // namespace

struct casl_mlp {
  int L = 0;                        // number of layers
  std::vector<int> dim;             // L + 1 widths
  DevBuf<float> W, b, gW, gb, mW, vW, mb, vb;  // concatenated per layer
  DevBuf<uint16_t> W16;
  std::vector<size_t> offW, offb;   // per-layer offsets
  DevBuf<float> mean, inv_std;
  int cap = 0;                      // activation capacity (rows)
  DevBuf<uint16_t> act16;           // L activations [cap x dim[l]] (l = 0 .. L-1) as bf16
  DevBuf<float> z32;                // FP32 scratch [cap x max width]
  DevBuf<uint16_t> d16a, d16b;      // BF16 back-propagated gradients
  DevBuf<float> y32, loss;
  DevBuf<float> part;               // split-K partial sums of weight gradients
  DevBuf<float> colpart;            // per-block column sums of bias gradients
  std::vector<size_t> offA;
  int maxw = 0;
  int64_t step = 0;
  // the fused training pass (mlp_chain.hpp): weights transposed, activations
  // and gradients by feature, the batch's partial sums, the loss on the host
  DevBuf<uint16_t> W16T, chain_act, chain_dz;
  DevBuf<float> chain_cols, chain_loss;
  PinnedBuf<float> host_loss;

  // (10 .. 32)-128-128-128-128-1
  bool chained() const {
    return L == 5 && dim[0] <= chain::K0 && dim[1] == chain::H && dim[2] == chain::H && dim[3] == chain::H &&
           dim[4] == chain::H && dim[5] == 1;
  }
  // uploads the transposed BF16 weights of host weights (layers concatenated)
  void upload_transposed(const std::vector<uint16_t> &w16) {
    if (!chained()) return;
    std::vector<uint16_t> t(size_t(chain::TRANSPOSED_SIZE), 0);
    for (size_t i = 0; i < w16.size(); ++i) {
      const int64_t k = chain::transposed_index(dim[0], int64_t(i));
      if (k >= 0) t[size_t(k)] = w16[i];
    }
    W16T.ensure(t.size());
    HIP_CHECK(hipMemcpy(W16T.p, t.data(), t.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
  }

  void ensure_cap(int n) {
    if (n <= cap) return;
    cap = n;
    size_t tot = 0;
    offA.assign(L, 0);
    for (int l = 0; l < L; ++l) {
      offA[l] = tot;
      tot += size_t(n) * dim[l];
    }
    act16.ensure(tot);
    z32.ensure(size_t(n) * maxw);
    d16a.ensure(size_t(n) * maxw);
    d16b.ensure(size_t(n) * maxw);
    y32.ensure(size_t(n) * dim[L]);
  }
};

namespace {

// forward pass; leaves activations in act16 and the output in out (FP32 [n x dim[L]])
void forward(casl_mlp *m, const float *x, int n, float *out, hipStream_t s) {
  m->ensure_cap(n);
  hipLaunchKernelGGL(k_pack_input, dim3(blocks(int64_t(n) * m->dim[0])), dim3(256), 0, s, x, m->mean.p,
                     m->inv_std.p, n, m->dim[0], m->act16.p + m->offA[0]);
  HIP_CHECK(hipGetLastError());
  for (int l = 0; l < m->L; ++l) {
    const int in = m->dim[l], o = m->dim[l + 1];
    const uint16_t *A = m->act16.p + m->offA[l];
    const bool last = (l == m->L - 1);
    gemm<false, false>(n, o, in, A, in, m->W16.p + m->offW[l], o, m->b.p + m->offb[l], nullptr, 0, last ? 0 : 1,
                       last ? out : nullptr, last ? nullptr : m->act16.p + m->offA[l + 1], o, s);
  }
}

// Forward, loss and all gradients of a (10 .. 32)-128x4-1 network in three
// launches (the layer by layer pass takes 43): the chain keeps 32 samples'
// activations in a wave's registers, one launch makes every layer's weight
// gradients, one sums them.  Same bits as the layer by layer pass, the loss
// aside (its sum there depends on the order of atomics).
void chain_backward(casl_mlp *m, const float *x, const float *t, int n, bool want_loss, hipStream_t s) {
  const int blocks64 = (n + 63) / 64, nb = (n + 31) / 32;
  const int sp = k_splits(chain::H, chain::H, n);
  const uint32_t nw = uint32_t(m->W.n);
  m->chain_act.ensure(size_t(m->dim[0] + 4 * chain::H) * 64 * blocks64);
  m->chain_dz.ensure(size_t(chain::COLS) * 64 * blocks64);
  m->chain_cols.ensure(size_t(nb) * chain::COLS);
  m->chain_loss.ensure(size_t(nb));
  m->part.ensure(size_t(sp) * nw);
  m->host_loss.ensure(1);
  chain::TrainArgs a{};
  a.x = x;
  a.t = t;
  a.n = n;
  a.in = m->dim[0];
  a.scale = 1.f / float(n);
  a.mean = m->mean.p;
  a.inv_std = m->inv_std.p;
  a.W16 = m->W16.p;
  a.W16T = m->W16T.p;
  a.b = m->b.p;
  a.act = m->chain_act.p;
  a.dz = m->chain_dz.p;
  a.colpart = m->chain_cols.p;
  a.losspart = m->chain_loss.p;
  chain::GradArgs g{};
  g.act = a.act;
  g.dz = a.dz;
  g.n = n;
  g.in = a.in;
  // chunks as gemm() cuts them
  g.kc = sp > 1 ? ((n + sp - 1) / sp + 15) / 16 * 16 : n;
  g.nw = nw;
  g.chunks = sp;
  g.part = m->part.p;
  prof_begin("k_train_chain", s);
  hipLaunchKernelGGL(chain::k_train_chain, dim3(unsigned(blocks64)), dim3(chain::TRAIN_BLOCK), 0, s, a);
  prof_end("k_train_chain", s);
  prof_begin("k_train_grads", s);
  hipLaunchKernelGGL(chain::k_train_grads, dim3(chain::grad_blocks(sp)), dim3(256), 0, s, g);
  prof_end("k_train_grads", s);
  chain::SumArgs u{};
  u.part = m->part.p;
  u.colpart = a.colpart;
  u.losspart = a.losspart;
  u.splits = sp;
  u.nb = nb;
  u.nw = nw;
  u.wblocks = (nw + chain::SUM_BLOCK - 1) / chain::SUM_BLOCK;
  u.gW = m->gW.p;
  u.gb = m->gb.p;
  u.loss = m->loss.p;
  u.host_loss = want_loss ? m->host_loss.p : nullptr;
  hipLaunchKernelGGL(chain::k_train_sums, dim3(u.wblocks + chain::COLS + 1), dim3(chain::SUM_BLOCK), 0, s, u);
  HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------ fused network curvature
// The learned h*kappa of samples in one launch: input normalisation, every
// layer of a (10|28)-128-128-128-128-1 network on MFMA with the activations in
// registers (mlp_chain.hpp), and the hybrid blend.  A block holds all weights
// in LDS, copied once; each of its eight waves then runs 64 network rows at a
// time by itself, two blocks of 32 that share every weight operand it reads
// (one block of 32 would need the LDS's whole bandwidth to feed the MFMAs).  2D
// samples give 2 rows each (as is, reflected), 3D samples one.  Every product,
// bias add, ReLU and BF16 rounding is the one k_gemm makes, in the same order
// (the K loop ascends in steps of 16), so the result equals
// casl_curvature_normalize(_3d) + casl_mlp_forward + casl_curvature_hybrid(_3d)
// bit for bit.  3.3M samples: 1.36 ms in 3D and 2.26 ms in 2D with activations in
// LDS and one wave per SIMD, 0.49 and 0.70 ms (710 and 950 TFLOP/s) here.
struct FusedNet {
  const uint16_t *W16T;  // transposed layers (mlp_chain.hpp)
  const uint16_t *W4;    // the last layer's 128 weights
  const float *b;        // per layer, concatenated
  const float *mean, *inv_std;
};
constexpr int NF_BLOCK = 512, NF_WAVES = NF_BLOCK / 64;
constexpr int NF_ROWS = 64;  // network rows of a wave at a time
constexpr int NF_FS = 28;    // LDS row stride of a wave's 32 samples' features (3D)

struct NetLds {
  uint16_t W0[chain::H * chain::W0S];
  uint16_t Wh[3][chain::H * chain::WS];
  uint16_t W4[chain::H];
  float bias[4 * chain::H];
  float mean[chain::K0], inv_std[chain::K0];
  float feat[NF_WAVES][32 * NF_FS];
};
static_assert(sizeof(NetLds) <= 160 * 1024, "fused network kernel exceeds the LDS of a compute unit");

// k_pack_input's rounding of the eight inputs o[v] from input k0 on (lds: the
// scaler), as one MFMA operand half; inputs past `in` are zero
__device__ __forceinline__ chain::bf16x8 pack_inputs(const NetLds &lds, const float (&o)[8], int k0, int in,
                                                     bool valid) {
  chain::u32x4 w;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float f[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int k = k0 + 2 * v + q;
      f[q] = (valid && k < in) ? (o[2 * v + q] - lds.mean[k]) * lds.inv_std[k] : 0.f;
    }
    w[v] = chain::pack_bf16(f[0], f[1]);
  }
  return __builtin_bit_cast(chain::bf16x8, w);
}

// The inputs of 3D sample li of the 32 whose features lie at f (curv_normalize3,
// the same operations on the values this half of the wave needs): new axis b
// reads old axis p[b] reflected by r, so value (i, j, k) of the canonical
// orientation is feature 13 + i S0 + j S1 + k S2 with S_b = r stride(p[b]).
__device__ __forceinline__ void inputs3(const NetLds &lds, const float *__restrict__ f, bool valid, int hh,
                                        chain::bf16x8 *op) {
  const float sg = f[27] > 0.f ? -1.f : 1.f;
  float g[3];
  int S[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    constexpr int stride[3] = {9, 3, 1};
    g[a] = f[13 + stride[a]] * sg - f[13 - stride[a]] * sg;
    if (g[a] == 0.f) g[a] = float(dev::EPS);
    S[a] = g[a] < 0.f ? -stride[a] : stride[a];
    g[a] = fabsf(g[a]);
  }
  auto swap_if = [&](int a, int b, bool c) {
    const float x = g[a], y = g[b];
    g[a] = c ? y : x;
    g[b] = c ? x : y;
    const int u = S[a], v = S[b];
    S[a] = c ? v : u;
    S[b] = c ? u : v;
  };
  swap_if(0, 1, g[1] > g[0]);
  const bool last = g[2] > g[1];
  swap_if(1, 2, last);
  swap_if(0, 1, last && g[1] > g[0]);
  const float f0 = f[13] * sg;
  const float gx = 0.5f * (f[13 + S[0]] * sg - f[13 - S[0]] * sg);
  const float gy = 0.5f * (f[13 + S[1]] * sg - f[13 - S[1]] * sg);
  const float gz = 0.5f * (f[13 + S[2]] * sg - f[13 - S[2]] * sg);
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    float o[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      // input q of this half: its place in the cube is known for each half
      float c[3];
      int at = 13;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int q0 = 16 * ks + v, q1 = q0 + 8, d = a == 0 ? 9 : (a == 1 ? 3 : 1);
        const int c0 = (q0 / d) % 3 - 1, c1 = (q1 / d) % 3 - 1;
        c[a] = hh ? float(c1) : float(c0);
        at += hh ? c1 * S[a] : c0 * S[a];
      }
      const int q0 = 16 * ks + v, q1 = q0 + 8;
      const bool cube = q1 < 27 || (q0 < 27 && !hh);
      const float x = cube ? f[at] * sg : 0.f;
      o[v] = x - (f0 + (c[0] * gx + c[1] * gy + c[2] * gz));
      if (q0 == 4) o[v] = hh ? (q1 == 12 ? gz : o[v]) : gx;  // inputs 4 and 12
      if (q1 == 10) o[v] = hh ? gy : o[v];
      if (q1 == 13) o[v] = hh ? f0 : o[v];
      if (q1 == 27) o[v] = hh ? f[27] * sg : o[v];
    }
    op[ks] = pack_inputs(lds, o, 16 * ks + 8 * hh, 28, valid);
  }
}

template <int D>
__global__ void __launch_bounds__(NF_BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_net_curvature(FusedNet net, const float *__restrict__ feat, int wide, int64_t n, float lo, float hi, int residual,
                    float dead, float *__restrict__ hk) {
  using namespace chain;
  constexpr int NFEAT = D == 2 ? 10 : 28;  // features per sample
  constexpr int RPS = D == 2 ? 2 : 1;      // network rows per sample
  constexpr int BS32 = 32 / RPS;           // samples of a block of 32 rows
  constexpr int KS0 = D == 2 ? 1 : 2;      // first layer's steps of 16
  extern __shared__ __align__(16) unsigned char raw[];
  NetLds &lds = *reinterpret_cast<NetLds *>(raw);
  const int tid = int(threadIdx.x), wave = tid >> 6, lane = tid & 63, li = lane & 31, hh = lane >> 5;
  // weights, 16 bytes at a time
  for (int c = tid; c < H * K0 / 8; c += NF_BLOCK)
    *reinterpret_cast<u32x4 *>(lds.W0 + (c >> 2) * W0S + (c & 3) * 8) = reinterpret_cast<const u32x4 *>(net.W16T)[c];
  for (int c = tid; c < 3 * H * H / 8; c += NF_BLOCK) {
    const int l = c / (H * H / 8), e = c % (H * H / 8);
    *reinterpret_cast<u32x4 *>(lds.Wh[l] + (e >> 4) * WS + (e & 15) * 8) =
        reinterpret_cast<const u32x4 *>(net.W16T + H * K0)[c];
  }
  if (tid < H) lds.W4[tid] = net.W4[tid];
  lds.bias[tid] = net.b[tid];
  if (tid < NFEAT) {
    lds.mean[tid] = net.mean[tid];
    lds.inv_std[tid] = net.inv_std[tid];
  }
  const float b4 = net.b[4 * H];
  __syncthreads();
  float *fw = lds.feat[wave];
  const int64_t ntiles = (n * RPS + NF_ROWS - 1) / NF_ROWS;
  for (int64_t tile = int64_t(wave) * gridDim.x + blockIdx.x; tile < ntiles; tile += int64_t(NF_WAVES) * gridDim.x) {
    bf16x8 op[2][8];
    float ihk[2];
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      const int64_t s0 = (tile * 2 + blk) * BS32, smp = s0 + li / RPS;
      const bool valid = smp < n;
      if constexpr (D == 3) {
        // the 32 samples' features through LDS, then each half's inputs
        wave_order();
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int c = lane + 64 * h;  // 224 pieces of four
          if (c < 32 * NFEAT / 4 && s0 * NFEAT + 4 * c < n * NFEAT) {
            const float *src = feat + s0 * NFEAT + 4 * c;
            float4 v;
            if (wide) {
              v = *reinterpret_cast<const float4 *>(src);
            } else {
              v.x = src[0];
              v.y = src[1];
              v.z = src[2];
              v.w = src[3];
            }
            *reinterpret_cast<float4 *>(fw + 4 * c) = v;
          }
        }
        wave_order();
        ihk[blk] = fw[li * NF_FS + 27];
        inputs3(lds, fw + li * NF_FS, valid, hh, op[blk]);
      } else {
        float o[20];
#pragma unroll
        for (int q = 0; q < 20; ++q) o[q] = 0.f;
        ihk[blk] = 0.f;
        if (valid) {
          curv_normalize2(feat + NFEAT * smp, o);
          ihk[blk] = feat[NFEAT * smp + 9];
        }
        const bool refl = (li & 1) != 0;
        float x[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) {
          const float a = refl ? o[10 + v] : o[v];
          const float b = v < 2 ? (refl ? o[18 + v] : o[8 + v]) : 0.f;
          x[v] = hh ? b : a;
        }
        op[blk][0] = pack_inputs(lds, x, 8 * hh, NFEAT, valid);
      }
      __builtin_amdgcn_sched_barrier(0);  // keeps one block's inputs from living beside the next one's
    }
    // hidden layers, 32 features at a time
    Packed<4> out[2];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      const uint16_t *W = l == 0 ? lds.W0 : lds.Wh[l - 1];
      const int KS = l == 0 ? KS0 : 8, S = l == 0 ? W0S : WS;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        f32x16 c[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) c[0][r] = c[1][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8 a = *reinterpret_cast<const bf16x8 *>(W + (32 * rb + li) * S + ks * 16 + hh * 8);
          c[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, op[0][ks], c[0], 0, 0, 0);
          c[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, op[1][ks], c[1], 0, 0, 0);
        }
        bias_relu(c[0], lds.bias + l * H + 32 * rb, lane, out[0].p[rb]);
        bias_relu(c[1], lds.bias + l * H + 32 * rb, lane, out[1].p[rb]);
      }
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) op[blk][ks] = operand(out[blk], ks);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      const float y = last_output(op[blk], lds.W4, lane) + b4;  // rows in lanes 0 .. 31
      const int64_t smp = (tile * 2 + blk) * BS32 + li / RPS;
      if constexpr (D == 2) {
        const float y1 = __shfl_down(y, 1);
        if (hh == 0 && (li & 1) == 0 && smp < n) hk[smp] = curv_hybrid2(ihk[blk], y, y1, lo, hi, residual);
      } else {
        if (hh == 0 && smp < n) hk[smp] = curv_hybrid3(ihk[blk], y, lo, hi, residual, dead);
      }
    }
  }
}

}  // namespace

extern "C" {

int casl_mlp_create(const int32_t *dims, int n_layers, uint64_t seed, casl_mlp_t **out) {
  return guarded([&]() {
    if (!out || !dims || n_layers < 1) throw std::invalid_argument("bad arguments");
    auto m = std::make_unique<casl_mlp>();
    m->L = n_layers;
    m->dim.assign(dims, dims + n_layers + 1);
    size_t nw = 0, nb = 0;
    for (int l = 0; l < n_layers; ++l) {
      if (m->dim[l] < 1 || m->dim[l + 1] < 1) throw std::invalid_argument("layer widths must be positive");
      m->offW.push_back(nw);
      m->offb.push_back(nb);
      nw += size_t(m->dim[l]) * m->dim[l + 1];
      nb += size_t(m->dim[l + 1]);
    }
    for (int d : m->dim) m->maxw = std::max(m->maxw, d);
    // He-normal initialisation (deterministic in seed), zero biases
    std::mt19937_64 rng(seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    std::vector<float> w(nw), bb(nb, 0.f);
    for (int l = 0; l < n_layers; ++l) {
      const double sd = std::sqrt(2.0 / m->dim[l]);
      for (size_t i = 0; i < size_t(m->dim[l]) * m->dim[l + 1]; ++i) w[m->offW[l] + i] = float(sd * nd(rng));
    }
    std::vector<uint16_t> w16(nw);
    for (size_t i = 0; i < nw; ++i) w16[i] = f2bf(w[i]);
    m->W.ensure(nw);
    m->W16.ensure(nw);
    m->gW.ensure(nw);
    m->mW.ensure(nw);
    m->vW.ensure(nw);
    m->b.ensure(nb);
    m->gb.ensure(nb);
    m->mb.ensure(nb);
    m->vb.ensure(nb);
    HIP_CHECK(hipMemcpy(m->W.p, w.data(), nw * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->W16.p, w16.data(), nw * 2, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->b.p, bb.data(), nb * 4, hipMemcpyHostToDevice));
    std::vector<float> zw(nw, 0.f), zb(nb, 0.f);
    HIP_CHECK(hipMemcpy(m->mW.p, zw.data(), nw * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->vW.p, zw.data(), nw * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->mb.p, zb.data(), nb * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->vb.p, zb.data(), nb * 4, hipMemcpyHostToDevice));
    std::vector<float> mean(m->dim[0], 0.f), inv(m->dim[0], 1.f);
    m->mean.ensure(mean.size());
    m->inv_std.ensure(inv.size());
    HIP_CHECK(hipMemcpy(m->mean.p, mean.data(), mean.size() * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->inv_std.p, inv.data(), inv.size() * 4, hipMemcpyHostToDevice));
    m->loss.ensure(1);
    m->upload_transposed(w16);
    *out = m.release();
  });
}

int casl_curvature_learned(casl_mlp_t *m, const float *feat, int64_t n, float lo, float hi, int residual,
                           float deadband, float *hk, void *stream) {
  return guarded([&]() {
    if (!m || n < 0 || (n > 0 && (!feat || !hk)) || !(hi > lo) || !(lo >= 0.f) || !(deadband >= 0.f))
      throw std::invalid_argument("bad arguments");
    if (m->L != 5 || (m->dim[0] != 10 && m->dim[0] != 28) || !m->chained())
      throw std::invalid_argument("casl_curvature_learned takes a (10|28)-128-128-128-128-1 network");
    if (n == 0) return;
    FusedNet net{};
    net.W16T = m->W16T.p;
    net.W4 = m->W16.p + m->offW[4];
    net.b = m->b.p;
    net.mean = m->mean.p;
    net.inv_std = m->inv_std.p;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int dev = 0, cus = 0;
    HIP_CHECK(hipGetDevice(&dev));
    HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // a wave per 64 rows, one block per compute unit; few rows spread over the
    // units before they share one
    const int64_t ntiles = (n * (m->dim[0] == 10 ? 2 : 1) + NF_ROWS - 1) / NF_ROWS;
    const unsigned grid = unsigned(std::max<int64_t>(1, std::min<int64_t>(ntiles, int64_t(cus))));
    const int wide = (reinterpret_cast<uintptr_t>(feat) & 15) == 0;
    prof_begin("k_net_curvature", s);
    auto launch = [&](auto kernel) {
      HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(sizeof(NetLds))));
      hipLaunchKernelGGL(kernel, dim3(grid), dim3(NF_BLOCK), sizeof(NetLds), s, net, feat, wide, n, lo, hi, residual,
                         deadband, hk);
    };
    if (m->dim[0] == 10)
      launch(&k_net_curvature<2>);
    else
      launch(&k_net_curvature<3>);
    prof_end("k_net_curvature", s);
    HIP_CHECK(hipGetLastError());
  });
}

int casl_mlp_destroy(casl_mlp_t *m) {
  delete m;
  return CASL_OK;
}

int casl_mlp_num_params(const casl_mlp_t *m, int64_t *n_weights, int64_t *n_biases) {
  return guarded([&]() {
    if (!m) throw std::invalid_argument("null mlp");
    if (n_weights) *n_weights = int64_t(m->W.n);
    if (n_biases) *n_biases = int64_t(m->b.n);
  });
}

int casl_mlp_set_scaler(casl_mlp_t *m, const float *mean, const float *stdev) {
  return guarded([&]() {
    if (!m || !mean || !stdev) throw std::invalid_argument("null argument");
    std::vector<float> inv(m->dim[0]);
    for (int i = 0; i < m->dim[0]; ++i) {
      if (!(stdev[i] > 0)) throw std::invalid_argument("scaler deviations must be positive");
      inv[i] = 1.f / stdev[i];
    }
    HIP_CHECK(hipMemcpy(m->mean.p, mean, m->dim[0] * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->inv_std.p, inv.data(), m->dim[0] * 4, hipMemcpyHostToDevice));
  });
}

int casl_mlp_get_params(const casl_mlp_t *m, float *weights, float *biases) {
  return guarded([&]() {
    if (!m) throw std::invalid_argument("null mlp");
    if (weights) HIP_CHECK(hipMemcpy(weights, m->W.p, m->W.n * 4, hipMemcpyDeviceToHost));
    if (biases) HIP_CHECK(hipMemcpy(biases, m->b.p, m->b.n * 4, hipMemcpyDeviceToHost));
  });
}

int casl_mlp_set_params(casl_mlp_t *m, const float *weights, const float *biases) {
  return guarded([&]() {
    if (!m || !weights || !biases) throw std::invalid_argument("null argument");
    std::vector<uint16_t> w16(m->W.n);
    for (size_t i = 0; i < m->W.n; ++i) w16[i] = f2bf(weights[i]);
    HIP_CHECK(hipMemcpy(m->W.p, weights, m->W.n * 4, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(m->W16.p, w16.data(), m->W.n * 2, hipMemcpyHostToDevice));
    m->upload_transposed(w16);
    HIP_CHECK(hipMemcpy(m->b.p, biases, m->b.n * 4, hipMemcpyHostToDevice));
  });
}

int casl_mlp_get_grads(const casl_mlp_t *m, float *gw, float *gb) {
  return guarded([&]() {
    if (!m) throw std::invalid_argument("null mlp");
    if (gw) HIP_CHECK(hipMemcpy(gw, m->gW.p, m->gW.n * 4, hipMemcpyDeviceToHost));
    if (gb) HIP_CHECK(hipMemcpy(gb, m->gb.p, m->gb.n * 4, hipMemcpyDeviceToHost));
  });
}

int casl_mlp_forward(casl_mlp_t *m, const float *x, int n, float *y, void *stream) {
  return guarded([&]() {
    if (!m || !x || !y || n < 0) throw std::invalid_argument("bad arguments");
    if (n == 0) return;
    forward(m, x, n, y, static_cast<hipStream_t>(stream));
  });
}

// Forward + backward of the mean squared error on (x, t); gradients stay on
// the device (casl_mlp_get_grads).  *loss (host, may be null) receives the MSE.
int casl_mlp_backward(casl_mlp_t *m, const float *x, const float *t, int n, float *loss, void *stream) {
  return guarded([&]() {
    if (!m || !x || !t || n <= 0) throw std::invalid_argument("bad arguments");
    if (m->dim[m->L] != 1) throw std::invalid_argument("training needs a scalar output");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (m->chained()) {
      chain_backward(m, x, t, n, loss != nullptr, s);
      if (loss) {
        HIP_CHECK(hipStreamSynchronize(s));
        *loss = *m->host_loss.p / float(n);
      }
      return;
    }
    m->ensure_cap(n);  // sizes y32 before its address is taken
    forward(m, x, n, m->y32.p, s);
    hipLaunchKernelGGL(k_zero_f, dim3(1), dim3(64), 0, s, m->loss.p, 1);
    // dZ_L = 2 (y - t) / n  -> z32 (FP32) and d16a (BF16), [n x 1]
    hipLaunchKernelGGL(k_mse_seed, dim3(blocks(n)), dim3(256), 0, s, m->y32.p, t, n, 1.f / float(n), m->z32.p,
                       m->d16a.p, m->loss.p);
    HIP_CHECK(hipGetLastError());
    uint16_t *dcur = m->d16a.p, *dnext = m->d16b.p;
    for (int l = m->L - 1; l >= 0; --l) {
      const int in = m->dim[l], o = m->dim[l + 1];
      // bias gradient from the FP32 dZ_l in z32
      const int nb = (n + COLSUM_ROWS - 1) / COLSUM_ROWS;
      m->colpart.ensure(size_t(std::max(nb, 1)) * o);
      hipLaunchKernelGGL(k_colsum_part, dim3(unsigned(std::max(nb, 1))), dim3(256), 0, s, m->z32.p, n, o,
                         m->colpart.p);
      hipLaunchKernelGGL(k_colsum_fin, dim3(unsigned(o)), dim3(256), 0, s, m->colpart.p, std::max(nb, 1), o,
                         m->gb.p + m->offb[l]);
      HIP_CHECK(hipGetLastError());
      const uint16_t *Aprev = m->act16.p + m->offA[l];  // [n x in]
      // dW_l = A_{l-1}^T dZ_l : (in x n)(n x o)
      const int sp = k_splits(in, o, n);
      if (sp == 1) {
        gemm<true, false>(in, o, n, Aprev, in, dcur, o, nullptr, nullptr, 0, 0, m->gW.p + m->offW[l], nullptr, o, s);
      } else {
        m->part.ensure(size_t(sp) * in * o);
        gemm<true, false>(in, o, n, Aprev, in, dcur, o, nullptr, nullptr, 0, 0, m->part.p, nullptr, o, s, sp);
        const int64_t e = int64_t(in) * o;
        hipLaunchKernelGGL(k_sum_splits, dim3(unsigned((e + 63) / 64)), dim3(64), 0, s, m->part.p, sp, e,
                           m->gW.p + m->offW[l]);
        HIP_CHECK(hipGetLastError());
      }
      if (l > 0) {
        // dZ_{l-1} = (dZ_l W_l^T) * relu'(A_{l-1}) : (n x o)(o x in)
        gemm<false, true>(n, in, o, dcur, o, m->W16.p + m->offW[l], o, nullptr, Aprev, in, 0, m->z32.p, dnext, in, s);
        std::swap(dcur, dnext);
      }
    }
    if (loss) {
      float h = 0.f;
      HIP_CHECK(hipMemcpyAsync(&h, m->loss.p, 4, hipMemcpyDeviceToHost, s));
      HIP_CHECK(hipStreamSynchronize(s));
      *loss = h / float(n);
    }
  });
}

int casl_mlp_adam_step(casl_mlp_t *m, float lr, float beta1, float beta2, float eps, void *stream) {
  return guarded([&]() {
    if (!m) throw std::invalid_argument("null mlp");
    hipStream_t s = static_cast<hipStream_t>(stream);
    m->step += 1;
    const float c1 = float(1.0 / (1.0 - std::pow(double(beta1), double(m->step))));
    const float c2 = float(1.0 / (1.0 - std::pow(double(beta2), double(m->step))));
    const int nw = int(m->W.n), nb = int(m->b.n);
    const AdamVec w{m->W.p, m->gW.p, m->mW.p, m->vW.p}, b{m->b.p, m->gb.p, m->mb.p, m->vb.p};
    hipLaunchKernelGGL(k_adam, dim3(blocks(nw + nb)), dim3(256), 0, s, w, nw, b, nb, m->W16.p, m->W16T.p,
                       m->chained() ? m->dim[0] : 0, lr, beta1, beta2, eps, c1, c2);
    HIP_CHECK(hipGetLastError());
  });
}

// Plain BF16 MFMA GEMM on device buffers (exposed for testing the kernel):
// C = op(A) op(B) (+ bias) (relu), C32 and/or C16 written with leading dim ldc.
int casl_bf16_gemm(int M, int N, int K, const uint16_t *A, int lda, int trans_a, const uint16_t *B, int ldb,
                   int trans_b, const float *bias, int relu, float *C32, uint16_t *C16, int ldc, void *stream) {
  return guarded([&]() {
    if (M < 0 || N < 0 || K < 0 || !A || !B || (!C32 && !C16)) throw std::invalid_argument("bad arguments");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!trans_a && !trans_b)
      gemm<false, false>(M, N, K, A, lda, B, ldb, bias, nullptr, 0, relu, C32, C16, ldc, s);
    else if (trans_a && !trans_b)
      gemm<true, false>(M, N, K, A, lda, B, ldb, bias, nullptr, 0, relu, C32, C16, ldc, s);
    else if (!trans_a && trans_b)
      gemm<false, true>(M, N, K, A, lda, B, ldb, bias, nullptr, 0, relu, C32, C16, ldc, s);
    else
      throw std::invalid_argument("both operands transposed is not supported");
  });
}

}  // extern "C"
