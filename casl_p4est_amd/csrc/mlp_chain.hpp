// The (in)-128-128-128-128-1 network on MFMA with the activations in registers.
//
// A wave owns 32 rows (samples) and computes each layer transposed, out
// features by samples: A operand = weights (rows = features) from LDS, B
// operand = the previous layer's output.  An accumulator lane then holds one
// sample's features 8 g + 4 (lane/32) + t of each 32-feature block, and the
// next layer's B operand wants features 8 (lane/32) + v of each 16: the two
// halves of the wave trade the registers of neighbouring g, one
// v_permlane32_swap per pair, so activations never leave the registers.
// Every product and every accumulation order (k ascending by 16) is k_gemm's,
// and so are bias, ReLU and the BF16 rounding: the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace casl {
namespace chain {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int H = 128;       // hidden width
constexpr int WS = H + 8;    // LDS row stride (halves) of a 128-wide weight matrix
constexpr int K0 = 32;       // padded input width of the transposed first layer
constexpr int W0S = K0 + 8;  // its LDS row stride

// Two floats to packed BF16, round to nearest even (one instruction).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  f32x2 v;
  v[0] = a;
  v[1] = b;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// NB x 32 features of a lane's sample as packed BF16: word [rb][g][u] holds
// features 32 rb + 8 g + 4 (lane/32) + 2 u and the next.
template <int NB>
struct Packed {
  uint32_t p[NB][4][2];
};
// The B operand of features 16 ks .. 16 ks + 15.
template <int NB>
__device__ __forceinline__ bf16x8 operand(const Packed<NB> &a, int ks) {
  const int rb = ks >> 1, g = 2 * (ks & 1);
  u32x4 w;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    // the low half keeps its g and takes the high half's g, the high half
    // keeps its g + 1 and takes the low half's
    const auto s = __builtin_amdgcn_permlane32_swap(a.p[rb][g][u], a.p[rb][g + 1][u], false, false);
    w[u] = s[0];
    w[2 + u] = s[1];
  }
  return __builtin_bit_cast(bf16x8, w);
}

template <int NB>
struct Acc {
  f32x16 a[NB];
};

// acc[rb] = rows 32 rb .. of W (row stride S halves, k contiguous) times b,
// KS steps of 16
template <int NB, int KS, int S>
__device__ __forceinline__ Acc<NB> product(const uint16_t *__restrict__ W, const bf16x8 *b, int lane) {
  const int li = lane & 31, lk = (lane >> 5) * 8;
  Acc<NB> c;
#pragma unroll
  for (int rb = 0; rb < NB; ++rb)
#pragma unroll
    for (int r = 0; r < 16; ++r) c.a[rb][r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int rb = 0; rb < NB; ++rb) {
      const bf16x8 a = *reinterpret_cast<const bf16x8 *>(W + (32 * rb + li) * S + ks * 16 + lk);
      c.a[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[ks], c.a[rb], 0, 0, 0);
    }
  return c;
}

// bias (LDS, from the first of the 32 features), ReLU, BF16 of one block
__device__ __forceinline__ void bias_relu(const f32x16 &c, const float *__restrict__ bias, int lane,
                                          uint32_t (&o)[4][2]) {
  const int h4 = (lane >> 5) * 4;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 b = *reinterpret_cast<const float4 *>(bias + 8 * g + h4);
    float v[4] = {c[4 * g] + b.x, c[4 * g + 1] + b.y, c[4 * g + 2] + b.z, c[4 * g + 3] + b.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = v[t] > 0.f ? v[t] : 0.f;
    o[g][0] = pack_bf16(v[0], v[1]);
    o[g][1] = pack_bf16(v[2], v[3]);
  }
}

// The last layer's one output of each of the 32 samples, before the bias, in
// lanes 0 .. 31: w = its 128 weights (LDS).
__device__ __forceinline__ float last_output(const bf16x8 *b, const uint16_t *__restrict__ w, int lane) {
  f32x16 c;
#pragma unroll
  for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    u32x4 q = *reinterpret_cast<const u32x4 *>(w + ks * 16 + (lane >> 5) * 8);
    if ((lane & 31) != 0) q = u32x4{0, 0, 0, 0};
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, q), b[ks], c, 0, 0, 0);
  }
  return c[0];
}

// ------------------------------------------------------------- training
// One pass over the batch: forward, the loss gradient and the whole backward
// chain of 32 samples per wave.  What the weight gradients need leaves as the
// MFMA operands of their products over samples: the activations A_0 .. A_4 and
// the gradients dZ_0 .. dZ_4 in BF16, 16 samples of each feature together and
// the features of those 16 samples in a row, so that an operand of 32 features
// is one contiguous 1 KB load (rows of all samples per feature touched 32
// cache lines a load: 20.3 us for the products of a 16384-row batch, 9.9 us so).
// The bias
// gradients' sums over each 32 rows and the squared errors leave beside them.
struct TrainArgs {
  const float *x, *t;          // [n][in], [n]
  int n, in;
  float scale;                 // 1 / n
  const float *mean, *inv_std;
  const uint16_t *W16;         // [in][out] per layer (backward)
  const uint16_t *W16T;        // [out][in] per layer, the first padded to K0 (forward)
  const float *b;
  uint16_t *act;               // features: in, then 4 x 128
  uint16_t *dz;                // features: 4 x 128 (dZ_0 .. dZ_3), then dZ_4
  float *colpart;              // [rows of 32][4 x 128 + 1]
  float *losspart;             // [rows of 32]
};
constexpr int COLS = 4 * H + 1;
// feature f of sample s among F features (see above)
__host__ __device__ inline size_t by_sixteen(int F, int f, int s) {
  return (size_t(s >> 4) * size_t(F) + size_t(f)) * 16 + size_t(s & 15);
}
// first weight of layer l; the biases are H a layer
__host__ __device__ constexpr uint32_t weight_offset(int in, int l) {
  return l == 0 ? 0u : uint32_t(in * H + (l - 1) * H * H);
}
constexpr int TRAIN_BLOCK = 256;
constexpr int FS = 33;  // LDS row stride of a wave's FP32 tile [feature][sample]
constexpr int BS = 40;  // and of its BF16 tile, in halves

// the 128 x 128 weights of one layer: loaded ahead, stored when the LDS is free
struct Staged {
  u32x4 q[8];
  __device__ __forceinline__ void load(const uint16_t *__restrict__ g, int tid) {
#pragma unroll
    for (int h = 0; h < 8; ++h) q[h] = reinterpret_cast<const u32x4 *>(g)[tid + TRAIN_BLOCK * h];
  }
  __device__ __forceinline__ void store(uint16_t *__restrict__ W, int tid) const {
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const int c = tid + TRAIN_BLOCK * h;
      *reinterpret_cast<u32x4 *>(W + (c >> 4) * WS + (c & 15) * 8) = q[h];
    }
  }
};

// Orders a wave's LDS accesses to its own tile (they execute in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// a wave's 64 x 32 BF16 tile to features f0 .. of dst (F in all), through LDS
__device__ __forceinline__ void store_tile(const Packed<2> &a, uint16_t *__restrict__ tile, uint16_t *__restrict__ dst,
                                           int F, int f0, int s0, int lane) {
  const int li = lane & 31, h4 = (lane >> 5) * 4;
  wave_order();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int f = 32 * rb + 8 * g + h4 + 2 * u;
        tile[f * BS + li] = uint16_t(a.p[rb][g][u]);
        tile[(f + 1) * BS + li] = uint16_t(a.p[rb][g][u] >> 16);
      }
  wave_order();
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int c = lane + 64 * h, f = (c >> 1) & 63, part = 16 * (c >> 7) + 8 * (c & 1);
    *reinterpret_cast<u32x4 *>(dst + by_sixteen(F, f0 + f, s0 + part)) =
        *reinterpret_cast<const u32x4 *>(tile + f * BS + part);
  }
  wave_order();
}

// A block runs 64 samples: two waves share 32 of them, each with half of the
// features (a wave alone on its SIMD is bound by the chain of one layer after
// the other; halves of 64 features shorten it and give every SIMD of the chip
// a wave at 16384 rows).  The halves' operands meet in LDS once a layer, where
// the next layer's weights are exchanged too.  16384 rows: 28 us with one wave
// per 32 samples, 21 us now.
__global__ void __launch_bounds__(TRAIN_BLOCK) __attribute__((amdgpu_waves_per_eu(1, 2)))
    k_train_chain(TrainArgs A) {
  __shared__ __align__(16) uint16_t W[H * WS];
  __shared__ __align__(16) float bias[4 * H];
  __shared__ __align__(16) uint16_t W4[H];
  __shared__ __align__(16) u32x4 xch[2][8][64];     // operands of each 32 samples
  __shared__ __align__(16) float tiles[4][64 * FS]; // FP32 tile of each wave; the BF16 tile shares it
  static_assert(64 * BS * 2 <= 64 * FS * 4, "the BF16 tile fits the FP32 one");
  const int tid = int(threadIdx.x), wave = tid >> 6, lane = tid & 63;
  const int li = lane & 31, hh = lane >> 5, sg = wave >> 1, fh = wave & 1;
  float *ft = tiles[wave];
  uint16_t *bt = reinterpret_cast<uint16_t *>(ft);
  const int s0 = int(blockIdx.x) * 64 + 32 * sg, smp = s0 + li;
  const bool valid = smp < A.n;
  const int FA = A.in + 4 * H, FD = COLS;
  const float b4 = A.b[4 * H];
  // first layer's weights, biases and the last layer's weights
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = tid + TRAIN_BLOCK * h;  // 128 rows of four 16-byte pieces
    *reinterpret_cast<u32x4 *>(W + (c >> 2) * W0S + (c & 3) * 8) = reinterpret_cast<const u32x4 *>(A.W16T)[c];
  }
  for (int e = tid; e < 4 * H; e += TRAIN_BLOCK) bias[e] = A.b[e];
  if (tid < H) W4[tid] = A.W16[weight_offset(A.in, 4) + tid];
  Staged next;
  next.load(A.W16T + H * K0, tid);
  // inputs, standardised, BF16 (both waves of the samples)
  bf16x8 op[8];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    u32x4 w;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float f[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int k = ks * 16 + hh * 8 + 2 * v + q;
        f[q] = (valid && k < A.in) ? (A.x[size_t(smp) * A.in + k] - A.mean[k]) * A.inv_std[k] : 0.f;
      }
      w[v] = pack_bf16(f[0], f[1]);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int k = ks * 16 + hh * 8 + 2 * v + q;
        if (k < A.in && fh == 0) A.act[by_sixteen(FA, k, smp)] = uint16_t(q ? w[v] >> 16 : w[v]);
      }
    }
    op[ks] = __builtin_bit_cast(bf16x8, w);
  }
  Packed<2> act[4];  // this half's activations A_1 .. A_4, for ReLU'
  Acc<2> c;
  // the other half's operands of p, and the staged weights, into LDS; then
  // every operand in op
  auto exchange = [&](const Packed<2> &p) {
    __syncthreads();  // the old weights and operands are read
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) xch[sg][4 * fh + ks][lane] = __builtin_bit_cast(u32x4, operand(p, ks));
    next.store(W, tid);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) op[ks] = __builtin_bit_cast(bf16x8, xch[sg][ks][lane]);
  };
  // forward
  __syncthreads();
  // a 10-wide input has one step of 16; the second would add exact zeros
  c = A.in <= 16 ? product<2, 1, W0S>(W + 64 * fh * W0S, op, lane) : product<2, 2, W0S>(W + 64 * fh * W0S, op, lane);
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    if (l > 0) {
      exchange(act[l - 1]);
      next.load(l < 3 ? A.W16T + H * K0 + l * H * H : A.W16 + weight_offset(A.in, 3), tid);
      c = product<2, 8, WS>(W + 64 * fh * WS, op, lane);
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) bias_relu(c.a[rb], bias + l * H + 64 * fh + 32 * rb, lane, act[l].p[rb]);
    store_tile(act[l], bt, A.act, FA, A.in + l * H + 64 * fh, s0, lane);
  }
  // loss and its gradient, in both waves (lanes 0 .. 31 hold the samples); the
  // exchange leaves W_3, the first matrix of the way back, in LDS
  exchange(act[3]);
  next.load(A.W16 + weight_offset(A.in, 2), tid);
  const float y = last_output(op, W4, lane) + b4;
  float e = 0.f, g = 0.f;
  if (valid && hh == 0) {
    e = y - A.t[smp];
    g = 2.f * e * A.scale;
  }
  if (fh == 0) {
    float s = e * e;
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    float tot = __shfl(g, 0);  // the 32 rows in order
    for (int r = 1; r < 32; ++r) tot += __shfl(g, r);
    if (lane == 0 && s0 < A.n) {
      A.losspart[s0 >> 5] = s;
      A.colpart[size_t(s0 >> 5) * COLS + 4 * H] = tot;
    }
  }
  const uint32_t dy = pack_bf16(g, 0.f) & 0xffffu;
  if (hh == 0 && fh == 0) A.dz[by_sixteen(FD, 4 * H, smp)] = uint16_t(dy);
  const float dyf = __shfl(bf16_lo(dy), li);  // the sample's, in both halves
  // dZ_3 = dZ_4 W_4^T: one product each
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint2 w = *reinterpret_cast<const uint2 *>(W4 + 64 * fh + 32 * rb + 8 * q + 4 * hh);
      c.a[rb][4 * q] = dyf * bf16_lo(w.x);
      c.a[rb][4 * q + 1] = dyf * bf16_hi(w.x);
      c.a[rb][4 * q + 2] = dyf * bf16_lo(w.y);
      c.a[rb][4 * q + 3] = dyf * bf16_hi(w.y);
    }
#pragma unroll
  for (int l = 3; l >= 0; --l) {
    // ReLU' (A_{l+1} is not negative: a half that is not zero is positive), the
    // rows' sums in FP32, BF16
    Packed<2> p;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t w = act[l].p[rb][q][u];
          const float lo = (w & 0xffffu) != 0 ? c.a[rb][4 * q + 2 * u] : 0.f;
          const float hi = w > 0xffffu ? c.a[rb][4 * q + 2 * u + 1] : 0.f;
          c.a[rb][4 * q + 2 * u] = lo;
          c.a[rb][4 * q + 2 * u + 1] = hi;
          p.p[rb][q][u] = pack_bf16(lo, hi);
        }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) ft[(32 * rb + 8 * (r >> 2) + 4 * hh + (r & 3)) * FS + li] = c.a[rb][r];
    wave_order();
    {  // even rows, then odd rows, each in order
      const float *row = ft + lane * FS;
      float se = 0.f, so = 0.f;
#pragma unroll
      for (int r = 0; r < 32; r += 2) {
        se += row[r];
        so += row[r + 1];
      }
      if (s0 < A.n) A.colpart[size_t(s0 >> 5) * COLS + l * H + 64 * fh + lane] = se + so;
    }
    store_tile(p, bt, A.dz, FD, l * H + 64 * fh, s0, lane);
    if (l > 0) {
      if (l == 3) {  // W_3 is in LDS; the operands are not
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) xch[sg][4 * fh + ks][lane] = __builtin_bit_cast(u32x4, operand(p, ks));
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) op[ks] = __builtin_bit_cast(bf16x8, xch[sg][ks][lane]);
      } else {
        exchange(p);
        if (l == 2) next.load(A.W16 + weight_offset(A.in, 1), tid);
      }
      c = product<2, 8, WS>(W + 64 * fh * WS, op, lane);
    }
  }
}

// Weight gradients dW_l = A_l dZ_l over one chunk of kc samples, every layer in
// one launch: 64 x 64 tiles of the five matrices, four waves of 32 x 32.  Both
// operands lie as the MFMA takes them.  Blocks go to the XCDs in turn: the tiles of one chunk, which
// read the same 0.6 MB, stay on one XCD and meet in its L2.
struct GradArgs {
  const uint16_t *act, *dz;
  int n, in, kc, chunks;
  uint32_t nw;   // all weights
  float *part;   // [chunks][nw]
};
constexpr int GRAD_TILES = 2 + 3 * 4 + 2;
constexpr int XCDS = 8;
inline unsigned grad_blocks(int chunks) { return unsigned((chunks + XCDS - 1) / XCDS * XCDS * GRAD_TILES); }

__global__ void __launch_bounds__(256) k_train_grads(GradArgs A) {
  const int turn = int(blockIdx.x) / XCDS;
  const int chunk = int(blockIdx.x) % XCDS + XCDS * (turn / GRAD_TILES);
  if (chunk >= A.chunks) return;
  int job = turn % GRAD_TILES, l, tm = 0, tn = 0;
  if (job < 2) {
    l = 0;
    tn = 64 * job;
  } else if (job < 14) {
    l = 1 + (job - 2) / 4;
    tm = 64 * (((job - 2) & 3) >> 1);
    tn = 64 * ((job - 2) & 1);
  } else {
    l = 4;
    tm = 64 * (job - 14);
  }
  const int M = l == 0 ? A.in : H, N = l == 4 ? 1 : H;
  const int wave = int(threadIdx.x) >> 6, lane = int(threadIdx.x) & 63;
  tm += (wave >> 1) * 32;
  tn += (wave & 1) * 32;
  if (tm >= M || tn >= N) return;
  const int li = lane & 31, lk = (lane >> 5) * 8;
  const int kb = chunk * A.kc, ke = min(A.n, kb + A.kc);
  const bool ia = tm + li < M, ib = tn + li < N;
  const int FA = A.in + 4 * H, FD = COLS;
  // kb is a multiple of 16: step k0 lies (k0 - kb) / 16 rows of features on
  const uint16_t *ra = A.act + by_sixteen(FA, (l == 0 ? 0 : A.in + (l - 1) * H) + (ia ? tm + li : 0), kb) + lk;
  const uint16_t *rb = A.dz + by_sixteen(FD, l * H + (ib ? tn + li : 0), kb) + lk;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  // eight steps' loads in flight; columns past n hold zero gradients
  for (int k0 = kb; k0 < ke; k0 += 128) {
    u32x4 a[8], b[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const bool in = k0 + 16 * q < ke;
      a[q] = b[q] = u32x4{0, 0, 0, 0};
      if (in && ia) a[q] = *reinterpret_cast<const u32x4 *>(ra + size_t(k0 - kb + 16 * q) * FA);
      if (in && ib) b[q] = *reinterpret_cast<const u32x4 *>(rb + size_t(k0 - kb + 16 * q) * FD);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (k0 + 16 * q < ke)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[q]),
                                                      __builtin_bit_cast(bf16x8, b[q]), acc, 0, 0, 0);
  }
  float *out = A.part + size_t(chunk) * A.nw + weight_offset(A.in, l);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = tm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = tn + li;
    if (row < M && col < N) out[size_t(row) * N + col] = acc[r];
  }
}

// The sums: chunks of the weight gradients in order (blocks 0 .. wblocks - 1),
// 32-row sums of the bias gradients as k_colsum_fin (one block a column), and
// the squared errors (the last block).
struct SumArgs {
  const float *part, *colpart, *losspart;
  int splits, nb;     // chunks, rows of 32
  uint32_t nw, wblocks;
  float *gW, *gb;     // layers concatenated
  float *loss, *host_loss;
};
constexpr int SUM_BLOCK = 256;

__global__ void __launch_bounds__(SUM_BLOCK) k_train_sums(SumArgs A) {
  __shared__ float red[SUM_BLOCK];
  const int t = int(threadIdx.x);
  if (blockIdx.x < A.wblocks) {
    const uint32_t e = blockIdx.x * SUM_BLOCK + t;
    if (e >= A.nw) return;
    float s = A.part[e];
    // sixteen loads in flight ahead of their additions, whatever the number of
    // chunks (a power of two up to 64: one to four batches after the first)
    for (int z = 1; z < A.splits; z += 16) {
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = z + k < A.splits ? A.part[size_t(z + k) * A.nw + e] : 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (z + k < A.splits) s += v[k];
    }
    A.gW[e] = s;
    return;
  }
  const int col = int(blockIdx.x - A.wblocks);
  const bool is_loss = col == COLS;
  float s = 0.f;
  for (int b = t; b < A.nb; b += SUM_BLOCK) s += is_loss ? A.losspart[b] : A.colpart[size_t(b) * COLS + col];
  red[t] = s;
  __syncthreads();
  for (int w = SUM_BLOCK / 2; w > 0; w >>= 1) {
    if (t < w) red[t] += red[t + w];
    __syncthreads();
  }
  if (t == 0) {
    if (is_loss) {
      *A.loss = red[0];
      if (A.host_loss) *A.host_loss = red[0];
    } else {
      A.gb[col] = red[0];
    }
  }
}

// the transposed BF16 copy's place of weight i (layers concatenated), -1: none
__host__ __device__ inline int64_t transposed_index(int in, int64_t i) {
  if (i < int64_t(in) * H) return (i % H) * K0 + i / H;
  i -= int64_t(in) * H;
  if (i >= 3 * H * H) return -1;
  const int64_t l = i / (H * H), e = i % (H * H);
  return H * K0 + l * H * H + (e % H) * H + e / H;
}
constexpr int64_t TRANSPOSED_SIZE = H * K0 + 3 * H * H;

}  // namespace chain
}  // namespace casl
