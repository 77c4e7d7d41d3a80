// scx_mlp.hip -- the learned warm start: a 16-128-128-3 multilayer perceptron (ReLU)
// in BF16 with FP32 accumulation on the matrix cores, inference over the active set and
// training (forward + backward, weight gradients, Adam) on collected samples.
//
// Every product is a 16x16x16 MFMA tile (v_mfma_f32_16x16x16_bf16) computed in the
// transposed form Out^T = W^T In^T, with samples on the N side: lane l holds sample
// l % 16, and the accumulator of one layer (rows 4 (l / 16) + e, column l % 16) is
// already the B operand of the next layer's K-tile, so activations stay in registers
// between layers. Weights are kept as the A operands themselves, fragment after fragment
// (64 lanes of 4 BF16), so a wave reads one as 512 consecutive bytes. Weight gradients are
// MFMAs with the samples as the K dimension, over activations stored unit-major per
// 16-sample tile.
#include "scx_device.h"
#include "scx_internal.h"

namespace scx {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN kept quiet); BF16 -> FP32 is exact.
__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// BF16 weight copies as A fragments: element (row i, column k) of a 16x16 tile is entry
// k % 4 of lane i + 16 (k / 4).
//   w1t [8]    tiles ut of W1^T [128][16]   (forward, layer 1)
//   w2t [8][8] tiles (ut, kt) of W2^T       (forward, layer 2)
//   w3t [8]    tiles kt of W3^T [16][128]   (forward, layer 3; rows 3 to 15 zero)
//   w2n [8][8] tiles (ut, kt) of W2         (backward, dH1 = W2 dH2)
//   w3n [8]    tiles ut of W3 [128][16]     (backward, dH2 = W3 dY; columns 3 to 15 zero)
// biases FP32: b1 [128], b2 [128], b3 [16] (3 used).
constexpr int kFrag = 256;  // BF16 of a fragment
constexpr int kW1T = 0, kW2T = kW1T + 8 * kFrag, kW3T = kW2T + 64 * kFrag, kForwardBf16 = kW3T + 8 * kFrag,
              kW2N = kForwardBf16, kW3N = kW2N + 64 * kFrag;
constexpr int kB1 = 0, kB2 = kMlpHid, kB3 = 2 * kMlpHid, kPackedBias = 2 * kMlpHid + 16;

// Place of element (i, k) of a matrix in its fragments, `kts` of them per row of tiles.
__device__ __forceinline__ uint32_t frag_at(uint32_t i, uint32_t k, uint32_t kts) {
  return ((i >> 4) * kts + (k >> 4)) * kFrag + ((i & 15) + 16 * ((k & 15) >> 2)) * 4 + (k & 3);
}

__global__ void __launch_bounds__(kBlock) k_mlp_pack(const float* __restrict__ p, uint16_t* __restrict__ w,
                                                     float* __restrict__ bias) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < kMlpHid * kMlpIn) {  // W1 [k][u], k < 16
    const uint32_t k = i / kMlpHid, u = i % kMlpHid;
    w[kW1T + frag_at(u, k, 1)] = f2bf(p[kMlpOffW1 + i]);
  }
  if (i < kMlpHid * kMlpHid) {  // W2 [u][v]
    const uint32_t u = i / kMlpHid, v = i % kMlpHid;
    const uint16_t h = f2bf(p[kMlpOffW2 + i]);
    w[kW2T + frag_at(v, u, 8)] = h;
    w[kW2N + frag_at(u, v, 8)] = h;
  }
  if (i < kMlpHid * 16) {  // W3 [v][o], padded to 16 outputs
    const uint32_t v = i / 16, o = i % 16;
    const uint16_t h = (o < (uint32_t)kMlpOut) ? f2bf(p[kMlpOffW3 + v * kMlpOut + o]) : (uint16_t)0;
    w[kW3T + frag_at(o, v, 8)] = h;
    w[kW3N + frag_at(v, o, 1)] = h;
  }
  if (i < kMlpHid) {
    bias[kB1 + i] = p[kMlpOffB1 + i];
    bias[kB2 + i] = p[kMlpOffB2 + i];
  }
  if (i < 16) bias[kB3 + i] = (i < (uint32_t)kMlpOut) ? p[kMlpOffB3 + i] : 0.f;
}

__device__ __forceinline__ bf16x4 frag(const uint16_t* w, int f, int lane) {
  return reinterpret_cast<const bf16x4*>(w)[f * 64 + lane];
}

// BF16 of relu(x + bias)
__device__ __forceinline__ bf16x4 relu4(f32x4 x, const float* bias) {
  bf16x4 h;
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = (short)f2bf(fmaxf(x[e] + bias[e], 0.f));
  return h;
}
// BF16 gradient, masked by the activation h > 0
__device__ __forceinline__ bf16x4 masked4(f32x4 x, bf16x4 h) {
  bf16x4 g;
#pragma unroll
  for (int e = 0; e < 4; ++e) g[e] = (short)((h[e] != 0 && (h[e] & 0x8000) == 0) ? f2bf(x[e]) : 0);
  return g;
}

// The forward pass of one 16-sample tile in one wave. x: the tile's B operand (features
// 4 (lane / 16) + e of sample lane % 16). Result: outputs o = 4 (lane / 16) + e of sample
// lane % 16 (o < 3 meaningful).
__device__ __forceinline__ f32x4 forward_tile(const uint16_t* w, const float* bias, bf16x4 x, int lane) {
  const int r = 4 * (lane >> 4);
  bf16x4 h1[8], h2[8];
#pragma unroll
  for (int ut = 0; ut < 8; ++ut)
    h1[ut] = relu4(mfma16(frag(w + kW1T, ut, lane), x, f32x4{0, 0, 0, 0}), bias + kB1 + ut * 16 + r);
#pragma unroll
  for (int ut = 0; ut < 8; ++ut) {
    f32x4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) acc = mfma16(frag(w + kW2T, ut * 8 + kt, lane), h1[kt], acc);
    h2[ut] = relu4(acc, bias + kB2 + ut * 16 + r);
  }
  f32x4 y = {0, 0, 0, 0};
#pragma unroll
  for (int kt = 0; kt < 8; ++kt) y = mfma16(frag(w + kW3T, kt, lane), h2[kt], y);
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] += bias[kB3 + r + e];
  return y;
}

// Features of sample s (row-major [n][16] FP32) as the tile's B operand.
__device__ __forceinline__ bf16x4 x_frag(const float* X, uint32_t n, uint32_t s, int lane) {
  bf16x4 x = {0, 0, 0, 0};
  if (s < n) {
    const float4 v = *reinterpret_cast<const float4*>(X + (size_t)s * kMlpIn + 4 * (lane >> 4));
    x[0] = (short)f2bf(v.x);
    x[1] = (short)f2bf(v.y);
    x[2] = (short)f2bf(v.z);
    x[3] = (short)f2bf(v.w);
  }
  return x;
}

// Weights and biases into LDS (all threads of the block).
__device__ __forceinline__ void stage_weights(const uint16_t* __restrict__ gw, const float* __restrict__ gb,
                                              uint16_t* sw, float* sb, int count) {
  const uint4* src = reinterpret_cast<const uint4*>(gw);
  uint4* dst = reinterpret_cast<uint4*>(sw);
  for (int i = threadIdx.x; i < count / 8; i += blockDim.x) dst[i] = src[i];
  for (int i = threadIdx.x; i < kPackedBias; i += blockDim.x) sb[i] = gb[i];
  __syncthreads();
}

// The perceptron predicts a correction to the transported cached impulse: the prediction
// of a sample is MLP(x) + x[kMlpBase .. kMlpBase + 2] (features 8-10), so an untrained or
// zero network reproduces the transported-cache warm start.
constexpr int kMlpBase = 8;

// Inference: Y [n][3] = MLP(X [n][16]) + X[:, 8:11]. One wave per 16-sample tile, grid-stride.
__global__ void __launch_bounds__(kBlock) k_mlp_infer(uint32_t n, const float* __restrict__ X,
                                                      const uint16_t* __restrict__ gw, const float* __restrict__ gb,
                                                      float* __restrict__ Y) {
  __shared__ __attribute__((aligned(16))) uint16_t sw[kForwardBf16];
  __shared__ float sb[kPackedBias];
  stage_weights(gw, gb, sw, sb, kForwardBf16);
  const int lane = threadIdx.x & 63;
  const uint32_t wave = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const uint32_t nwaves = gridDim.x * (kBlock / 64);
  const uint32_t ntiles = (n + 15) / 16;
  for (uint32_t t = wave; t < ntiles; t += nwaves) {
    const uint32_t s = t * 16 + (lane & 15);
    const f32x4 y = forward_tile(sw, sb, x_frag(X, n, s, lane), lane);
    // outputs 0..2 of sample lane are in lanes 0..15, elements 0..2
    if (lane < 16 && s < n)
#pragma unroll
      for (int o = 0; o < kMlpOut; ++o) Y[(size_t)s * kMlpOut + o] = y[o] + X[(size_t)s * kMlpIn + kMlpBase + o];
  }
}

// Training, pass 1: forward and backward of each 16-sample tile of a batch (samples
// idx[b0 .. b0 + nb) of the pool, or b0 + i when idx is null). Loss = mean over samples
// and outputs of (y + x[8:11] - t)^2. Stores per tile, BF16, unit-major with the 16 samples
// contiguous: H1T, H2T [tile][128][16], G1T, G2T (gradients w.r.t. the pre-activations)
// [tile][128][16], GY [tile][16][16] (dLoss/dy, outputs padded to 16), XT [tile][16][16]
// (features), and the block's sum of squared errors.
//
// A batch of 2,048 samples is 128 tiles: what bounds the pass is the latency of one tile, not
// the 0.2 GFLOP or the 2 MB. So a tile is shared by four waves, each with two of the eight
// 16-unit tiles of every layer and only their weight fragments (44, in registers, loaded once
// and together instead of 78 KB staged through LDS); the activations, in the accumulators'
// layout, which is the next layer's operand, pass through LDS. The order of every sum is that
// of one wave's chain over kt. 2,048 samples: 7 us (one wave per tile, weights in LDS: 29 us).
struct TrainBufs {
  uint16_t* h1t;
  uint16_t* h2t;
  uint16_t* g1t;
  uint16_t* g2t;
  uint16_t* gy;
  uint16_t* xt;
  float* sse;  // per block
};

__global__ void __launch_bounds__(kBlock) k_mlp_fwdbwd(uint32_t nb, const uint32_t* __restrict__ idx, uint32_t b0,
                                                       const float* __restrict__ X, const float* __restrict__ Tgt,
                                                       const uint16_t* __restrict__ gw, const float* __restrict__ gb,
                                                       float loss_scale, TrainBufs B) {
  static_assert(kBlock == 256, "four waves, two unit tiles each");
  __shared__ bf16x4 s_h1[8][64], s_h2[8][64], s_g2[8][64];
  const int lane = threadIdx.x & 63;
  const int r = 4 * (lane >> 4), sl = lane & 15;
  const int u0 = 2 * (int)(threadIdx.x >> 6);  // the wave's unit tiles: u0, u0 + 1
  const uint32_t ntiles = (nb + 15) / 16;
  // the sample of this lane in tile t; read ahead of the weights and of the tile before, as its
  // features wait for it
  auto sample = [&](uint32_t t) {
    const uint32_t i = t * 16 + sl;
    return i < nb ? (idx ? idx[b0 + i] : b0 + i) : 0u;
  };
  uint32_t ahead = sample(blockIdx.x);
  bf16x4 w1[2], w2[2][8], w3[8], n3[2], n2[2][8];
  float b1[2][4], b2[2][4], b3[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    w1[i] = frag(gw + kW1T, u0 + i, lane);
    n3[i] = frag(gw + kW3N, u0 + i, lane);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      w2[i][kt] = frag(gw + kW2T, (u0 + i) * 8 + kt, lane);
      n2[i][kt] = frag(gw + kW2N, (u0 + i) * 8 + kt, lane);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      b1[i][e] = gb[kB1 + (u0 + i) * 16 + r + e];
      b2[i][e] = gb[kB2 + (u0 + i) * 16 + r + e];
    }
  }
#pragma unroll
  for (int kt = 0; kt < 8; ++kt) w3[kt] = frag(gw + kW3T, kt, lane);
#pragma unroll
  for (int e = 0; e < 4; ++e) b3[e] = gb[kB3 + r + e];
  float sse = 0.f;
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const bool valid = t * 16 + sl < nb;
    const uint32_t s = ahead;
    ahead = sample(t + gridDim.x);
    const bf16x4 x = valid ? x_frag(X, 0xFFFFFFFFu, s, lane) : bf16x4{0, 0, 0, 0};
    float base[kMlpOut], tgt[kMlpOut];
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) {
      base[o] = X[(size_t)s * kMlpIn + kMlpBase + o];
      tgt[o] = Tgt[(size_t)s * kMlpOut + o];
    }
    bf16x4 h1[2], h2[2], g1[2], g2[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      h1[q] = relu4(mfma16(w1[q], x, f32x4{0, 0, 0, 0}), b1[q]);
      s_h1[u0 + q][lane] = h1[q];
    }
    __syncthreads();
    f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      const bf16x4 h = s_h1[kt][lane];
      acc[0] = mfma16(w2[0][kt], h, acc[0]);
      acc[1] = mfma16(w2[1][kt], h, acc[1]);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      h2[q] = relu4(acc[q], b2[q]);
      s_h2[u0 + q][lane] = h2[q];
    }
    __syncthreads();
    // every wave computes the outputs and dLoss/dy, for outputs o = r + e < 3
    f32x4 y = {0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) y = mfma16(w3[kt], s_h2[kt][lane], y);
    bf16x4 gy = {0, 0, 0, 0};
    if (valid && r == 0) {
#pragma unroll
      for (int o = 0; o < kMlpOut; ++o) {
        const float d = ((y[o] + b3[o]) + base[o]) - tgt[o];
        sse += d * d;
        gy[o] = (short)f2bf(loss_scale * 2.f * d);
      }
    }
    // dH2 = W3 dY, masked by h2 > 0
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      g2[q] = masked4(mfma16(n3[q], gy, f32x4{0, 0, 0, 0}), h2[q]);
      s_g2[u0 + q][lane] = g2[q];
    }
    __syncthreads();
    // dH1 = W2 dH2, masked by h1 > 0
    acc[0] = acc[1] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      const bf16x4 g = s_g2[kt][lane];
      acc[0] = mfma16(n2[0][kt], g, acc[0]);
      acc[1] = mfma16(n2[1][kt], g, acc[1]);
    }
    // (the next tile writes a buffer of this one only behind a barrier that its readers pass
    // after reading it)
    // stores: element (unit ut*16 + r + e, sample lane % 16) of each tile block
    const size_t tb = (size_t)t * kMlpHid * 16;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      g1[q] = masked4(acc[q], h1[q]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const size_t o = tb + (size_t)((u0 + q) * 16 + r + e) * 16 + sl;
        B.h1t[o] = (uint16_t)h1[q][e];
        B.h2t[o] = (uint16_t)h2[q][e];
        B.g1t[o] = (uint16_t)g1[q][e];
        B.g2t[o] = (uint16_t)g2[q][e];
      }
    }
    if (u0 == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        B.gy[(size_t)t * 256 + (r + e) * 16 + sl] = (uint16_t)gy[e];
        B.xt[(size_t)t * 256 + (r + e) * 16 + sl] = (uint16_t)x[e];
      }
    }
  }
  sse = wave_reduce_sum_f32(sse);
  if (threadIdx.x == 0) B.sse[blockIdx.x] = sse;
}

// Adam (Kingma & Ba 2015) on the FP32 parameters, bias-corrected.
struct Adam {
  float* p;
  float* m;
  float* v;
  uint16_t* w;  // the packed copies of the new parameters
  float* bias;
  float lr, b1, b2, eps, c1, c2;
  __device__ __forceinline__ float step(uint32_t i, float pi, float mi, float vi, float gi) const {
    // (one rounding each fixed by hand: a small gradient's step has the size of the rate either
    // way its moments round, so steps repeat only to the bit)
    mi = fmaf(1.f - b1, gi, b1 * mi);
    vi = fmaf(gi, (1.f - b2) * gi, b2 * vi);
    m[i] = mi;
    v[i] = vi;
    pi -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    return pi;
  }
};

// Training, pass 2: weight gradients, one wave per 16x16 output tile, K = samples:
//   dW1 [16][128]  = X^T G1     (8 tiles: columns of 16 hidden units)
//   dW2 [128][128] = H1^T G2    (64 tiles)
//   dW3 [128][3]   = H2^T GY    (8 tiles: rows of 16 hidden units)
// A operand: rows of the unit-major activations (4 consecutive samples per lane), B
// operand: the gradient tile's rows likewise (element (k = sample, n = unit)).
// Bias gradients (sums over samples of G1, G2, GY) ride along on the first tiles.
//
// A wave's chain of products over the sample tiles is serial (its order is the order of the
// sums), so the pass is bound by that chain, 128 dependent products for 2,048 samples, once the
// loads no longer stand in it: they run kAhead tiles in front, in registers. One wave per
// workgroup, each with a CU of its own; the eight waves that read the same rows of H1 are on
// one XCD. kTrain: every parameter's gradient is in one lane's hands, which takes the Adam
// step itself and writes the packed copies; otherwise the gradients are the result. 2,048 samples
// with the Adam step: 9 us (loads inside the chain, four waves per workgroup, Adam and the
// packing in launches of their own: 36 us and two launches).
constexpr uint32_t kAhead = 16;

template <bool kTrain>
__global__ void __launch_bounds__(64) k_mlp_wgrad(uint32_t ntiles, TrainBufs B, float* __restrict__ grad, Adam A) {
  const int lane = threadIdx.x;
  const int r = 4 * (lane >> 4), n = lane & 15;
  const uint32_t job = blockIdx.x;
  const uint32_t mt = job < 64 ? job % 8 : job < 72 ? 0 : job - 72;  // row tile
  const uint32_t nt = job < 64 ? job / 8 : job < 72 ? job - 64 : 0;  // column tile
  const uint16_t *am, *bm;
  uint32_t ald = kMlpHid * 16, bld = kMlpHid * 16, off, ldo;  // strides of a sample tile; the result's place
  if (job < 64) {  // dW2 tile (mt, nt)
    am = B.h1t;
    bm = B.g2t;
    off = kMlpOffW2;
    ldo = kMlpHid;
  } else if (job < 72) {  // dW1 tile (rows 0..15, units nt*16..)
    am = B.xt;
    ald = 256;
    bm = B.g1t;
    off = kMlpOffW1;
    ldo = kMlpHid;
  } else {  // dW3 tile (rows of units mt*16.., outputs 0..15)
    am = B.h2t;
    bm = B.gy;
    bld = 256;
    off = kMlpOffW3;
    ldo = kMlpOut;
  }
  const bool used = job < 72 || n < kMlpOut;
  off += (mt * 16 + r) * ldo + nt * 16 + n;  // of element (r, n); (r + e, n) follow at ldo each
  // the bias with this wave: gradient of column n
  const bool has_bias = mt == 0 && (job < 72 || n < kMlpOut);
  const uint32_t boff = (job < 64 ? kMlpOffB2 : job < 72 ? kMlpOffB1 : kMlpOffB3) + nt * 16 + n;
  float p[5], m[5], v[5];
  if (kTrain) {
#pragma unroll
    for (int e = 0; e < 5; ++e) {
      const uint32_t i = e < 4 ? off + e * ldo : boff;
      if (e < 4 ? used : has_bias) p[e] = A.p[i], m[e] = A.m[i], v[e] = A.v[i];
    }
  }
  am += mt * 256 + n * 16 + r;
  bm += nt * 256 + n * 16 + r;
  bf16x4 a[2][kAhead], b[2][kAhead];
  auto load = [&](int k, uint32_t t0) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
      const uint32_t t = min(t0 + i, ntiles - 1);  // (past the end: not used)
      a[k][i] = *reinterpret_cast<const bf16x4*>(am + (size_t)t * ald);
      b[k][i] = *reinterpret_cast<const bf16x4*>(bm + (size_t)t * bld);
    }
  };
  f32x4 acc = {0, 0, 0, 0};
  float bsum = 0.f;
  auto add = [&](bf16x4 x, bf16x4 y) __attribute__((always_inline)) {
    acc = mfma16(x, y, acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) bsum += bf2f((uint16_t)y[e]);
  };
  auto sum = [&](int k, uint32_t t0) __attribute__((always_inline)) {
    if (t0 + kAhead <= ntiles) {
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i) add(a[k][i], b[k][i]);
    } else {
#pragma unroll
      for (uint32_t i = 0; i < kAhead; ++i)
        if (t0 + i < ntiles) add(a[k][i], b[k][i]);
    }
  };
  load(0, 0);
  for (uint32_t t0 = 0; t0 < ntiles; t0 += 2 * kAhead) {
    load(1, t0 + kAhead);
    sum(0, t0);
    load(0, t0 + 2 * kAhead);
    sum(1, t0 + kAhead);
  }
  // lanes with the same lane % 16 hold partial sums over their samples
  bsum += __shfl_xor(bsum, 16, 64);
  bsum += __shfl_xor(bsum, 32, 64);
  if (!kTrain) {
    if (used)
#pragma unroll
      for (int e = 0; e < 4; ++e) grad[off + e * ldo] = acc[e];
    if (has_bias && lane < 16) grad[boff] = bsum;
    return;
  }
  bf16x4 h = {0, 0, 0, 0};
  if (used)
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = (short)f2bf(A.step(off + e * ldo, p[e], m[e], v[e], acc[e]));
  if (has_bias && lane < 16)
    A.bias[(job < 64 ? kB2 : job < 72 ? kB1 : kB3) + nt * 16 + n] = A.step(boff, p[4], m[4], v[4], bsum);
  // element (r + e, n) of the tile: the transposed copy's fragment has it in this lane
  bf16x4* w = reinterpret_cast<bf16x4*>(A.w);
  if (job < 64) {
    w[kW2T / 4 + (nt * 8 + mt) * 64 + lane] = h;
#pragma unroll
    for (int e = 0; e < 4; ++e) A.w[kW2N + frag_at(mt * 16 + r + e, nt * 16 + n, 8)] = (uint16_t)h[e];
  } else if (job < 72) {
    w[kW1T / 4 + nt * 64 + lane] = h;
  } else {
    w[kW3T / 4 + mt * 64 + lane] = h;
#pragma unroll
    for (int e = 0; e < 4; ++e) A.w[kW3N + frag_at(mt * 16 + r + e, n, 1)] = (uint16_t)h[e];
  }
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
hipError_t launch_mlp_pack(scx_ctx* c) {
  const uint32_t nb = (kMlpHid * kMlpHid + kBlock - 1) / kBlock;
  k_mlp_pack<<<nb, kBlock, 0, c->stream>>>(c->d.mlp_params, c->d.mlp_w, c->d.mlp_b);
  return hipGetLastError();
}

hipError_t launch_mlp_infer(scx_ctx* c, uint32_t n, const float* X, float* Y) {
  const uint32_t ntiles = (n + 15) / 16;
  if (ntiles == 0) return hipSuccess;
  const uint32_t blocks = std::min<uint32_t>((ntiles + 3) / 4, 4u * (uint32_t)c->num_cus);
  k_mlp_infer<<<blocks, kBlock, 0, c->stream>>>(n, X, c->d.mlp_w, c->d.mlp_b, Y);
  return hipGetLastError();
}

// One batch: forward/backward over samples idx[b0 .. b0 + nb) (idx null: b0 + i) of
// (X, Tgt), squared-error partials into d.mlp_sse. step > 0: an Adam step with rate lr; 0: the
// gradients into d.mlp_grad.
static hipError_t launch_batch(scx_ctx* c, uint32_t nb, const uint32_t* idx, uint32_t b0, const float* X,
                               const float* Tgt, float lr, uint32_t step) {
  DeviceBuffers& d = c->d;
  const uint32_t ntiles = (nb + 15) / 16;
  if (ntiles == 0 || ntiles > d.mlp_cap_tiles) return hipErrorInvalidValue;
  const size_t act = (size_t)d.mlp_cap_tiles * kMlpHid * 16;
  TrainBufs B{d.mlp_act, d.mlp_act + act, d.mlp_act + 2 * act, d.mlp_act + 3 * act, d.mlp_act + 4 * act,
              d.mlp_act + 4 * act + (size_t)d.mlp_cap_tiles * 256, d.mlp_sse};
  const uint32_t blocks = std::min<uint32_t>(ntiles, (uint32_t)kMlpSseBlocks);
  d.mlp_sse_blocks = blocks;  // the loss partials this pass writes
  k_mlp_fwdbwd<<<blocks, kBlock, 0, c->stream>>>(nb, idx, b0, X, Tgt, d.mlp_w, d.mlp_b,
                                                  1.0f / ((float)nb * (float)kMlpOut), B);
  const float b1 = 0.9f, b2 = 0.999f;
  Adam A{d.mlp_params, d.mlp_m, d.mlp_v, d.mlp_w, d.mlp_b, lr, b1, b2, 1e-8f, 1.f - powf(b1, (float)step),
         1.f - powf(b2, (float)step)};
  if (step > 0) k_mlp_wgrad<true><<<80, 64, 0, c->stream>>>(ntiles, B, nullptr, A);
  else k_mlp_wgrad<false><<<80, 64, 0, c->stream>>>(ntiles, B, d.mlp_grad, A);
  return hipGetLastError();
}

hipError_t launch_mlp_gradients(scx_ctx* c, uint32_t nb, const uint32_t* idx, uint32_t b0, const float* X,
                                const float* Tgt) {
  return launch_batch(c, nb, idx, b0, X, Tgt, 0.f, 0);
}

hipError_t launch_mlp_train(scx_ctx* c, uint32_t nb, const uint32_t* idx, uint32_t b0, const float* X,
                            const float* Tgt, float lr, uint32_t step) {
  return launch_batch(c, nb, idx, b0, X, Tgt, lr, step);
}

}  // namespace scx
