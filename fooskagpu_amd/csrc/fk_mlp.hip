// Surrogate of the phase-relaxation Newton solve: a 3-64-64-64-3 tanh MLP
// mapping (log rho, e, alpha_L) of a cell to the equilibrium (T, asinh(p /
// 1e4), alpha_L) that warm-starts an FP64 Newton polish.  No counterpart in
// the reference (its relaxation.cu / thermRlx.cu / chemRlx.cu always start
// from the cell state).
//
// Numerics of the network (the CPU check restates the same; inference takes
// tanh as tanh_fast, within ~1e-7 of it, training tanhf):
//   layer 1: FP32 FMA, tanh, rounded to BF16
//   layers 2, 3: BF16 x BF16 MFMA (v_mfma_f32_16x16x32_bf16), FP32
//                accumulate, + bias, tanh, rounded to BF16
//   layer 4: FP32 FMA on the BF16 activations
// Operand layouts of v_mfma_f32_16x16x32_bf16 (one wave, lane l):
//   A (16x32, row m, col k):  A[l % 16][8 (l / 16) + i], i = 0..7
//   B (32x16, row k, col n):  B[8 (l / 16) + i][l % 16]
//   D (16x16):                D[4 (l / 16) + i][l % 16], i = 0..3
// Training: per-wave forward + backward over 32-sample chunks, weight
// gradients by MFMA with the sample index as K, per-wave partial sums
// reduced in a fixed order (deterministic), then Adam on FP32 master weights.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/fooska.h"
#include "fk_device.h"
#include "fk_internal.h"
#include "fk_relax.h"
#include "fk_xfer.h"

using namespace fkx;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

constexpr int HID = 64;
constexpr int kParams = 8771;
constexpr int oW1 = 0, oB1 = 192, oW2 = 256, oB2 = 4352, oW3 = 4416, oB3 = 8512, oW4 = 8576, oB4 = 8768;
// BF16 copies (uint16 offsets): W2, W3 row-major [out][in], W2T, W3T [in][out]
constexpr int bW2 = 0, bW3 = 4096, bW2T = 8192, bW3T = 12288, kBf = 16384;
constexpr float kPScale = 1e4f;  // pressure target is asinh(p / kPScale)

struct Norm {
  float xm[3], xs[3], ym[3], ys[3];
};

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  const uint32_t u = __float_as_uint(f);
  uint32_t r = (u + (0x7fffu + ((u >> 16) & 1u))) >> 16, n = (u >> 16) | 0x40;  // NaN stays NaN
  asm("" : "+v"(r), "+v"(n));  // a select, not a branch around either
  return (uint16_t)((u & 0x7fffffffu) > 0x7f800000u ? n : r);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

// tanh(z) = 1 - 2 / (1 + e^(2z)) with the hardware exponential and
// reciprocal: within about 1e-7 of tanh, far below the BF16 rounding
// (2^-9 relative) of every activation.  Inference only (the relaxation's
// warm start); training and its CPU check use tanhf.
__device__ __forceinline__ float tanh_fast(float z) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __expf(2.f * z));
}

__device__ __forceinline__ bf16x8 ld_bf8(const uint16_t *p) {  // 16-byte aligned
  return *reinterpret_cast<const bf16x8 *>(p);
}

// Row strides in LDS: 64 (or 32) values padded by 8, so that the 16 rows of an
// MFMA operand start in different banks (unpadded, 128-byte rows put them all
// in two).
constexpr int kRow = HID + 8, kRowT = 32 + 8;

// Per-wave LDS scratch of the forward pass over 16 samples.
struct FwdLds {
  uint16_t h[16 * kRow];  // activations of the current layer, [m][k]
  float x[16 * 3];
  float y[16 * 3];
};

// The FP32 parameters of the forward pass, copied into LDS once per block:
// layer 1 as (W1 row k, b1[k]) quads, the biases of layers 2 and 3, W4, b4.
struct SmallW {
  float4 w1b[HID];
  float b2[HID], b3[HID];
  __attribute__((aligned(16))) float w4[3 * HID];
  float b4[4];
};

// Forward of 16 samples by one wave (inference: tanh_fast).  x: LDS [16][3]
// (normalised), result in lds.y [16][3] (normalised).  Weights: sw (LDS: W1,
// b1, b2, b3, W4, b4), bf16 wb in LDS (W2, W3, rows of kRow).
__device__ __forceinline__ void mlp_fwd16(const SmallW &sw, const uint16_t *wb, FwdLds &lds) {
  const int l = threadIdx.x & 63;
  const int m = l & 15, q = l >> 4;
  // layer 1 (FP32): this lane computes neurons k = 32 ks + 8 q + i of sample m
  const float x0 = lds.x[m * 3 + 0], x1 = lds.x[m * 3 + 1], x2 = lds.x[m * 3 + 2];
  bf16x8 a[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = 32 * ks + 8 * q + i;
      const float4 c = sw.w1b[k];
      const float z = c.w + c.x * x0 + c.y * x1 + c.z * x2;
      a[ks][i] = __builtin_bit_cast(__bf16, f2bf(tanh_fast(z)));
    }
  // layers 2 and 3 (BF16 MFMA)
#pragma unroll
  for (int layer = 0; layer < 2; ++layer) {
    const uint16_t *W = wb + (layer == 0 ? 0 : HID * kRow);
    const float *bias = layer == 0 ? sw.b2 : sw.b3;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      const int n = 16 * nt + m;  // B column of this lane
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8 b = ld_bf8(W + n * kRow + 32 * ks + 8 * q);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks], b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * q + i;
        lds.h[row * kRow + n] = f2bf(tanh_fast(acc[i] + bias[n]));
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a[ks] = ld_bf8(lds.h + m * kRow + 32 * ks + 8 * q);
    __builtin_amdgcn_wave_barrier();
  }
  // layer 4 (FP32) on the last activations: this lane's 16 neurons of sample
  // m (in a[]), then the sum over the sample's 4 lanes q = 0..3,
  // (p_0 + p_1) + (p_2 + p_3) on every one of them
  float p[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    // the whole vector reinterpreted (a bit_cast of one element of a[ks]
    // reads element 0)
    const u16x8 ab = __builtin_bit_cast(u16x8, a[ks]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float h = bf2f(ab[i]);
      const int k = 32 * ks + 8 * q + i;
#pragma unroll
      for (int j = 0; j < 3; ++j) p[j] += sw.w4[j * HID + k] * h;
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    p[j] += __shfl_xor(p[j], 16, 64);
    p[j] += __shfl_xor(p[j], 32, 64);
  }
  if (q == 0)
#pragma unroll
    for (int j = 0; j < 3; ++j) lds.y[m * 3 + j] = sw.b4[j] + p[j];
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_wave_barrier();
}

// Copies of the weights into LDS by blocks of NT threads: the FP32 forward
// parameters (SmallW, as one array) and the first ROWS rows of the BF16
// weights, padded.  Neither part has a branch, so that all loads go out before
// the first is stored: a block begins with one memory latency, not one for
// each.
template <int ROWS, int NT>
struct WeightCopy {
  static constexpr int K = ROWS * (HID / 8) / NT, S = 9 * HID + 3, KS = (S + NT - 1) / NT;
  static_assert(K * NT == ROWS * (HID / 8), "whole words per thread");
  uint4 v[K];
  float c[KS];
  // parameter behind float j of SmallW
  static __device__ __forceinline__ int param(int j) {
    const int r = j >> 2, k = j & 3;
    int p = k < 3 ? oW1 + 3 * r + k : oB1 + r;
    if (j >= 4 * HID) p = oB2 + j - 4 * HID;
    if (j >= 5 * HID) p = oB3 + j - 5 * HID;
    if (j >= 6 * HID) p = oW4 + j - 6 * HID;
    if (j >= 9 * HID) p = oB4 + (j < S ? j - 9 * HID : 0);
    return p;
  }
  __device__ __forceinline__ void load(const float *__restrict__ w, const uint16_t *__restrict__ g) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = reinterpret_cast<const uint4 *>(g)[k * NT + threadIdx.x];
#pragma unroll
    for (int k = 0; k < KS; ++k) c[k] = w[param(k * NT + threadIdx.x)];
  }
  __device__ __forceinline__ void store(SmallW &s, uint16_t *wb) const {
    static_assert(offsetof(SmallW, b2) == 16 * HID && offsetof(SmallW, b3) == 20 * HID &&
                  offsetof(SmallW, w4) == 24 * HID && offsetof(SmallW, b4) == 36 * HID, "SmallW as one array");
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int j = k * NT + threadIdx.x;
      reinterpret_cast<float *>(&s)[j < S ? j : S] = c[k];  // the rest on the spare word b4[3]
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int j = k * NT + threadIdx.x, row = j / (HID / 8), col = j % (HID / 8) * 8;
      *reinterpret_cast<uint4 *>(wb + row * kRow + col) = v[k];
    }
  }
};
template <int ROWS>
__device__ __forceinline__ void load_weights(const float *__restrict__ w, const uint16_t *__restrict__ g, SmallW &s,
                                             uint16_t *wb) {
  WeightCopy<ROWS, 256> wc;
  wc.load(w, g);
  wc.store(s, wb);
  __syncthreads();
}

// Inference on host-provided inputs x [n][3] (raw features) -> y [n][3] (raw
// targets).  Grid-stride over 64-sample chunks per wave.
__global__ void __launch_bounds__(256) mlp_infer_k(int64_t n, const float *__restrict__ x, float *__restrict__ y,
                                                   const float *__restrict__ w, const uint16_t *__restrict__ wbg,
                                                   Norm nm) {
  __shared__ __attribute__((aligned(16))) uint16_t wb[2 * HID * kRow];
  __shared__ FwdLds lds[4];
  __shared__ SmallW sw;
  load_weights<2 * HID>(w, wbg, sw, wb);
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int64_t nchunk = (n + 63) / 64;
  for (int64_t ch = (int64_t)blockIdx.x * 4 + wv; ch < (nchunk + 3) / 4 * 4; ch += (int64_t)gridDim.x * 4) {
    for (int t = 0; t < 4; ++t) {
      const int64_t base = ch * 64 + t * 16;
      if (l < 48) {
        const int mm = l / 3, j = l % 3;
        const int64_t s = base + mm;
        lds[wv].x[mm * 3 + j] = s < n ? (x[s * 3 + j] - nm.xm[j]) / nm.xs[j] : 0.f;
      }
      __builtin_amdgcn_s_waitcnt(0);
      __builtin_amdgcn_wave_barrier();
      mlp_fwd16(sw, wb, lds[wv]);
      if (l < 48) {
        const int mm = l / 3, j = l % 3;
        const int64_t s = base + mm;
        if (s < n) y[s * 3 + j] = lds[wv].y[mm * 3 + j] * nm.ys[j] + nm.ym[j];
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ---------------- training ----------------

struct TrainLds {
  uint16_t wb[4 * HID * kRow];                           // W2, W3, W2T, W3T
  uint16_t h1[32 * kRow], h2[32 * kRow], h3[32 * kRow];  // [m][k]
  uint16_t dz[32 * kRow];                                // [m][k] of the current layer
  uint16_t hT[HID * kRowT];                              // [k][m] of the layer input
  uint16_t dzT[HID * kRowT];                             // [n][m]
  float dzf[32 * HID];                                   // dz of layer 3 before rounding
  float x[32 * 3], y[32 * 3];                            // normalised inputs and targets
  float err[32 * 3], dy[32 * 3];                         // error of each output, its share of the gradient
};

// Sample i of a training run: splitmix64 of (seed, i) modulo n.
__device__ __forceinline__ int64_t sample_index(uint64_t seed, uint64_t i, uint64_t n) {
  uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return (int64_t)((z ^ (z >> 31)) % n);
}

// 32 samples of the batch per block: idx[32 b .. 32 b + 32), or with idx null
// samples first + 32 b .. of the run (sample_index over n).  Writes this
// block's share of the gradient of sum_m sum_j (y - t)^2 / (3 B) to
// part[blockIdx.x] (each weight-gradient tile as soon as it is formed).
//
// A batch of 8192 is 256 blocks, one per CU, so the time is that of one
// block's chain of layers: eight waves share it.  In the forward pass a wave
// takes a tile of 16 samples and 16 neurons (4 of the 64 tanh a lane would take
// alone), in the backward pass four waves form the weight gradients, the other
// four the sums over the samples beside them, and all eight the errors of the
// layer below.  Weights, inputs and targets are asked for together at the
// start.  Each sum keeps its terms and their order, so the gradient is that of
// one wave, bit for bit (44 us with one wave per block, 20 with four and the
// targets fetched where they are used; 13 us).
constexpr int kTrainThreads = 512;
__global__ void __launch_bounds__(kTrainThreads) mlp_train_k(int64_t B, const int64_t *__restrict__ idx, uint64_t seed,
                                                   uint64_t first, uint64_t n, const float *__restrict__ X,
                                                   const float *__restrict__ Y, const float *__restrict__ w,
                                                   const uint16_t *__restrict__ wbg, Norm nm,
                                                   float *__restrict__ part, float *__restrict__ loss_part) {
  __shared__ __attribute__((aligned(16))) TrainLds L;
  __shared__ SmallW sw;
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, m16 = l & 15, q = l >> 4;
  const int t = wv & 1, nt = wv >> 1;  // tile of 16 samples, tile of 16 neurons
  float *g = part + (int64_t)blockIdx.x * kParams;
  const int64_t s0 = (int64_t)blockIdx.x * 32;
  const int ns = (int)(s0 + 32 < B ? 32 : B - s0);
  const float inv = 2.0f / (3.0f * (float)B);
  // weights, and normalised by waves 6 and 7 the targets, by the others the
  // inputs (each pair of waves the same ones: no branch); padding samples get
  // x = 0 and, below, dy = 0
  {
    const int e = (threadIdx.x & 127) < 96 ? threadIdx.x & 127 : 95, mm = e / 3, j = e % 3;
    const bool in = wv < 6;
    int64_t k = s0 + (mm < ns ? mm : ns - 1);
    k = idx ? idx[k] : sample_index(seed, first + k, n);
    WeightCopy<4 * HID, kTrainThreads> wc;
    wc.load(w, wbg);
    const float raw = (in ? X : Y)[k * 3 + j];
    const float v = fk::quot(raw - (in ? nm.xm[j] : nm.ym[j]), in ? nm.xs[j] : nm.ys[j]);
    wc.store(sw, L.wb);
    (in ? L.x : L.y)[e] = mm < ns ? v : 0.f;
  }
  __syncthreads();
  // layer 1 (FP32): neurons k = 16 nt + 4 q + i of sample 16 t + m16
  {
    const int m = 16 * t + m16;
    const float x0 = L.x[m * 3 + 0], x1 = L.x[m * 3 + 1], x2 = L.x[m * 3 + 2];
    u16x4 hv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 c = sw.w1b[16 * nt + 4 * q + i];
      hv[i] = f2bf(tanhf(c.w + c.x * x0 + c.y * x1 + c.z * x2));
    }
    *reinterpret_cast<u16x4 *>(L.h1 + m * kRow + 16 * nt + 4 * q) = hv;
  }
  __syncthreads();
  // layers 2 and 3 (BF16 MFMA)
  const int nn = 16 * nt + m16;
#pragma unroll
  for (int layer = 0; layer < 2; ++layer) {
    const uint16_t *hin = layer == 0 ? L.h1 : L.h2, *W = L.wb + (layer == 0 ? 0 : HID * kRow);
    uint16_t *hout = layer == 0 ? L.h2 : L.h3;
    const float bias = (layer == 0 ? sw.b2 : sw.b3)[nn];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld_bf8(hin + (16 * t + m16) * kRow + 32 * ks + 8 * q),
                                                    ld_bf8(W + nn * kRow + 32 * ks + 8 * q), acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) hout[(16 * t + 4 * q + i) * kRow + nn] = f2bf(tanhf(acc[i] + bias));
    __syncthreads();
  }
  // layer 4 (FP32), waves 0 and 1: 16 neurons a lane, then the sample's four
  // lanes; the error of each output
  if (nt == 0) {
    const int m = 16 * t + m16;
    float p[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const u16x8 ab = *reinterpret_cast<const u16x8 *>(L.h3 + m * kRow + 32 * ks + 8 * q);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float h = bf2f(ab[i]);
        const int k = 32 * ks + 8 * q + i;
#pragma unroll
        for (int j = 0; j < 3; ++j) p[j] += sw.w4[j * HID + k] * h;
      }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      p[j] += __shfl_xor(p[j], 16, 64);
      p[j] += __shfl_xor(p[j], 32, 64);
    }
    if (q < 3) {
      const float pj = q == 0 ? p[0] : (q == 1 ? p[1] : p[2]);
      const float d = m < ns ? (sw.b4[q] + pj) - L.y[m * 3 + q] : 0.f;
      L.err[m * 3 + q] = d;
      L.dy[m * 3 + q] = d * inv;
    }
  }
  __syncthreads();
  // layer 4 backward: dz3[m][k] = (sum_j dy W4[j][k]) (1 - h3^2), lane k = l,
  // 4 samples a wave
  {
    const int k = l;
    const float w4[3] = {sw.w4[k], sw.w4[HID + k], sw.w4[2 * HID + k]};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int mm = 4 * wv + u;
      const float h = bf2f(L.h3[mm * kRow + k]);
      float dh = 0;
#pragma unroll
      for (int j = 0; j < 3; ++j) dh += L.dy[mm * 3 + j] * w4[j];
      const float dz = dh * (1.f - h * h);
      const uint16_t db = f2bf(dz);
      L.dzf[mm * HID + k] = dz;
      L.dz[mm * kRow + k] = db;
      L.dzT[k * kRowT + mm] = db;
      L.hT[k * kRowT + mm] = L.h2[mm * kRow + k];
    }
  }
  __syncthreads();
  // layers 3 then 2.  Waves 4 to 7: gW = dz^T h (K = 32 samples), 16 rows each.
  // Waves 0 to 3, lane k = l: sums over the samples, at layer 3 gb3 and gb4
  // (wave 0) and gW4[j][k], at layer 2 gb2 (wave 0).  Then all: dh = dz W, a
  // tile each; dz_below = dh (1 - h^2)
#pragma unroll
  for (int layer = 3; layer >= 2; --layer) {
    if (wv >= 4) {
      const int oW = layer == 3 ? oW3 : oW2, r = 16 * (wv - 4);
      const bf16x8 a = ld_bf8(L.dzT + (r + m16) * kRowT + 8 * q);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const bf16x8 b = ld_bf8(L.hT + (16 * c + m16) * kRowT + 8 * q);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) g[oW + (r + 4 * q + i) * HID + 16 * c + m16] = acc[i];
      }
    } else if (layer == 3 && wv == 0) {
      float gb3 = 0;
#pragma unroll 8
      for (int mm = 0; mm < 32; ++mm) gb3 += L.dzf[mm * HID + l];
      g[oB3 + l] = gb3;
      if (l < 3) {
        float sb = 0;
#pragma unroll 8
        for (int mm = 0; mm < 32; ++mm) sb += L.dy[mm * 3 + l];
        g[oB4 + l] = sb;
      }
    } else if (layer == 3) {
      const int j = wv - 1;
      float gw4 = 0;
#pragma unroll 8
      for (int mm = 0; mm < 32; ++mm) gw4 += L.dy[mm * 3 + j] * bf2f(L.h3[mm * kRow + l]);
      g[oW4 + j * HID + l] = gw4;
    } else if (wv == 0) {
      float sb = 0;
#pragma unroll 8
      for (int mm = 0; mm < 32; ++mm) sb += bf2f(L.dz[mm * kRow + l]);
      g[oB2 + l] = sb;
    }
    const uint16_t *WT = L.wb + (layer == 3 ? 3 : 2) * HID * kRow;
    const uint16_t *hin = layer == 3 ? L.h2 : L.h1;  // activations feeding this layer
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld_bf8(L.dz + (16 * t + m16) * kRow + 32 * ks + 8 * q),
                                                  ld_bf8(WT + nn * kRow + 32 * ks + 8 * q), d, 0, 0, 0);
    uint16_t db[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float h = bf2f(hin[(16 * t + 4 * q + i) * kRow + nn]);
      db[i] = f2bf(d[i] * (1.f - h * h));
    }
    __syncthreads();  // every wave has read dz, dzT and hT
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * t + 4 * q + i;
      L.dz[row * kRow + nn] = db[i];
      L.dzT[nn * kRowT + row] = db[i];
    }
    if (layer == 3)
#pragma unroll
      for (int u = 0; u < 4; ++u) L.hT[l * kRowT + 4 * wv + u] = L.h1[(4 * wv + u) * kRow + l];
    __syncthreads();
  }
  // gb1 (wave 0), gW1 (waves 1 to 3), the loss (wave 4: outputs l < 48 of tile
  // 0, then of tile 1)
  if (wv == 0) {
    float sb = 0;
#pragma unroll 8
    for (int mm = 0; mm < 32; ++mm) sb += bf2f(L.dz[mm * kRow + l]);
    g[oB1 + l] = sb;
  } else if (wv < 4) {
    const int j = wv - 1;
    float gw1 = 0;
#pragma unroll 8
    for (int mm = 0; mm < 32; ++mm) gw1 += bf2f(L.dz[mm * kRow + l]) * L.x[mm * 3 + j];
    g[oW1 + 3 * l + j] = gw1;
  } else if (wv == 4) {
    float lsum = 0;
    if (l < 48)
      for (int tt = 0; tt < 2; ++tt) {
        const float d = L.err[tt * 48 + l];
        lsum += d * d;
      }
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_down(lsum, off, 64);
    if (l == 0) loss_part[blockIdx.x] = lsum;
  }
}

// BF16 copies of parameter i (W2, W3 and their transposes).
__device__ __forceinline__ void pack_param(int i, float v, uint16_t *__restrict__ wb) {
  const bool w3 = i >= oW3 && i < oB3;
  if (!w3 && !(i >= oW2 && i < oB2)) return;
  const int k = i - (w3 ? oW3 : oW2), r = k / HID, c = k % HID;
  const uint16_t b = f2bf(v);
  wb[(w3 ? bW3 : bW2) + k] = b;
  wb[(w3 ? bW3T : bW2T) + c * HID + r] = b;
}

// Fixed-order sum of the per-block partials (deterministic), and with ADAM the
// update of the FP32 master weights and their BF16 copies.  A block takes 64
// parameters; the kernel waits for memory, not for its 138 blocks, so four
// waves hold 64 partials each in flight (a wave counts no more than 63 loads),
// add them one wave after the other, and the moments and weights are there by
// then (58 us for 256 partials with one load at a time and 256 threads a
// block, and 9 us for the update and the copies as kernels of their own; 8 us
// in one wave with 32 ahead; 4 us).
template <bool ADAM>
__global__ void __launch_bounds__(256) mlp_update_k(int nb, const float *__restrict__ part, float *__restrict__ g,
                                                    float *__restrict__ w, float *__restrict__ m,
                                                    float *__restrict__ v, uint16_t *__restrict__ wb, float lr,
                                                    float b1t, float b2t) {
  __shared__ float sum[64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int it = blockIdx.x * 64 + l, i = it < kParams ? it : kParams - 1;
  float m0 = 0, v0 = 0, w0 = 0;
  if constexpr (ADAM) {
    m0 = m[i];
    v0 = v[i];
    w0 = w[i];
  }
  float s = 0;
  for (int b0 = 0; b0 < nb; b0 += 256) {
    const int b = b0 + 64 * wv, n = nb - b;
    const float *p0 = part + (int64_t)b * kParams + i;
    float p[64];
    if (n >= 64) {
#pragma unroll
      for (int k = 0; k < 64; ++k) p[k] = p0[(int64_t)k * kParams];
    } else {
#pragma unroll
      for (int k = 0; k < 64; ++k) {
        const float x = part[(int64_t)(b + k < nb ? b + k : nb - 1) * kParams + i];
        p[k] = k < n ? x : 0.f;
      }
    }
#pragma unroll 1
    for (int o = 0; o < 4; ++o) {
      if (wv == o) {
        if (b > 0) s = sum[l];
#pragma unroll
        for (int k = 0; k < 64; ++k) s += p[k];
        sum[l] = s;
      }
      __syncthreads();
    }
  }
  if (wv != 3 || it != i) return;
  s = sum[l];
  if constexpr (!ADAM) {
    g[i] = s;
  } else {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mi = b1 * m0 + (1 - b1) * s;
    const float vi = b2 * v0 + (1 - b2) * s * s;
    m[i] = mi;
    v[i] = vi;
    const float wi = w0 - lr * (mi / (1 - b1t)) / (sqrtf(vi / (1 - b2t)) + eps);
    w[i] = wi;
    pack_param(i, wi, wb);
  }
}

__global__ void __launch_bounds__(256) mlp_pack_k(const float *__restrict__ w, uint16_t *__restrict__ wb) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < kParams) pack_param(i, w[i], wb);
}

// Training target of a state: the chemical (p-T-g) equilibrium of its
// mixture density and internal energy, (T, asinh(p / 1e4), alpha_L), by the
// (ln p, T) Newton from the liquid's (T, p) to 1e-10 (fk::chem_polish), or NaN
// where that solve finds no two-phase equilibrium.  The equilibrium depends
// on (rho, e) alone, so the labels of every state, whatever its class, are
// values of the one map the network learns.  u is not modified.
__device__ inline void chem_label(const fk_params &P, const double *u, float *y) {
  double uc[10];
  for (int v = 0; v < 10; ++v) uc[v] = u[v];
  double T0, p0;
  fk::chem_cold(P, uc, T0, p0);
  if (fk::chem_polish(P, uc, T0, p0, P.polishTol, 30) > 0 && fk::mlp_targets(P, uc, y)) return;
  for (int j = 0; j < 3; ++j) y[j] = NAN;
}

// Labels host-provided states: features of U, and for the chemical-class
// states (those the relaxation hands to the network) the equilibrium target.
__global__ void __launch_bounds__(256) mlp_label_k(fk_params P, int64_t n, const double *__restrict__ U,
                                                   float *__restrict__ x, float *__restrict__ y) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  double u[10];
  for (int v = 0; v < 10; ++v) u[v] = U[c * 10 + v];
  fk::mlp_features(P, u, x + c * 3);
  int ts = 0;
  int chem = 0;
  if (P.chemFlag == 1) {
    const double avf = fk::clampd(P, u[0]);
    const double rho = u[1] / avf, enr = u[6] / (avf * rho);
    const double tL = fk::eos_T(P, 0, rho, enr), pL = fk::eos_p(P, 0, rho, enr);
    chem = tL > fk::tsat_dev(P, pL, tL, P.satTempUrf, &ts) && avf > P.chemLimit;
  }
  if (chem) chem_label(P, u, y + c * 3);
  else  // the network serves chemical cells only
    for (int j = 0; j < 3; ++j) y[c * 3 + j] = NAN;
}

// Surrogate relaxation, stage 1 (every cell, one thread each): exact
// classification by the sign of f(T_L; p_L); thermal cells try at most
// kColdIters analytic-Jacobian Newton iterations from the cell's own state
// (one hydro step away from the previous equilibrium, so most converge in 2-3)
// and are written back when converged (fk::screen_cell).  Chemical cells and
// thermal cells that did not converge go to the work list as
// (cell << 1) | chem for stage 2.  The last RK stage's fused pass F runs the
// same stage 1 on the state it produces (fk_kernels.hip).
// counts: [n_chem, newton iterations, -, fallbacks, warm-started, list
// lengths (chemical from the front in the low half, thermal from the back in
// the high half), -, fallback list length].

__global__ void __launch_bounds__(256) relax_screen_k(fk_params P, int64_t nc, double *__restrict__ U,
                                                      uint32_t *__restrict__ list,
                                                      unsigned long long *__restrict__ counts,
                                                      unsigned long long *__restrict__ part, float *__restrict__ W) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int chem = 0, it = 0, push = 0;
  if (c < nc) {
    double u[10];
    fk::load_rec<10>(U + c * 10, u);
    push = fk::screen_cell(P, u, &chem, &it);
    if (!push) {
      U[c * 10 + 0] = u[0];
      U[c * 10 + 6] = u[6];
      U[c * 10 + 7] = u[7];
    }
    // primitive records of pass G for the cells solved here (list cells:
    // relax_list_k)
    if (W && !push) fk::store_prims<10>(fk::make_mat<double>(P), u, W + c * 10);
  }
  fk::list_push_block(push != 0, chem != 0, (uint32_t)((c << 1) | chem), list, nc, counts);
  unsigned long long v[2] = {(unsigned long long)chem, (unsigned long long)it};
  fk::block_partials<2>(v, part);  // [n_chem, newton iterations]
}

// Surrogate relaxation, stage 2a (FK_RELAX_MLP): the network's equilibrium
// (T*, p*) of each chemical entry of the work list (its front),
// by wave-cooperative inference, 64 entries per wave, into start[e].  Apart
// from the polish (stage 2b) so that the registers of neither limit the
// occupancy of the other.
__global__ void __launch_bounds__(256) relax_infer_k(fk_params P, const double *__restrict__ U,
                                                     const uint32_t *__restrict__ list, const float *__restrict__ w,
                                                     const uint16_t *__restrict__ wbg, Norm nm,
                                                     const unsigned long long *__restrict__ counts,
                                                     float2 *__restrict__ start) {
  __shared__ __attribute__((aligned(16))) uint16_t wb[2 * HID * kRow];
  __shared__ FwdLds lds[4];
  __shared__ SmallW sw;
  const int64_t nfr = fk::list_front(counts[5]);
  const int64_t cf = (nfr + 63) / 64;
  if ((int64_t)blockIdx.x * 4 >= cf) return;  // whole block idle: skip the weight load
  load_weights<2 * HID>(w, wbg, sw, wb);
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int64_t per = (cf + 3) / 4 * 4;
  for (int64_t ch = (int64_t)blockIdx.x * 4 + wv; ch < per; ch += (int64_t)gridDim.x * 4) {
    const int64_t e = ch * 64 + l;
    const bool live = e < nfr;
    const int64_t c = live ? (int64_t)(list[e] >> 1) : 0;
    double u[10];
    for (int v = 0; v < 10; ++v) u[v] = live ? U[c * 10 + v] : (v == 1 || v == 2 ? 1.0 : 0.0);
    float xf[3];
    fk::mlp_features(P, u, xf);
    float yw[3];
    for (int t = 0; t < 4; ++t) {  // wave-uniform: every lane joins
      if ((l >> 4) == t)
        for (int j = 0; j < 3; ++j) lds[wv].x[(l & 15) * 3 + j] = (xf[j] - nm.xm[j]) / nm.xs[j];
      __builtin_amdgcn_s_waitcnt(0);
      __builtin_amdgcn_wave_barrier();
      mlp_fwd16(sw, wb, lds[wv]);
      if ((l >> 4) == t)
        for (int j = 0; j < 3; ++j) yw[j] = lds[wv].y[(l & 15) * 3 + j] * nm.ys[j] + nm.ym[j];
      __builtin_amdgcn_wave_barrier();
    }
    // (T*, p*); the alpha_L* output is not needed: the polish takes alpha_L
    // from the mass balance at (p, T)
    if (live) start[e] = make_float2(yw[0], (float)((double)kPScale * sinh((double)yw[1])));
  }
}

// Surrogate relaxation, stage 2b (the work list, 64 entries per wave): FP64
// Newton polish from the network's start (WARM, chemical entries) or from the
// cell state (thermal entries, and FK_RELAX_COLD); a cell whose polish fails
// goes to the fallback list.
template <bool WARM>
__global__ void __launch_bounds__(256) relax_list_k(fk_params P, double *__restrict__ U,
                                                    const uint32_t *__restrict__ list,
                                                    const float2 *__restrict__ start,
                                                    unsigned long long *__restrict__ counts, float *__restrict__ W,
                                                    int64_t cap, uint32_t *__restrict__ fall) {
  // chunks of 64 entries: the chemical ones from the list's front, then the
  // thermal ones from its back
  // (short lists 4 lanes to an entry, fk::chem_polish4)
  const int64_t nfr = fk::list_front(counts[5]), nbk = fk::list_back(counts[5]);
  const int per = polish_lanes(nfr, (int64_t)gridDim.x * 256), epw = 64 / per;
  const int64_t cf = (nfr + epw - 1) / epw, nchunk = cf + (nbk + 63) / 64;
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  unsigned long long nit = 0, nwarm = 0;
  for (int64_t ch = (int64_t)blockIdx.x * 4 + wv; ch < nchunk; ch += (int64_t)gridDim.x * 4) {
    const bool front = ch < cf;  // wave-uniform
    const int64_t e = front ? ch * epw + l / per : (ch - cf) * 64 + l;
    const bool live = e < (front ? nfr : nbk);
    const bool lead = !front || per == 1 || (l & 3) == 0;
    const uint32_t ent = live ? list[front ? e : cap - 1 - e] : 0u;
    const int64_t c = (int64_t)(ent >> 1);
    const int chem = (int)(ent & 1u);
    double u[10];
    for (int v = 0; v < 10; ++v) u[v] = live ? U[c * 10 + v] : 0.0;
    double T0 = 0, p0 = 0;  // chemical cells: start (T, p)
    if (WARM && front && live) {
      const float2 y = start[e];
      T0 = (double)y.x;
      p0 = (double)y.y;
    }
    if (!live) continue;
    if (chem && !WARM) fk::chem_cold(P, u, T0, p0);
    nwarm += (WARM && chem && lead) ? 1 : 0;
    int it;
    if (chem) {
      it = per == 4 ? fk::chem_polish4(P, u, T0, p0, P.polishTol, 30) : fk::chem_polish(P, u, T0, p0, P.polishTol, 30);
    } else {  // thermal cells: the cell state
      fk::ThermProb t;
      fk::therm_setup(P, u, t);
      double rk, ek;
      fk::therm_cold(P, u, t, rk, ek);
      it = fk::therm_polish(P, u, rk, ek, P.polishTol, 30);
    }
    if (!lead) continue;
    // a failed polish leaves U as it was: the cell goes to the fallback list
    // (relax_fallback_k runs the reference solve from the cell state)
    const bool failed = it < 0;
    const unsigned long long mf = __ballot(failed);
    if (mf) {
      const int leader = __ffsll((long long)mf) - 1;
      unsigned long long b = 0;
      if (l == leader) b = atomicAdd(&counts[7], (unsigned long long)__popcll(mf));
      b = __shfl(b, leader, 64);
      if (failed) fall[b + __popcll(mf & ((1ull << l) - 1ull))] = ent;
    }
    if (failed) continue;
    nit += it;
    U[c * 10 + 0] = u[0];
    U[c * 10 + 1] = u[1];
    U[c * 10 + 2] = u[2];
    U[c * 10 + 6] = u[6];
    U[c * 10 + 7] = u[7];
    U[c * 10 + 9] = u[9];
    if (W) fk::store_prims<10>(fk::make_mat<double>(P), u, W + c * 10);
  }
  fk::block_add(nit, &counts[1]);
  fk::block_add(nwarm, &counts[4]);
}

// Fallback of the surrogate relaxation: the reference solve (thermRlx /
// chemRlx, as the plain relaxation) from the cell state for the cells whose
// polish failed (fall[0 .. counts[7]), entries (cell << 1) | chem).  Apart
// from relax_list_k so that the reference solves' registers do not limit the
// occupancy of the polish.  A fallback counts 30 iterations plus those of the
// reference solve.
__global__ void __launch_bounds__(256) relax_fallback_k(fk_params P, double *__restrict__ U,
                                                        const uint32_t *__restrict__ fall,
                                                        unsigned long long *__restrict__ counts,
                                                        float *__restrict__ W) {
  const int64_t n = (int64_t)counts[7];
  unsigned long long nit = 0, nfb = 0;
  // short lists 8 lanes per cell (fk::chem_dev8, thermal cells on each of them
  // alike)
  const int per = chem_lanes(n, (int64_t)gridDim.x * 256);
  const int64_t nt = (int64_t)gridDim.x * 256 / per;
  const bool lead = per == 1 || (threadIdx.x & 7) == 0;
  for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) / per; e < n; e += nt) {
    const uint32_t ent = fall[e];
    const int64_t c = (int64_t)(ent >> 1);
    double u[10];
    for (int v = 0; v < 10; ++v) u[v] = U[c * 10 + v];
    int it;
    if (ent & 1u) it = per == 8 ? fk::chem_dev8(P, u) : fk::chem_dev(P, u);
    else it = fk::therm_dev(P, u);
    if (!lead) continue;
    nit += 30 + (unsigned long long)it;
    ++nfb;
    for (int v = 0; v < 10; ++v) U[c * 10 + v] = u[v];
    if (W) fk::store_prims<10>(fk::make_mat<double>(P), u, W + c * 10);
  }
  const int l = threadIdx.x & 63;
  for (int off = 32; off > 0; off >>= 1) {
    nit += __shfl_down(nit, off, 64);
    nfb += __shfl_down(nfb, off, 64);
  }
  if (l == 0 && nfb) {
    atomicAdd(&counts[1], nit);
    atomicAdd(&counts[3], nfb);
  }
}

// Emission of solver states: plain relaxation that also writes (features,
// equilibrium target) of the pre-relaxation states of cells c = phase +
// k stride, whatever their class, into slot k of the training set.
__global__ void __launch_bounds__(256) relax_emit_k(fk_params P, int64_t nc, double *__restrict__ U, int64_t stride,
                                                    int64_t phase, float *__restrict__ dx, float *__restrict__ dy,
                                                    int64_t cap) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= nc) return;
  double u[10];
  for (int v = 0; v < 10; ++v) u[v] = U[c * 10 + v];
  const bool emit = stride > 0 && (c % stride) == phase;
  float xf[3], yl[3];
  if (emit) {
    fk::mlp_features(P, u, xf);
    chem_label(P, u, yl);  // from the pre-relaxation state, whatever the cell's class
  }
  int chem = 0, ts = 0;
  if (P.chemFlag == 1) {
    const double avf = fk::clampd(P, u[0]);
    const double rho = u[1] / avf, enr = u[6] / (avf * rho);
    const double tL = fk::eos_T(P, 0, rho, enr), pL = fk::eos_p(P, 0, rho, enr);
    chem = tL > fk::tsat_dev(P, pL, tL, P.satTempUrf, &ts) && avf > P.chemLimit;
  }
  if (chem) fk::chem_dev(P, u);
  else fk::therm_dev(P, u);
  for (int v = 0; v < 10; ++v) U[c * 10 + v] = u[v];
  if (emit) {
    const int64_t slot = (c - phase) / stride;
    if (slot < cap) {
      for (int j = 0; j < 3; ++j) {
        dx[slot * 3 + j] = xf[j];
        dy[slot * 3 + j] = yl[j];
      }
    }
  }
}

// ---------------- host side ----------------

Norm norm_of(const Mlp &m) {
  Norm n;
  for (int j = 0; j < 3; ++j) {
    n.xm[j] = m.norm[j];
    n.xs[j] = m.norm[3 + j];
    n.ym[j] = m.norm[6 + j];
    n.ys[j] = m.norm[9 + j];
  }
  return n;
}

int ensure_mlp(fk_ctx *c) {
  Mlp &m = c->mlp;
  if (m.w) return FK_OK;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipMalloc(&m.w, kParams * 4));
  HIPCHK(hipMalloc(&m.m, kParams * 4));
  HIPCHK(hipMalloc(&m.v, kParams * 4));
  HIPCHK(hipMalloc(&m.grad, kParams * 4));
  HIPCHK(hipMalloc(&m.wb, kBf * 2));
  HIPCHK(hipMemset(m.w, 0, kParams * 4));
  HIPCHK(hipMemset(m.m, 0, kParams * 4));
  HIPCHK(hipMemset(m.v, 0, kParams * 4));
  HIPCHK(hipMemset(m.wb, 0, kBf * 2));
  return FK_OK;
}

int pack(fk_ctx *c) {
  hipLaunchKernelGGL(mlp_pack_k, dim3((kParams + 255) / 256), dim3(256), 0, c->stream, c->mlp.w, c->mlp.wb);
  HIPCHK(hipGetLastError());
  return FK_OK;
}

// Device scratch of one label or inference call (m.work), its parts on 16-byte
// words as the copies take them; work_done gives a large one back.
size_t pad16(size_t bytes) { return (bytes + 15) / 16 * 16; }
int work_take(fk_ctx *c, size_t bytes) {
  Mlp &m = c->mlp;
  if (bytes <= m.work_cap) return FK_OK;
  if (m.work) (void)hipFree(m.work);
  m.work = nullptr;
  m.work_cap = 0;
  HIPCHK(hipMalloc(&m.work, bytes));
  m.work_cap = bytes;
  return FK_OK;
}
void work_done(fk_ctx *c) {
  Mlp &m = c->mlp;
  if (m.work_cap <= kWorkKeep) return;
  (void)hipFree(m.work);
  m.work = nullptr;
  m.work_cap = 0;
}

int ensure_data(fk_ctx *c, int64_t cap) {
  Mlp &m = c->mlp;
  if (cap <= m.cap_data) return FK_OK;
  float *nx = nullptr, *ny = nullptr;
  HIPCHK(hipMalloc(&nx, (size_t)cap * 12));
  HIPCHK(hipMalloc(&ny, (size_t)cap * 12));
  if (m.n_data) {
    HIPCHK(hipMemcpyAsync(nx, m.dx, (size_t)m.n_data * 12, hipMemcpyDeviceToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(ny, m.dy, (size_t)m.n_data * 12, hipMemcpyDeviceToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
  }
  if (m.dx) (void)hipFree(m.dx);
  if (m.dy) (void)hipFree(m.dy);
  m.dx = nx;
  m.dy = ny;
  m.cap_data = cap;
  return FK_OK;
}

}  // namespace

// called from the relaxation entry point of fk_kernels.hip; counts layout as
// relax_screen_k / relax_list_k (slots [0, 8) of c->lcount, zeroed here).
// Checks, scratch and zeroed counts of the surrogate relaxation (before stage
// 1, which relax_screen_k or the last stage's fused pass F runs).
int fk_relax_mlp_begin(fk_ctx *c, bool warm) {
  Mlp &m = c->mlp;
  if (warm && !m.ready) return fail(FK_ESTATE, "surrogate relaxation needs trained or loaded MLP weights");
  // the exact classification needs f(T) increasing: B <= 0 and C >= 0
  const fk_params &P = c->p;
  if (P.chemFlag == 1 && !((P.eta[0] - P.eta[1]) <= 0 && (P.Cp[1] - P.Cp[0]) >= 0))
    return fail(FK_EINVAL, "surrogate classification needs eta_L <= eta_G and Cp_G >= Cp_L");
  int rc = ensure_rlist(c);
  if (rc) return rc;
  return zero_counts(c);
}

int fk_relax_mlp_impl(fk_ctx *c, bool warm, bool reduce) {
  int rc = fk_relax_mlp_begin(c, warm);
  if (rc) return rc;
  unsigned long long *cnt = (unsigned long long *)c->lcount;
  const unsigned gs = (unsigned)((c->nc + 255) / 256);
  // mixed precision: the relaxation also writes the primitive records of pass G
  float *W = (c->p.precision == FK_MIXED && c->prims_w) ? c->wprim : nullptr;
  LAUNCH_TIMED(c, "relax_screen", hipLaunchKernelGGL(relax_screen_k, dim3(gs), dim3(256), 0, c->stream, c->p, c->nc,
                                                     c->U[c->ia], c->rlist, cnt, c->rpart, W));
  if (reduce)
    LAUNCH_TIMED(c, "relax_count", hipLaunchKernelGGL(fk::reduce_partials<2>, dim3(fk::reduce_grid(gs)), dim3(256), 0,
                                                      c->stream, c->rpart, (int64_t)gs, cnt));
  return fk_relax_mlp_finish(c, warm);
}

// Stage 2 (the work list) after stage 1.
int fk_relax_mlp_finish(fk_ctx *c, bool warm) {
  Mlp &m = c->mlp;
  unsigned long long *cnt = (unsigned long long *)c->lcount;
  float *W = (c->p.precision == FK_MIXED && c->prims_w) ? c->wprim : nullptr;
  const unsigned grid = list_blocks(c->nc, 1), glist = list_blocks(c->nc, 4);
  if (warm) {
    int rc = ensure_rstart(c);  // fk_run_steps has allocated it before its first stage
    if (rc) return rc;
    float2 *st = static_cast<float2 *>(c->rstart);
    LAUNCH_TIMED(c, "relax_infer", hipLaunchKernelGGL(relax_infer_k, dim3(grid), dim3(256), 0, c->stream, c->p,
                                                      c->U[c->ia], c->rlist, m.w, m.wb, norm_of(m), cnt, st));
    LAUNCH_TIMED(c, "relax_list", hipLaunchKernelGGL(relax_list_k<true>, dim3(glist), dim3(256), 0, c->stream, c->p,
                                                     c->U[c->ia], c->rlist, st, cnt, W, c->nc, c->rfall));
  } else {
    LAUNCH_TIMED(c, "relax_list", hipLaunchKernelGGL(relax_list_k<false>, dim3(glist), dim3(256), 0, c->stream, c->p,
                                                     c->U[c->ia], c->rlist, nullptr, cnt, W, c->nc, c->rfall));
  }
  const unsigned gfb = std::min(list_blocks(c->nc, 8), 512u);
  LAUNCH_TIMED(c, "relax_fallback", hipLaunchKernelGGL(relax_fallback_k, dim3(gfb), dim3(256), 0, c->stream, c->p,
                                                       c->U[c->ia], c->rfall, cnt, W));
  c->w_valid = W != nullptr;
  return FK_OK;
}

// plain relaxation with emission of training pairs (when enabled)
int fk_relax_emit_impl(fk_ctx *c, bool *done) {
  *done = false;
  Mlp &m = c->mlp;
  if (m.emit_stride <= 0) return FK_OK;
  const int64_t room = m.cap_data - m.n_data;
  if (room <= 0) return FK_OK;
  LAUNCH_TIMED(c, "relax_emit", hipLaunchKernelGGL(relax_emit_k, dim3((unsigned)((c->nc + 255) / 256)), dim3(256), 0,
                                                   c->stream, c->p, c->nc, c->U[c->ia], m.emit_stride, m.emit_phase,
                                                   m.dx + m.n_data * 3, m.dy + m.n_data * 3, room));
  const int64_t emitted = m.emit_phase < c->nc ? (c->nc - m.emit_phase + m.emit_stride - 1) / m.emit_stride : 0;
  m.n_data += std::min<int64_t>(emitted, room);
  m.emit_phase = (m.emit_phase + 1) % m.emit_stride;
  *done = true;
  return FK_OK;
}

void fk_mlp_free(fk_ctx *c) {
  Mlp &m = c->mlp;
  void *ptrs[] = {m.w, m.m, m.v, m.wb, m.grad, m.part, m.dx, m.dy, m.work};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  m = Mlp{};
}

extern "C" {

int fk_mlp_set_weights(fk_ctx *c, const float *w, const float *norm) {
  if (!c || !w || !norm) return fail(FK_EINVAL, "null argument");
  int rc = ensure_mlp(c);
  if (rc) return rc;
  HIPCHK(hipMemcpy(c->mlp.w, w, kParams * 4, hipMemcpyHostToDevice));
  std::memcpy(c->mlp.norm, norm, sizeof c->mlp.norm);
  for (int j = 0; j < 3; ++j)
    if (!(norm[3 + j] > 0) || !(norm[9 + j] > 0)) return fail(FK_EINVAL, "normalisation scales must be positive");
  rc = pack(c);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(c->stream));
  c->mlp.ready = true;
  c->mlp.adam_t = 0;
  HIPCHK(hipMemset(c->mlp.m, 0, kParams * 4));
  HIPCHK(hipMemset(c->mlp.v, 0, kParams * 4));
  return FK_OK;
}

int fk_mlp_get_weights(fk_ctx *c, float *w, float *norm) {
  if (!c || !w || !norm) return fail(FK_EINVAL, "null argument");
  if (!c->mlp.w) return fail(FK_ESTATE, "no MLP weights");
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(w, c->mlp.w, kParams * 4, hipMemcpyDeviceToHost));
  std::memcpy(norm, c->mlp.norm, sizeof c->mlp.norm);
  return FK_OK;
}

int fk_mlp_label(fk_ctx *c, const double *U, int64_t n, float *x, float *y) {
  if (!c || !U || !x || !y || n < 0) return fail(FK_EINVAL, "bad argument");
  if (c->p.model != FK_MODEL_TWO_PHASE) return fail(FK_EINVAL, "labels need the two-phase model");
  if (n == 0) return FK_OK;
  HIPCHK(hipSetDevice(c->device));
  const size_t nx = pad16((size_t)n * 12);
  int rc = work_take(c, (size_t)n * 80 + 2 * nx);
  if (rc) return rc;
  double *dU = reinterpret_cast<double *>(c->mlp.work);
  float *dx = reinterpret_cast<float *>(dU + n * 10), *dy = dx + nx / 4;
  rc = copy_up(c, dU, U, (size_t)n * 80);
  if (!rc) {
    hipLaunchKernelGGL(mlp_label_k, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, c->p, n, dU, dx, dy);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = fail(FK_EDEVICE, std::string("mlp_label: ") + hipGetErrorString(e));
  }
  if (!rc) rc = copy_down(c, x, dx, (size_t)n * 12);
  if (!rc) rc = copy_down(c, y, dy, (size_t)n * 12);
  work_done(c);
  return rc;
}

int fk_mlp_data(fk_ctx *c, const float *x, const float *y, int64_t n, int append) {
  if (!c || n < 0 || (n > 0 && (!x || !y))) return fail(FK_EINVAL, "bad argument");
  int rc = ensure_mlp(c);
  if (rc) return rc;
  Mlp &m = c->mlp;
  if (!append) m.n_data = 0;
  rc = ensure_data(c, m.n_data + n);
  if (rc) return rc;
  if (n) {
    HIPCHK(hipMemcpy(m.dx + m.n_data * 3, x, (size_t)n * 12, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(m.dy + m.n_data * 3, y, (size_t)n * 12, hipMemcpyHostToDevice));
  }
  m.n_data += n;
  return FK_OK;
}

int fk_mlp_emit(fk_ctx *c, int64_t stride, int64_t capacity) {
  if (!c || stride < 0 || capacity < 0) return fail(FK_EINVAL, "bad argument");
  int rc = ensure_mlp(c);
  if (rc) return rc;
  c->mlp.emit_stride = stride;
  c->mlp.emit_phase = 0;
  return ensure_data(c, c->mlp.n_data + capacity);
}

int fk_mlp_download_data(fk_ctx *c, float *x, float *y, int64_t max, int64_t *n) {
  if (!c || !n) return fail(FK_EINVAL, "bad argument");
  const int64_t k = std::min<int64_t>(max, c->mlp.n_data);
  *n = c->mlp.n_data;
  if (k > 0) {
    if (!x || !y) return fail(FK_EINVAL, "null buffers");
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(x, c->mlp.dx, (size_t)k * 12, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(y, c->mlp.dy, (size_t)k * 12, hipMemcpyDeviceToHost));
  }
  return FK_OK;
}

int fk_mlp_set_norm(fk_ctx *c, const float *norm) {
  if (!c || !norm) return fail(FK_EINVAL, "null argument");
  for (int j = 0; j < 3; ++j)
    if (!(norm[3 + j] > 0) || !(norm[9 + j] > 0)) return fail(FK_EINVAL, "normalisation scales must be positive");
  std::memcpy(c->mlp.norm, norm, sizeof c->mlp.norm);
  return FK_OK;
}

// Per-block gradients of the mean squared error (normalised outputs) over B
// samples of the device training set: didx[0, B), or with didx null samples
// first .. first + B of the run of `seed`.  Their sum is left to mlp_update_k.
static int grad_on(fk_ctx *c, const int64_t *didx, uint64_t seed, uint64_t first, int64_t B, int *nblocks) {
  Mlp &m = c->mlp;
  const int nb = (int)((B + 31) / 32);
  if (nb > m.part_cap) {
    if (m.part) (void)hipFree(m.part);
    m.part = nullptr;
    m.part_cap = 0;
    HIPCHK(hipMalloc(&m.part, (size_t)(nb + 1) * kParams * 4));
    m.part_cap = nb;
  }
  hipLaunchKernelGGL(mlp_train_k, dim3(nb), dim3(kTrainThreads), 0, c->stream, B, didx, seed, first, (uint64_t)m.n_data, m.dx,
                     m.dy, m.w, m.wb, norm_of(m), m.part, m.part + (size_t)nb * kParams);
  HIPCHK(hipGetLastError());
  *nblocks = nb;
  return FK_OK;
}

// Loss of the last grad_on.
static int read_loss(fk_ctx *c, int nb, int64_t B, float *loss) {
  std::vector<float> lp((size_t)nb);
  HIPCHK(hipMemcpyAsync(lp.data(), c->mlp.part + (size_t)nb * kParams, (size_t)nb * 4, hipMemcpyDeviceToHost,
                        c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  double s = 0;
  for (float v : lp) s += v;
  *loss = (float)(s / (3.0 * (double)B));
  return FK_OK;
}

int fk_mlp_grad(fk_ctx *c, const int64_t *idx, int64_t B, float *grad, float *loss) {
  if (!c || !idx || B <= 0 || !grad) return fail(FK_EINVAL, "bad argument");
  Mlp &m = c->mlp;
  if (!m.w || m.n_data <= 0) return fail(FK_ESTATE, "no weights or no training set");
  for (int64_t i = 0; i < B; ++i)
    if (idx[i] < 0 || idx[i] >= m.n_data) return fail(FK_EINVAL, "sample index out of range");
  int64_t *didx = nullptr;
  HIPCHK(hipMalloc(&didx, (size_t)B * 8));
  HIPCHK(hipMemcpy(didx, idx, (size_t)B * 8, hipMemcpyHostToDevice));
  int nb = 0;
  int rc = grad_on(c, didx, 0, 0, B, &nb);
  if (!rc) {
    hipLaunchKernelGGL(mlp_update_k<false>, dim3((kParams + 63) / 64), dim3(256), 0, c->stream, nb, m.part, m.grad,
                       nullptr, nullptr, nullptr, nullptr, 0.f, 0.f, 0.f);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = fail(FK_EDEVICE, std::string("mlp_update: ") + hipGetErrorString(e));
  }
  if (!rc && loss) rc = read_loss(c, nb, B, loss);
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(didx);
  if (rc) return rc;
  HIPCHK(hipMemcpy(grad, m.grad, kParams * 4, hipMemcpyDeviceToHost));
  return FK_OK;
}

int fk_mlp_train(fk_ctx *c, int steps, int batch, float lr, uint64_t seed, float *loss_first, float *loss_last) {
  if (!c || steps < 0 || batch <= 0) return fail(FK_EINVAL, "bad argument");
  Mlp &m = c->mlp;
  if (!m.w) return fail(FK_ESTATE, "set initial weights first (fk_mlp_set_weights)");
  if (m.n_data <= 0) return fail(FK_ESTATE, "empty training set");
  HIPCHK(hipSetDevice(c->device));
  // batch indices come from the step and the seed on the device: two kernels
  // a step, no copies, no waits (139 us a step of 8192 samples with indices
  // drawn and uploaded by the host; 19 us)
  int rc = FK_OK;
  for (int st = 0; st < steps && rc == FK_OK; ++st) {
    int nb = 0;
    if ((rc = grad_on(c, nullptr, seed, (uint64_t)st * (uint64_t)batch, batch, &nb))) break;
    if (st == 0 && loss_first && (rc = read_loss(c, nb, batch, loss_first))) break;
    if (st == steps - 1 && loss_last) {
      if (st == 0 && loss_first) *loss_last = *loss_first;
      else if ((rc = read_loss(c, nb, batch, loss_last))) break;
    }
    ++m.adam_t;
    const float b1t = std::pow(0.9f, (float)m.adam_t), b2t = std::pow(0.999f, (float)m.adam_t);
    hipLaunchKernelGGL(mlp_update_k<true>, dim3((kParams + 63) / 64), dim3(256), 0, c->stream, nb, m.part, nullptr, m.w,
                       m.m, m.v, m.wb, lr, b1t, b2t);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = fail(FK_EDEVICE, hipGetErrorString(e));
  }
  const hipError_t e = hipStreamSynchronize(c->stream);
  if (!rc && e != hipSuccess) rc = fail(FK_EDEVICE, hipGetErrorString(e));
  if (rc == FK_OK) m.ready = true;
  return rc;
}

int fk_mlp_infer(fk_ctx *c, const float *x, int64_t n, float *y) {
  if (!c || n < 0 || (n > 0 && (!x || !y))) return fail(FK_EINVAL, "bad argument");
  if (!c->mlp.w) return fail(FK_ESTATE, "no MLP weights");
  if (n == 0) return FK_OK;
  HIPCHK(hipSetDevice(c->device));
  const size_t nx = pad16((size_t)n * 12);
  int rc = work_take(c, 2 * nx);
  if (rc) return rc;
  float *dx = reinterpret_cast<float *>(c->mlp.work), *dy = dx + nx / 4;
  rc = copy_up(c, dx, x, (size_t)n * 12);
  if (!rc) {
    const int64_t nchunk = (n + 63) / 64;
    const unsigned grid = (unsigned)std::min<int64_t>((nchunk + 3) / 4, 4096);
    hipLaunchKernelGGL(mlp_infer_k, dim3(grid), dim3(256), 0, c->stream, n, dx, dy, c->mlp.w, c->mlp.wb,
                       norm_of(c->mlp));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = fail(FK_EDEVICE, std::string("mlp_infer: ") + hipGetErrorString(e));
  }
  if (!rc) rc = copy_down(c, y, dy, (size_t)n * 12);
  work_done(c);
  return rc;
}

}  // extern "C"
