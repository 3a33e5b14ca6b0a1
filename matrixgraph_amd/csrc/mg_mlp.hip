// Small MLP cost model: n_in -> 64 -> 64 -> n_out, ReLU hidden layers, linear outputs.
// Weights are used in BF16 (round-to-nearest-even from FP32 master copies), every product
// is accumulated in FP32. Training minimises the mean squared error with Adam on the
// device. Gradients are deterministic: each block writes the partial gradient of its
// samples, and a second kernel sums the partials in a fixed order (no float atomics).
//
// Parameter layout (FP32 master and BF16 copy): W1[64][n_in], b1[64], W2[64][64], b2[64],
// W3[n_out][64], b3[n_out].
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "mg_device.hpp"
#include "mg_internal.hpp"

namespace mgamd {
namespace {

constexpr int kH = 64;        // hidden width
constexpr int kMlpBlock = 64;  // one wave per block

// IEEE binary32 -> bfloat16, round to nearest even (NaN kept quiet).
__host__ __device__ inline uint16_t f32_to_bf16(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return static_cast<uint16_t>((u >> 16) | 0x40);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}
__host__ __device__ inline float bf16_to_f32(uint16_t h) {
  const uint32_t u = static_cast<uint32_t>(h) << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

struct Dims {
  uint32_t n_in, n_out;
  uint32_t o_w1, o_b1, o_w2, o_b2, o_w3, o_b3, n_params;
};

Dims make_dims(uint32_t n_in, uint32_t n_out) {
  Dims d{};
  d.n_in = n_in;
  d.n_out = n_out;
  d.o_w1 = 0;
  d.o_b1 = d.o_w1 + kH * n_in;
  d.o_w2 = d.o_b1 + kH;
  d.o_b2 = d.o_w2 + kH * kH;
  d.o_w3 = d.o_b2 + kH;
  d.o_b3 = d.o_w3 + n_out * kH;
  d.n_params = d.o_b3 + n_out;
  return d;
}

// The network on the matrix cores, in FP32 (v_mfma_f32_32x32x2_f32: FP32 operands and sums, as on
// the vector ALUs), one wave per tile of 32 samples. Every layer is computed transposed, units x
// samples: then lane l of a result holds sample l % 32, register v unit
//   unit_of(t, v, l) = 32t + 8 (v / 4) + 4 (l / 32) + v % 4        (t: half of the 64 units)
// and that same register is the B operand of the next layer's k-step over the units
// (unit_of(t, v, 0), unit_of(t, v, 32)) with no data moved between lanes; the weights (A operands)
// are loaded once per wave in that order. A wave that streamed samples with lane = unit needed a
// broadcast per multiply and 256 samples in series: 200 K rows forward took 104 us, the gradient of
// 4096 rows 370 us; now 36 (the matrix instructions alone 12) and 14. Relative error against 64
// bits, 100 to 40 K rows: outputs 1.36e-7 (1.60e-7 before), gradients 0.81e-7 (1.25e-7).
typedef float mg_v16f __attribute__((ext_vector_type(16)));
constexpr uint32_t kTileRows = 32;
// Workgroups at most: one wave per SIMD fits the registers; a workgroup takes every such tile.
constexpr uint32_t kForwardBlocks = 1024;
constexpr uint32_t kGradBlocks = 512;

__device__ inline uint32_t unit_of(int t, int v, uint32_t hi) { return 32 * t + 8 * (v / 4) + 4 * hi + v % 4; }

__device__ inline float wave_sum_f(float v) {
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

// A wave's weights as FP32 values of the BF16 ones.
template <int NI, int NO>
struct NetRegs {
  float w1[2][NI / 2];   // [t][s]: W1[32t + l % 32][2s + l / 32]
  float w2[2][32];       // [t][16 k + v]: W2[32t + l % 32][unit_of(k, v, l)]
  mg_v16f b1[2], b2[2];  // bias of unit_of(t, v, l)
  mg_v16f w3[NO][2];     // W3[o][unit_of(t, v, l)]
  float b3[NO];
};

template <int NI, int NO>
__device__ inline void load_net(const Dims& d, const uint16_t* __restrict__ w16, uint32_t lane, NetRegs<NI, NO>& R) {
  const uint32_t lo = lane & 31, hi = lane >> 5;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int s = 0; s < NI / 2; ++s) R.w1[t][s] = bf16_to_f32(w16[d.o_w1 + (32 * t + lo) * NI + 2 * s + hi]);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        R.w2[t][16 * k + v] = bf16_to_f32(w16[d.o_w2 + (32 * t + lo) * kH + unit_of(k, v, hi)]);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t u = unit_of(t, v, hi);
      R.b1[t][v] = bf16_to_f32(w16[d.o_b1 + u]);
      R.b2[t][v] = bf16_to_f32(w16[d.o_b2 + u]);
#pragma unroll
      for (int o = 0; o < NO; ++o) R.w3[o][t][v] = bf16_to_f32(w16[d.o_w3 + o * kH + u]);
    }
  }
#pragma unroll
  for (int o = 0; o < NO; ++o) R.b3[o] = bf16_to_f32(w16[d.o_b3 + o]);
}

__device__ inline void relu(mg_v16f& h) {
#pragma unroll
  for (int v = 0; v < 16; ++v) h[v] = h[v] > 0.f ? h[v] : 0.f;
}

__device__ inline float tree8(const float (&p)[8]) {
  return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
}

// Forward of one tile: this lane's sample (l % 32) has inputs xs[s] = x[2s + l / 32]; h1, h2 hold
// the lane's half of its units, y the outputs (the same in both halves).
template <int NI, int NO>
__device__ inline void forward_tile(const NetRegs<NI, NO>& R, const float (&xs)[NI / 2], mg_v16f (&h1)[2],
                                    mg_v16f (&h2)[2], float (&y)[NO]) {
  h1[0] = R.b1[0];
  h1[1] = R.b1[1];
#pragma unroll
  for (int s = 0; s < NI / 2; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t) h1[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(R.w1[t][s], xs[s], h1[t], 0, 0, 0);
  relu(h1[0]);
  relu(h1[1]);
  // Two sums of half the units each: shorter chains, in time and in rounding.
  mg_v16f part[2] = {R.b2[0], R.b2[1]};
#pragma unroll
  for (int v = 0; v < 16; ++v) h2[0][v] = h2[1][v] = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      part[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(R.w2[t][v], h1[0][v], part[t], 0, 0, 0);
      h2[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(R.w2[t][16 + v], h1[1][v], h2[t], 0, 0, 0);
    }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    h2[t] += part[t];
    relu(h2[t]);
  }
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    float p[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) p[c] = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) p[v % 8] += R.w3[o][t][v] * h2[t][v];
    const float half = tree8(p);
    y[o] = R.b3[o] + (half + __shfl_xor(half, 32, kWave));
  }
}

// Inputs of the lane's sample; rows past n read as zero.
template <int NI>
__device__ inline void load_inputs(const float* __restrict__ x, uint64_t row, bool valid, uint32_t hi,
                                   float (&xs)[NI / 2]) {
#pragma unroll
  for (int s = 0; s < NI / 2; ++s) xs[s] = valid ? x[row * NI + 2 * s + hi] : 0.f;
}

// y of every row; with t, no y but the wave's sum of squared errors in loss_part[block].
template <int NI, int NO>
__global__ void __launch_bounds__(kMlpBlock) mlp_forward_kernel(Dims d, const uint16_t* __restrict__ w16,
                                                                const float* __restrict__ x, uint32_t n,
                                                                float* __restrict__ y, const float* __restrict__ t,
                                                                float* __restrict__ loss_part) {
  const uint32_t lane = lane_id();
  const uint32_t lo = lane & 31, hi = lane >> 5;
  NetRegs<NI, NO> R;
  load_net<NI, NO>(d, w16, lane, R);
  const uint32_t n_tiles = n / kTileRows + (n % kTileRows != 0);
  float loss = 0.f;
  float xs[NI / 2];
  load_inputs<NI>(x, static_cast<uint64_t>(blockIdx.x) * kTileRows + lo, blockIdx.x * kTileRows + lo < n, hi, xs);
  for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const uint64_t row = static_cast<uint64_t>(tile) * kTileRows + lo;
    const uint64_t next = row + static_cast<uint64_t>(gridDim.x) * kTileRows;
    float xn[NI / 2];
    load_inputs<NI>(x, next, next < n, hi, xn);  // in flight during this tile
    mg_v16f h1[2], h2[2];
    float yo[NO];
    forward_tile<NI, NO>(R, xs, h1, h2, yo);
    if (row < n && hi == 0) {
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        if (t) {
          const float e = yo[o] - t[row * NO + o];
          loss += e * e;
        } else {
          y[row * NO + o] = yo[o];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < NI / 2; ++s) xs[s] = xn[s];
  }
  if (t) {
    loss = wave_sum_f(loss);
    if (lane == 0) loss_part[blockIdx.x] = loss;
  }
}

// Partial gradient of L = scale * sum over samples and outputs of (y - t)^2 over the block's tiles,
// accumulated in tile order; written to partial[block][param].
// Two waves per tile, wave q with the units 32q .. 32q + 31 of every layer: half the serial chain of
// matrix instructions (a mini-batch of 4096 is only 128 tiles, so a tile's latency is the kernel's
// time), and half the weights per wave (one wave alone spilled). The halves meet in LDS (rows of
// 33 words, which the weight gradients read along samples anyway): dW2 on the matrix cores, the
// small gradients with lane = unit, each wave half of the samples.
template <int NI, int NO>
__global__ void __launch_bounds__(2 * kWave) mlp_grad_kernel(Dims d, const uint16_t* __restrict__ w16,
                                                             const float* __restrict__ x, const float* __restrict__ t,
                                                             uint32_t n, float scale, float* __restrict__ partial,
                                                             float* __restrict__ loss_part) {
  constexpr uint32_t kRow = kTileRows + 1;
  constexpr int kSmall = NI + NO + 2;  // per unit: dW1 row, dW3 column, db1, db2
  __shared__ float s_h1[kH * kRow], s_h2[kH * kRow], s_d1[kH * kRow], s_d2[kH * kRow];
  __shared__ float s_x[kTileRows][NI];
  __shared__ float s_dy[kTileRows][NO];
  __shared__ float s_y[2][NO][kTileRows];
  __shared__ float s_small[kSmall][kH];
  const uint32_t lane = lane_id();
  const uint32_t q = read_first_lane(threadIdx.x / kWave);
  const uint32_t lo = lane & 31, hi = lane >> 5;
  const uint32_t unit = 32 * q + lo;  // A operand row of this wave's half
  float w1[NI / 2], w2[2][16], w2t[2][16];
  mg_v16f b1, b2, w3[NO];
#pragma unroll
  for (int s = 0; s < NI / 2; ++s) w1[s] = bf16_to_f32(w16[d.o_w1 + unit * NI + 2 * s + hi]);
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t u = unit_of(k, v, hi);
      w2[k][v] = bf16_to_f32(w16[d.o_w2 + unit * kH + u]);
      w2t[k][v] = bf16_to_f32(w16[d.o_w2 + u * kH + unit]);
    }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const uint32_t u = 32 * q + unit_of(0, v, hi);
    b1[v] = bf16_to_f32(w16[d.o_b1 + u]);
    b2[v] = bf16_to_f32(w16[d.o_b2 + u]);
#pragma unroll
    for (int o = 0; o < NO; ++o) w3[o][v] = bf16_to_f32(w16[d.o_w3 + o * kH + u]);
  }
  float b3[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) b3[o] = bf16_to_f32(w16[d.o_b3 + o]);
  mg_v16f g2[2];  // dW2 rows 32q + ..., columns 32 b + l % 32
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) g2[b][v] = 0.f;
  float g1[NI], g3[NO], gb1 = 0.f, gb2 = 0.f, gb3[NO], loss = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) g1[i] = 0.f;
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    g3[o] = 0.f;
    gb3[o] = 0.f;
  }
  const auto put = [&](float* buf, const mg_v16f& h) {
#pragma unroll
    for (int v = 0; v < 16; ++v) buf[(32 * q + unit_of(0, v, hi)) * kRow + lo] = h[v];
  };
  // The other wave's half, as B operands.
  const auto other = [&](const float* buf) {
    mg_v16f h;
#pragma unroll
    for (int v = 0; v < 16; ++v) h[v] = buf[(32 * (1 - q) + unit_of(0, v, hi)) * kRow + lo];
    return h;
  };
  // acc += (A rows of this wave) x (all 64 units); a[k] goes with the units 32k ... of `own` / `far`.
  const auto layer = [&](const float (&a)[2][16], const mg_v16f& own, const mg_v16f& far, mg_v16f acc) {
    const mg_v16f& k0 = q ? far : own;
    const mg_v16f& k1 = q ? own : far;
    mg_v16f part;
#pragma unroll
    for (int v = 0; v < 16; ++v) part[v] = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[0][v], k0[v], acc, 0, 0, 0);
      part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[1][v], k1[v], part, 0, 0, 0);
    }
    return acc + part;
  };
  const uint32_t n_tiles = n / kTileRows + (n % kTileRows != 0);
  for (uint32_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const uint64_t row = static_cast<uint64_t>(tile) * kTileRows + lo;
    const bool valid = row < n;
    float xs[NI / 2];
    load_inputs<NI>(x, row, valid, hi, xs);
    float target[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) target[o] = valid ? t[row * NO + o] : 0.f;
    mg_v16f h1 = b1;
#pragma unroll
    for (int s = 0; s < NI / 2; ++s) h1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w1[s], xs[s], h1, 0, 0, 0);
    relu(h1);
    __syncthreads();  // the previous tile's readers are done
    put(s_h1, h1);
    if (q == 0) {
#pragma unroll
      for (int s = 0; s < NI / 2; ++s) s_x[lo][2 * s + hi] = xs[s];
    }
    __syncthreads();
    mg_v16f h2 = layer(w2, h1, other(s_h1), b2);
    relu(h2);
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      float p[8];
#pragma unroll
      for (int v = 0; v < 16; ++v) p[v % 8] = v < 8 ? w3[o][v] * h2[v] : p[v % 8] + w3[o][v] * h2[v];
      const float half = tree8(p);
      const float whole = half + __shfl_xor(half, 32, kWave);
      if (hi == 0) s_y[q][o][lo] = whole;
    }
    put(s_h2, h2);
    __syncthreads();
    float dy[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const float y = b3[o] + (s_y[0][o][lo] + s_y[1][o][lo]);
      const float e = valid ? y - target[o] : 0.f;
      if (q == 0 && hi == 0) loss += e * e;
      dy[o] = 2.f * e * scale;
    }
    mg_v16f d2, d1;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float a = 0.f;
#pragma unroll
      for (int o = 0; o < NO; ++o) a += w3[o][v] * dy[o];
      d2[v] = h2[v] > 0.f ? a : 0.f;
      d1[v] = 0.f;
    }
    put(s_d2, d2);
    if (q == 0 && hi == 0) {
#pragma unroll
      for (int o = 0; o < NO; ++o) s_dy[lo][o] = dy[o];
    }
    __syncthreads();
    d1 = layer(w2t, d2, other(s_d2), d1);
#pragma unroll
    for (int v = 0; v < 16; ++v) d1[v] = h1[v] > 0.f ? d1[v] : 0.f;
    put(s_d1, d1);
#pragma unroll 4
    for (uint32_t k = 0; k < kTileRows / 2; ++k) {
      const uint32_t s = 2 * k + hi;
      const float a = s_d2[unit * kRow + s];
      g2[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s_h1[lo * kRow + s], g2[0], 0, 0, 0);
      g2[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s_h1[(32 + lo) * kRow + s], g2[1], 0, 0, 0);
    }
    __syncthreads();
#pragma unroll 4
    for (uint32_t k = 0; k < kTileRows / 2; ++k) {
      const uint32_t s = 16 * q + k;
      const float e1 = s_d1[lane * kRow + s], v2 = s_h2[lane * kRow + s];
      gb1 += e1;
      gb2 += s_d2[lane * kRow + s];
#pragma unroll
      for (int i = 0; i < NI; ++i) g1[i] += e1 * s_x[s][i];
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        g3[o] += s_dy[s][o] * v2;
        gb3[o] += s_dy[s][o];
      }
    }
  }
  // The two waves' small gradients, then everything to memory.
  if (q == 1) {
#pragma unroll
    for (int i = 0; i < NI; ++i) s_small[i][lane] = g1[i];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      s_small[NI + o][lane] = g3[o];
      if (lane == 0) s_y[0][o][0] = gb3[o];
    }
    s_small[NI + NO][lane] = gb1;
    s_small[NI + NO + 1][lane] = gb2;
  }
  __syncthreads();
  float* out = partial + static_cast<uint64_t>(blockIdx.x) * d.n_params;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) out[d.o_w2 + (32 * q + unit_of(0, v, hi)) * kH + 32 * b + lo] = g2[b][v];
  if (q == 1) return;
#pragma unroll
  for (int i = 0; i < NI; ++i) out[d.o_w1 + lane * NI + i] = g1[i] + s_small[i][lane];
  out[d.o_b1 + lane] = gb1 + s_small[NI + NO][lane];
  out[d.o_b2 + lane] = gb2 + s_small[NI + NO + 1][lane];
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    out[d.o_w3 + o * kH + lane] = g3[o] + s_small[NI + o][lane];
    if (lane == 0) out[d.o_b3 + o] = gb3[o] + s_y[0][o][0];
  }
  loss = wave_sum_f(loss);
  if (lane == 0) loss_part[blockIdx.x] = loss;
}

// Supported (n_in, n_out) shapes; F(ni, no) receives the compile-time pair.
template <class F>
void dispatch_shape(uint32_t ni, uint32_t no, F&& f) {
#define MG_MLP_SHAPE(A, B) \
  if (ni == A && no == B) return f(std::integral_constant<int, A>{}, std::integral_constant<int, B>{});
  MG_MLP_SHAPE(4, 1) MG_MLP_SHAPE(4, 2) MG_MLP_SHAPE(8, 1) MG_MLP_SHAPE(8, 2) MG_MLP_SHAPE(16, 1) MG_MLP_SHAPE(16, 2)
#undef MG_MLP_SHAPE
  fail(MG_ERR_UNSUPPORTED, "mlp: (n_in, n_out) must be in {4, 8, 16} x {1, 2}");
}

// grad[i] = sum over blocks of partial[b][i]: kReduceSlices threads per parameter take every
// kReduceSlices-th block in order, then their sums in slice order (a fixed order, no atomics). The first
// workgroup sums the losses the same way. With adam.w set, the Adam step on the FP32 masters and
// the BF16 copy follow in the same launch.
constexpr uint32_t kReduceSlices = 4;
constexpr uint32_t kReduceParams = 64;  // parameters per workgroup
struct AdamStep {
  float *w, *m, *v;
  uint16_t* w16;
  float lr, b1, b2, eps, c1, c2;
};
__global__ void __launch_bounds__(kReduceSlices* kReduceParams)
    mlp_reduce_kernel(const float* __restrict__ partial, const float* __restrict__ loss_part, uint32_t n_blocks,
                      uint32_t n_params, float* __restrict__ grad, float* __restrict__ loss, AdamStep adam) {
  __shared__ float s_sum[kReduceSlices][kReduceParams];
  const uint32_t slice = threadIdx.x / kReduceParams, col = threadIdx.x % kReduceParams;
  const uint32_t i = blockIdx.x * kReduceParams + col;
  float a = 0.f;
  if (i < n_params) {
#pragma unroll 8
    for (uint32_t b = slice; b < n_blocks; b += kReduceSlices) a += partial[static_cast<uint64_t>(b) * n_params + i];
  }
  s_sum[slice][col] = a;
  __syncthreads();
  if (slice == 0 && i < n_params) {
    float g = s_sum[0][col];
#pragma unroll
    for (uint32_t q = 1; q < kReduceSlices; ++q) g += s_sum[q][col];
    grad[i] = g;
    if (adam.w) {
      const float mi = adam.b1 * adam.m[i] + (1.f - adam.b1) * g;
      const float vi = adam.b2 * adam.v[i] + (1.f - adam.b2) * g * g;
      adam.m[i] = mi;
      adam.v[i] = vi;
      const float upd = adam.lr * (mi / adam.c1) / (sqrtf(vi / adam.c2) + adam.eps);
      const float w = adam.w[i] - upd;
      adam.w[i] = w;
      adam.w16[i] = f32_to_bf16(w);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < kWave) {
    float l = 0.f;
    for (uint32_t b = threadIdx.x; b < n_blocks; b += kWave) l += loss_part[b];
    l = wave_sum_f(l);
    if (threadIdx.x == 0) *loss = l;
  }
}

__global__ void to_bf16_kernel(const float* __restrict__ w, uint32_t n, uint16_t* __restrict__ w16) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w16[i] = f32_to_bf16(w[i]);
}

}  // namespace
}  // namespace mgamd

using namespace mgamd;

struct mg_mlp {
  int device = 0;
  Dims d{};
  DevBuf<float> w, m, v, grad, loss;
  DevBuf<uint16_t> w16;
  DevBuf<float> partial, loss_part;
  uint32_t partial_blocks = 0;
  uint64_t steps = 0;
};

namespace {

void ensure_partials(mg_mlp* p, uint32_t blocks) {
  if (blocks <= p->partial_blocks) return;
  p->partial.alloc(static_cast<size_t>(blocks) * p->d.n_params);
  p->loss_part.alloc(blocks);
  p->partial_blocks = blocks;
}

uint32_t tile_blocks(uint32_t n, uint32_t most) {
  return std::min(static_cast<uint32_t>((static_cast<uint64_t>(n) + kTileRows - 1) / kTileRows), most);
}

// Gradient of the mean loss over n samples, through p->grad and p->loss; then the Adam step if given.
void compute_grad(mg_context* ctx, mg_mlp* p, const float* x, const float* t, uint32_t n, const AdamStep& adam = {}) {
  const uint32_t blocks = tile_blocks(n, kGradBlocks);
  ensure_partials(p, blocks);
  const float scale = 1.f / (static_cast<float>(n) * p->d.n_out);
  dispatch_shape(p->d.n_in, p->d.n_out, [&](auto ni, auto no) {
    mlp_grad_kernel<decltype(ni)::value, decltype(no)::value>
        <<<blocks, 2 * kWave, 0, ctx->stream>>>(p->d, p->w16.get(), x, t, n, scale, p->partial.get(),
                                                p->loss_part.get());
  });
  MG_LAUNCH_CHECK();
  mlp_reduce_kernel<<<grid_for(p->d.n_params, kReduceParams), kReduceSlices * kReduceParams, 0, ctx->stream>>>(
      p->partial.get(), p->loss_part.get(), blocks, p->d.n_params, p->grad.get(), p->loss.get(), adam);
  MG_LAUNCH_CHECK();
}

// Forward of n rows into y, or with t their summed squared error into p->loss.
void launch_forward(mg_context* ctx, const mg_mlp* p, const float* x, uint32_t n, float* y, const float* t,
                    float* loss_part) {
  dispatch_shape(p->d.n_in, p->d.n_out, [&](auto ni, auto no) {
    mlp_forward_kernel<decltype(ni)::value, decltype(no)::value>
        <<<tile_blocks(n, kForwardBlocks), kMlpBlock, 0, ctx->stream>>>(p->d, p->w16.get(), x, n, y, t, loss_part);
  });
  MG_LAUNCH_CHECK();
}

}  // namespace

namespace mgamd {
void mlp_dims(const mg_mlp* p, uint32_t* n_in, uint32_t* n_out) {
  *n_in = p->d.n_in;
  *n_out = p->d.n_out;
}
}  // namespace mgamd

extern "C" int mg_mlp_create(mg_context* ctx, uint32_t n_in, uint32_t n_out, uint64_t seed, mg_mlp** out) {
  return guarded([&] {
    MG_REQUIRE(ctx && out, "mg_mlp_create: NULL argument");
    *out = nullptr;
    dispatch_shape(n_in, n_out, [](auto, auto) {});  // rejects unsupported shapes
    DeviceGuard g(ctx->device);
    auto p = std::make_unique<mg_mlp>();
    p->device = ctx->device;
    p->d = make_dims(n_in, n_out);
    const uint32_t np = p->d.n_params;
    // He-uniform initial weights from the SplitMix64 stream of `seed`; zero biases.
    std::vector<float> w(np, 0.f);
    const uint64_t key = stream_key(seed, 5);
    auto fill = [&](uint32_t off, uint32_t count, uint32_t fan_in) {
      const float lim = std::sqrt(6.f / static_cast<float>(fan_in));
      for (uint32_t i = 0; i < count; ++i) {
        const double u = static_cast<double>(sm64_at(key, off + i) >> 11) * (1.0 / 9007199254740992.0);
        w[off + i] = static_cast<float>((2.0 * u - 1.0) * lim);
      }
    };
    fill(p->d.o_w1, kH * n_in, n_in);
    fill(p->d.o_w2, kH * kH, kH);
    fill(p->d.o_w3, n_out * kH, kH);
    p->w.alloc(np);
    p->m.alloc(np);
    p->v.alloc(np);
    p->grad.alloc(np);
    p->loss.alloc(1);
    p->w16.alloc(np);
    MG_HIP(hipMemcpyAsync(p->w.get(), w.data(), sizeof(float) * np, hipMemcpyHostToDevice, ctx->stream));
    MG_HIP(hipMemsetAsync(p->m.get(), 0, sizeof(float) * np, ctx->stream));
    MG_HIP(hipMemsetAsync(p->v.get(), 0, sizeof(float) * np, ctx->stream));
    to_bf16_kernel<<<grid_for(np, 256), 256, 0, ctx->stream>>>(p->w.get(), np, p->w16.get());
    MG_LAUNCH_CHECK();
    MG_HIP(hipStreamSynchronize(ctx->stream));
    *out = p.release();
  });
}

extern "C" int mg_mlp_num_params(const mg_mlp* p, uint32_t* n_params) {
  return guarded([&] {
    MG_REQUIRE(p && n_params, "mg_mlp_num_params: NULL argument");
    *n_params = p->d.n_params;
  });
}

extern "C" int mg_mlp_get_params(mg_context* ctx, const mg_mlp* p, float* master, uint16_t* bf16) {
  return guarded([&] {
    MG_REQUIRE(ctx && p, "mg_mlp_get_params: NULL argument");
    DeviceGuard g(ctx->device);
    if (master)
      MG_HIP(hipMemcpyAsync(master, p->w.get(), sizeof(float) * p->d.n_params, hipMemcpyDeviceToHost, ctx->stream));
    if (bf16)
      MG_HIP(hipMemcpyAsync(bf16, p->w16.get(), sizeof(uint16_t) * p->d.n_params, hipMemcpyDeviceToHost, ctx->stream));
    MG_HIP(hipStreamSynchronize(ctx->stream));
  });
}

extern "C" int mg_mlp_set_params(mg_context* ctx, mg_mlp* p, const float* master) {
  return guarded([&] {
    MG_REQUIRE(ctx && p && master, "mg_mlp_set_params: NULL argument");
    DeviceGuard g(ctx->device);
    MG_HIP(hipMemcpyAsync(p->w.get(), master, sizeof(float) * p->d.n_params, hipMemcpyHostToDevice, ctx->stream));
    to_bf16_kernel<<<grid_for(p->d.n_params, 256), 256, 0, ctx->stream>>>(p->w.get(), p->d.n_params, p->w16.get());
    MG_LAUNCH_CHECK();
    MG_HIP(hipStreamSynchronize(ctx->stream));
  });
}

extern "C" int mg_mlp_forward(mg_context* ctx, const mg_mlp* p, const float* x, uint32_t n, float* y) {
  return guarded([&] {
    MG_REQUIRE(ctx && p && (n == 0 || (x && y)), "mg_mlp_forward: NULL argument");
    if (n == 0) return;
    DeviceGuard g(ctx->device);
    launch_forward(ctx, p, x, n, y, nullptr, nullptr);
  });
}

extern "C" int mg_mlp_loss_grad(mg_context* ctx, mg_mlp* p, const float* x, const float* t, uint32_t n, float* loss,
                                float* grad) {
  return guarded([&] {
    MG_REQUIRE(ctx && p && x && t && n > 0, "mg_mlp_loss_grad: bad argument");
    DeviceGuard g(ctx->device);
    compute_grad(ctx, p, x, t, n);
    float l = 0.f;
    if (grad) MG_HIP(hipMemcpyAsync(grad, p->grad.get(), sizeof(float) * p->d.n_params, hipMemcpyDeviceToHost, ctx->stream));
    read_words(ctx, {p->loss.get(), &l, sizeof(l)});
    if (loss) *loss = l / (static_cast<float>(n) * p->d.n_out);
  });
}

extern "C" int mg_mlp_train(mg_context* ctx, mg_mlp* p, const float* x, const float* t, uint32_t n, uint32_t epochs,
                            uint32_t batch, float lr, float* final_loss) {
  return guarded([&] {
    MG_REQUIRE(ctx && p && x && t && n > 0 && batch > 0, "mg_mlp_train: bad argument");
    DeviceGuard g(ctx->device);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
      for (uint32_t s0 = 0; s0 < n; s0 += batch) {
        const uint32_t nb = std::min(batch, n - s0);
        ++p->steps;
        const float c1 = 1.f - std::pow(b1, static_cast<float>(p->steps));
        const float c2 = 1.f - std::pow(b2, static_cast<float>(p->steps));
        compute_grad(ctx, p, x + static_cast<uint64_t>(s0) * p->d.n_in, t + static_cast<uint64_t>(s0) * p->d.n_out, nb,
                     AdamStep{p->w.get(), p->m.get(), p->v.get(), p->w16.get(), lr, b1, b2, eps, c1, c2});
      }
    }
    if (final_loss) {
      // The loss needs no gradient: forward only, then the sum of its parts.
      const uint32_t blocks = tile_blocks(n, kForwardBlocks);
      ensure_partials(p, blocks);
      launch_forward(ctx, p, x, n, nullptr, t, p->loss_part.get());
      mlp_reduce_kernel<<<1, kReduceSlices * kReduceParams, 0, ctx->stream>>>(
          p->partial.get(), p->loss_part.get(), blocks, 0, p->grad.get(), p->loss.get(), AdamStep{});
      MG_LAUNCH_CHECK();
      float l = 0.f;
      read_words(ctx, {p->loss.get(), &l, sizeof(l)});
      *final_loss = l / (static_cast<float>(n) * p->d.n_out);
    }
  });
}

extern "C" int mg_mlp_destroy(mg_mlp* p) {
  return guarded([&] {
    if (!p) return;
    DeviceGuard g(p->device);
    FreeScope frees;
    delete p;
  });
}
