// Training and batch-inference kernels of the learned weno5 weights.
//
// The network (5 -> 32 -> 32 -> 3, GELU, softmax) maps the normalised
// one-sided differences of a weno5 stencil to the weights of its three
// candidate polynomials.  A training sample is 8 floats (5 inputs, the 3
// candidate polynomials divided by max|d|) plus a target (the fine-grid
// derivative times dx / max|d|); the loss is the mean squared error of
// sum_k w_k p_k.
//
// kMlpGrad: four waves per workgroup, 32 samples per tile.  A step of the
// optimiser is a chain of dependent launches over a few thousand samples, so
// the length of a tile's own chain bounds it: a thread holds one sample and
// four of the 32 hidden units, and each 32x32 product of the tile is one
// v_mfma_f32_16x16x32_bf16 per wave (bf16 operands, fp32 accumulate) -- the
// forward product H1 W2^T, the input gradient dZ2 W2, and the weight
// gradient dZ2^T H1, which stays in the accumulators over all tiles.  The
// 5->32 and 32->3 layers, GELU, softmax and loss run on the vector ALUs in
// fp32, with the inputs and the activations rounded to bf16 where the
// inference's matrix products take them.  8192 samples: 30 -> 9.7 us against
// one wave per tile of 64 samples (128 waves on 256 CUs, 32 units a lane one
// after the other).
// kMlpReduce: the partial rows of the workgroups summed in a fixed order
// (deterministic), 16 lanes to a parameter; a training step's Adam update of
// the fp32 master parameters follows in the same launch.  256 rows: 4 us
// (one lane to a parameter: 32 us for 128 rows, and 5 us for a launch of its
// own for Adam).
//
// MFMA lane layouts (16x16x32 bf16): A operand lane l holds row l%16,
// k = 8*(l/16) .. +7; B operand lane l holds column l%16, same k; the fp32
// accumulator element r of lane l is row 4*(l/16) + r, column l%16.
#include <hip/hip_runtime.h>

#include "lsg_device.hpp"
#include "lsg_items.hpp"
#include "lsg_learned.hpp"

namespace lsg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// GELU x sigmoid(2u) (mlpGelu) and its derivative
// sigmoid(2u) + 2 x sigmoid(2u) (1 - sigmoid(2u)) u'.
__device__ inline float geluD(float x, float &dg) {
  const float c = 0.7978845608028654f, a = 0.044715f;
  const float x2 = x * x;
  const float u = c * (x + a * x2 * x);
  const float sg = mlpSigmoid2(u);
  dg = sg + 2.0f * x * sg * (1.0f - sg) * c * (1.0f + 3.0f * a * x2);
  return x * sg;
}

__device__ inline bf16x8 loadBf16x8(const uint16_t *v) {  // 16-byte aligned
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const i16x8 *>(v));
}

constexpr int TILE = 32;  // samples of a tile
constexpr int HP = 40;    // padded row length (bf16) of the bf16 tiles: 16-byte rows on distinct banks
constexpr int FP = 33;    // padded row length (fp32) of the fp32 tiles
constexpr int UNITS = 4;  // hidden units of a thread
constexpr int PARTS = MLP_H / UNITS;
constexpr int SUMS = MLP_IN + 2 + MLP_OUT + 1;  // column sums: dW1, db1, db2, dW3, db3
static_assert(MLP_H == 32 && TILE == 32 && PARTS * TILE == 256, "four waves, one 16x16 tile of a product each");

struct MlpLds {
  alignas(16) uint16_t w2[MLP_H][HP];   // W2 as bf16, row j (output), column i (input)
  alignas(16) uint16_t w2t[MLP_H][HP];  // W2 transposed
  alignas(16) uint16_t h1[TILE][HP];    // bf16 activations of layer 1, row = sample
  alignas(16) uint16_t h1t[MLP_H][HP];  // the same, row = unit
  alignas(16) uint16_t dz2b[TILE][HP];  // dz2 as bf16, row = sample
  alignas(16) uint16_t dz2t[MLP_H][HP]; // the same, row = unit
  float w1[MLP_H * MLP_IN], b1[MLP_H], b2[MLP_H], w3[MLP_OUT * MLP_H], b3[4];
  float buf1[TILE][FP];  // z2, then dz2
  float buf2[TILE][FP];  // h2
  float buf3[TILE][FP];  // dh1, then dz1
  float z3[PARTS][TILE][MLP_OUT];
  float xs[TILE][MLP_IN];
  float dz3[TILE][4];
  float sums[PARTS][MLP_H][SUMS];
  float loss[TILE];
};

// Partial gradient of a workgroup over its tiles of samples [0, n): row
// partials[blockIdx.x][0..MLP_NPARAM) and the summed squared residual at
// [MLP_NPARAM].  invCount = 1 / (number of samples of the loss).
__global__ __launch_bounds__(256) void kMlpGrad(const float *X, const float *T, uint32_t n, float invCount,
                                               const float *P, float *partials) {
  __shared__ MlpLds L;
  const int t = threadIdx.x, l = t & 63, wave = t >> 6;
  // stage the parameters (weights as their bf16 values)
  for (int e = t; e < MLP_H * MLP_H; e += 256) {
    const int j = e / MLP_H, i = e % MLP_H;
    const uint16_t b = bf16Bits(P[MLP_W2 + e]);
    L.w2[j][i] = b;
    L.w2t[i][j] = b;
  }
  if (t < MLP_H * MLP_IN) L.w1[t] = bf16Float(bf16Bits(P[MLP_W1 + t]));
  if (t < MLP_OUT * MLP_H) L.w3[t] = bf16Float(bf16Bits(P[MLP_W3 + t]));
  if (t < MLP_H) {
    L.b1[t] = P[MLP_B1 + t];
    L.b2[t] = P[MLP_B2 + t];
  }
  if (t < MLP_OUT) L.b3[t] = P[MLP_B3 + t];
  __syncthreads();

  // thread: sample s of the tile, units u0 .. u0 + 3; as column sums: unit s,
  // samples u0 .. u0 + 3
  const int s = t % TILE, part = t / TILE, u0 = part * UNITS;
  // wave: the 16x16 tile (row block tr, column block tc) of each product
  const int tr = 16 * (wave >> 1), tc = 16 * (wave & 1), col = l & 15, k0 = 8 * (l >> 4), r0 = 4 * (l >> 4);
  const bf16x8 bForward = loadBf16x8(&L.w2[tc + col][k0]), bBack = loadBf16x8(&L.w2t[tc + col][k0]);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 accW2 = zero;
  float sum[SUMS];
  for (int q = 0; q < SUMS; ++q) sum[q] = 0.f;
  float lossAcc = 0;

  for (uint32_t base = blockIdx.x * TILE; base < n; base += gridDim.x * TILE) {
    const uint32_t g = base + s;
    float x[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    float target = 0;
    if (g < n) {
      for (int q = 0; q < 8; ++q) x[q] = X[(size_t)g * 8 + q];
      target = T[g];
    }
    // the inputs enter layer 1 as bf16 (as in the matrix-core inference)
    for (int i = 0; i < MLP_IN; ++i) x[i] = bf16Float(bf16Bits(x[i]));
    // layer 1, keep gelu'
    float d1[UNITS];
    for (int q = 0; q < UNITS; ++q) {
      const int u = u0 + q;
      float z = L.b1[u];
      for (int i = 0; i < MLP_IN; ++i) z += L.w1[u * MLP_IN + i] * x[i];
      const uint16_t h = bf16Bits(geluD(z, d1[q]));
      L.h1[s][u] = h;
      L.h1t[u][s] = h;
    }
    if (part == 0)
      for (int i = 0; i < MLP_IN; ++i) L.xs[s][i] = x[i];
    __syncthreads();
    // layer 2 forward: Z2[s][j] = sum_i H1[s][i] W2[j][i]
    {
      const f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(loadBf16x8(&L.h1[tr + col][k0]), bForward, zero, 0, 0, 0);
      for (int r = 0; r < 4; ++r) L.buf1[tr + r0 + r][tc + col] = z[r];
    }
    __syncthreads();
    // layer 2 activation, this thread's part of layer 3
    float d2[UNITS], z3[MLP_OUT] = {0.f, 0.f, 0.f};
    for (int q = 0; q < UNITS; ++q) {
      const int u = u0 + q;
      const float h = bf16Float(bf16Bits(geluD(L.buf1[s][u] + L.b2[u], d2[q])));  // enters layer 3 as bf16
      L.buf2[s][u] = h;
      for (int k = 0; k < MLP_OUT; ++k) z3[k] += L.w3[k * MLP_H + u] * h;
    }
    for (int k = 0; k < MLP_OUT; ++k) L.z3[part][s][k] = z3[k];
    __syncthreads();
    // softmax and loss, by each of the sample's threads
    for (int k = 0; k < MLP_OUT; ++k) {
      z3[k] = L.b3[k];
      for (int p = 0; p < PARTS; ++p) z3[k] += L.z3[p][s][k];
    }
    const float m = fmaxf(z3[0], fmaxf(z3[1], z3[2]));
    float w[MLP_OUT], se = 0;
    for (int k = 0; k < MLP_OUT; ++k) {
      w[k] = mlpExp(z3[k] - m);
      se += w[k];
    }
    for (int k = 0; k < MLP_OUT; ++k) w[k] = w[k] / se;
    const float pred = w[0] * x[5] + w[1] * x[6] + w[2] * x[7];
    const float res = (g < n) ? pred - target : 0.f;
    lossAcc += res * res;
    const float dpred = 2.f * res * invCount;
    float dw[MLP_OUT], dz3[MLP_OUT];
    for (int k = 0; k < MLP_OUT; ++k) dw[k] = dpred * x[5 + k];
    const float wdw = w[0] * dw[0] + w[1] * dw[1] + w[2] * dw[2];
    for (int k = 0; k < MLP_OUT; ++k) {
      dz3[k] = w[k] * (dw[k] - wdw);
      if (part == 0) L.dz3[s][k] = dz3[k];
    }
    for (int q = 0; q < UNITS; ++q) {
      const int u = u0 + q;
      float dh = 0;
      for (int k = 0; k < MLP_OUT; ++k) dh += L.w3[k * MLP_H + u] * dz3[k];
      const float dz2 = dh * d2[q];
      L.buf1[s][u] = dz2;  // this thread's own z2 before
      const uint16_t b = bf16Bits(dz2);
      L.dz2b[s][u] = b;
      L.dz2t[u][s] = b;
    }
    __syncthreads();
    // layer 2 backward: dH1[s][i] = sum_j dZ2[s][j] W2[j][i] and
    // dW2[j][i] += sum_s dZ2[s][j] H1[s][i]
    {
      const f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(loadBf16x8(&L.dz2b[tr + col][k0]), bBack, zero, 0, 0, 0);
      accW2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(loadBf16x8(&L.dz2t[tr + col][k0]),
                                                      loadBf16x8(&L.h1t[tc + col][k0]), accW2, 0, 0, 0);
      for (int r = 0; r < 4; ++r) L.buf3[tr + r0 + r][tc + col] = z[r];
    }
    __syncthreads();
    for (int q = 0; q < UNITS; ++q) L.buf3[s][u0 + q] *= d1[q];  // dz1
    __syncthreads();
    for (int q = 0; q < UNITS; ++q) {
      const int sm = u0 + q, u = s;
      const float dz1 = L.buf3[sm][u], h2 = L.buf2[sm][u];
      for (int i = 0; i < MLP_IN; ++i) sum[i] += dz1 * L.xs[sm][i];
      sum[MLP_IN] += dz1;
      sum[MLP_IN + 1] += L.buf1[sm][u];
      for (int k = 0; k < MLP_OUT; ++k) sum[MLP_IN + 2 + k] += L.dz3[sm][k] * h2;
      if (u < MLP_OUT) sum[SUMS - 1] += L.dz3[sm][u];
    }
    __syncthreads();
  }
  // combine the parts and write the partial row
  float *out = partials + (size_t)blockIdx.x * MLP_PSTRIDE;
  for (int q = 0; q < SUMS; ++q) L.sums[part][s][q] = sum[q];
  if (part == 0) L.loss[s] = lossAcc;
  __syncthreads();
  for (int e = t; e < MLP_H * SUMS; e += 256) {
    const int u = e / SUMS, q = e % SUMS;
    float v = 0;
    for (int p = 0; p < PARTS; ++p) v += L.sums[p][u][q];
    if (q < MLP_IN) out[MLP_W1 + u * MLP_IN + q] = v;
    else if (q == MLP_IN) out[MLP_B1 + u] = v;
    else if (q == MLP_IN + 1) out[MLP_B2 + u] = v;
    else if (q < SUMS - 1) out[MLP_W3 + (q - MLP_IN - 2) * MLP_H + u] = v;
    else if (u < MLP_OUT) out[MLP_B3 + u] = v;
  }
  for (int r = 0; r < 4; ++r) out[MLP_W2 + (tr + r0 + r) * MLP_H + tc + col] = accW2[r];
  if (t == 0) {
    float v = 0;
    for (int q = 0; q < TILE; ++q) v += L.loss[q];
    out[MLP_NPARAM] = v;
  }
}

// Sum of the partial rows in a fixed order, 16 parameters a workgroup; with
// P given, Adam on the fp32 master parameters (Kingma & Ba 2015), step >= 1.
constexpr int RED = 16;
__global__ __launch_bounds__(RED * RED) void kMlpReduce(const float *partials, int rows, float *grad, float *P,
                                                        float *M, float *V, int step, float lr, float b1, float b2,
                                                        float eps) {
  __shared__ float sum[RED][RED + 1];
  const int q = threadIdx.x % RED, g = threadIdx.x / RED;
  const int p = blockIdx.x * RED + q;
  float s = 0;
  if (p < MLP_PSTRIDE) {
#pragma unroll 8
    for (int r = g; r < rows; r += RED) s += partials[(size_t)r * MLP_PSTRIDE + p];
  }
  sum[g][q] = s;
  __syncthreads();
  if (g != 0 || p > MLP_NPARAM) return;
  s = 0;
  for (int r = 0; r < RED; ++r) s += sum[r][q];
  grad[p] = s;
  if (!P || p == MLP_NPARAM) return;
  const float m = b1 * M[p] + (1.f - b1) * s;
  const float v = b2 * V[p] + (1.f - b2) * s * s;
  M[p] = m;
  V[p] = v;
  const float mh = m / (1.f - powf(b1, (float)step));
  const float vh = v / (1.f - powf(b2, (float)step));
  P[p] -= lr * mh / (sqrtf(vh) + eps);
}

// Learned weno5 on n stencils of 7 values (test and inspection entry).
__global__ void kWenoLearned(uint32_t n, const double *x, double dx, int plus, const uint16_t *prm, double *out) {
  __shared__ float W[MLP_NPARAM];
  for (int i = threadIdx.x; i < MLP_NPARAM; i += blockDim.x) W[i] = bf16Float(prm[i]);
  __syncthreads();
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double st[7];
    for (int k = 0; k < 7; ++k) st[k] = x[(size_t)i * 7 + k];
    out[i] = weno5Learned(st, dx, plus != 0, W);
  }
}

void launchWenoLearned(hipStream_t s, uint32_t n, const double *x, double dx, int plus, const uint16_t *prm,
                       double *out) {
  uint32_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks == 0) blocks = 1;
  kWenoLearned<<<blocks, 256, 0, s>>>(n, x, dx, plus, prm, out);
}

int mlpGradRows(uint32_t n, int most) {
  const uint32_t tiles = (n + TILE - 1) / TILE;
  return tiles < (uint32_t)most ? (int)tiles : most;
}

void launchMlpGrad(hipStream_t s, const float *X, const float *T, uint32_t n, float *P, float *partials, int rows,
                   float *grad, float *M, float *V, int step, float lr) {
  kMlpGrad<<<rows, 256, 0, s>>>(X, T, n, 1.0f / (float)n, P, partials);
  kMlpReduce<<<(MLP_PSTRIDE + RED - 1) / RED, RED * RED, 0, s>>>(partials, rows, grad, M ? P : nullptr, M, V, step, lr,
                                                                 0.9f, 0.999f, 1e-8f);
}

}  // namespace lsg
