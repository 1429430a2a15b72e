// The learned warm-start network: an 8 -> 64 -> 64 -> 1 MLP with GELU, BF16 weights and
// activations on the matrix cores (v_mfma_f32_16x16x16_bf16) with FP32 accumulation.
// No reference counterpart: it predicts a particle's initial lambda for the PBF solver.
//
// A wave works on tiles of 16 rows (particles or training samples), transposed: the weights
// are the A operand and the rows the columns of B, so a layer's result has the layout of
// the next layer's B operand (a lane keeps its row and four consecutive hidden units) and
// activations go from layer to layer in registers.  The 64 -> 1 head and the elementwise
// work run on the VALU.
//
// Operand layout of v_mfma_f32_16x16x16_bf16 (lane l, j = 0..3):
//   A (16 x 16, M x K): A[l % 16][4 * (l / 16) + j]
//   B (16 x 16, K x N): B[4 * (l / 16) + j][l % 16]
//   D (16 x 16, M x N): D[4 * (l / 16) + j][l % 16]
//
// Parameter vector (fp32 master copy, 4801 values):
//   W1[8][64] (input k, hidden n) | b1[64] | W2[64][64] (k, n) | b2[64] | w3[64] | b3
#include "rtp_mlp.hpp"

namespace rtp {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short f2bf(float f)
{
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (short)(u >> 16);
}

constexpr float kGeluA = 0.7978845608028654f;  // sqrt(2 / pi)
constexpr float kGeluB = 0.044715f;

// tanh-form GELU, 0.5 z (1 + tanh u) with u = sqrt(2/pi) (z + 0.044715 z^3), evaluated as
// z * sigmoid(2u) = z / (1 + exp(-2u)) with the hardware exponential and reciprocal (about
// 1e-6 relative; the network is trained with these same functions).
__device__ __forceinline__ float sigmoid2u(float z)
{
  const float u = kGeluA * (z + kGeluB * (z * z) * z);
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(u * (-2.0f * 1.44269504f)));
}

__device__ __forceinline__ float gelu(float z) { return z * sigmoid2u(z); }

// d/dz [z sigmoid(2u)] = s + z s (1 - s) 2 u'(z),  u' = sqrt(2/pi) (1 + 3 * 0.044715 z^2)
__device__ __forceinline__ float gelu_grad(float z)
{
  const float sg = sigmoid2u(z);
  return sg + z * sg * (1.0f - sg) * (2.0f * kGeluA) * (1.0f + 3.0f * kGeluB * z * z);
}

// Four consecutive bf16 (8-byte aligned) as one operand register.
__device__ __forceinline__ bf16x4 ld4(const short* p) { return *reinterpret_cast<const bf16x4*>(p); }

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Four floats rounded to bf16 (nearest even, as f2bf).
__device__ __forceinline__ bf16x4 to_bf16(f32x4 v)
{
  typedef __bf16 bfv4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(bf16x4, __builtin_convertvector(v, bfv4));
}

// GELU and its derivative of four pre-activations (gelu, gelu_grad).
__device__ __forceinline__ f32x4 gelu4(f32x4 z)
{
  return f32x4{ gelu(z[0]), gelu(z[1]), gelu(z[2]), gelu(z[3]) };
}
__device__ __forceinline__ f32x4 gelu_grad4(f32x4 z)
{
  return f32x4{ gelu_grad(z[0]), gelu_grad(z[1]), gelu_grad(z[2]), gelu_grad(z[3]) };
}

// The lane's part of a row's standardised inputs as layer 1's B operand: inputs 4 lq + j for
// lq < 2; inputs 8..15 of the padded layer are zero, an invalid row standardises zeros.
struct InputScale {
  f32x4 mu, inv;
  __device__ __forceinline__ InputScale(const MlpDev& m, uint32_t lq)
  {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      mu[j] = lq == 1u ? m.mu[4 + j] : m.mu[j];
      inv[j] = lq == 1u ? m.invSigma[4 + j] : m.invSigma[j];
    }
  }
  __device__ __forceinline__ bf16x4 operator()(const float* __restrict__ feat, uint32_t src, bool valid,
                                               uint32_t lq) const
  {
    f32x4 x = { 0.0f, 0.0f, 0.0f, 0.0f };
    if (lq < 2u) {
      if (valid)  // feat rows are 32-byte aligned
        x = *reinterpret_cast<const f32x4*>(feat + (size_t)src * 8 + 4 * lq);
      x = (x - mu) * inv;
    }
    return to_bf16(x);
  }
};

// The head of a row from this lane's y[j] = sum over t of gelu(z2) w3 at hidden units 16 t + 4 lq
// + j: the sums of lanes lq ^ 2, lq ^ 1, then j ^ 2, j ^ 1.
__device__ __forceinline__ float head_sum(f32x4 y)
{
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    y[j] += __shfl_xor(y[j], 32, 64);
    y[j] += __shfl_xor(y[j], 16, 64);
  }
  return (y[0] + y[2]) + (y[1] + y[3]);
}

// Inference: each wave keeps its lanes' weights in registers and runs two tiles of 16 rows at
// a time (two independent chains) in a grid-stride loop.  Bound by issue: 128 GELUs a row, two
// quarter-rate transcendentals each.
constexpr uint32_t kFwdTiles = 2;
__global__ __launch_bounds__(256) void k_mlp_forward(const float* __restrict__ feat, uint32_t n, MlpDev m,
                                                     float* __restrict__ out,
                                                     float4* __restrict__ packed)
{
  const uint32_t l = threadIdx.x & 63u, lr = l % 16u, lq = l / 16u;
  const InputScale inputs(m, lq);
  bf16x4 w1[4], w2[4][4];
  f32x4 b1[4], b2[4], w3[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    w1[u] = ld4(m.w1t + (u * 16 + lr) * 16 + 4 * lq);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      w2[u][t] = ld4(m.w2t + (u * 16 + lr) * 64 + t * 16 + 4 * lq);
    const float* at = m.p + u * 16 + 4 * lq;  // the offsets are multiples of four floats
    b1[u] = *reinterpret_cast<const f32x4*>(at + kMlpB1);
    b2[u] = *reinterpret_cast<const f32x4*>(at + kMlpB2);
    w3[u] = *reinterpret_cast<const f32x4*>(at + kMlpW3);
  }
  const float b3 = m.p[kMlpB3];
  const uint32_t rows = 16u * kFwdTiles, waves = gridDim.x * 4u;
  const uint32_t groups = (n + rows - 1u) / rows;
  for (uint32_t g = blockIdx.x * 4u + (threadIdx.x >> 6); g < groups; g += waves) {
    const uint32_t row0 = g * rows;
    bf16x4 h[kFwdTiles][4];
#pragma unroll
    for (uint32_t k = 0; k < kFwdTiles; ++k) {
      const uint32_t r = row0 + k * 16u + lr;
      const bf16x4 x = inputs(feat, r, r < n, lq);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f32x4 z = mfma(w1[t], x, f32x4{ 0.0f, 0.0f, 0.0f, 0.0f });
        h[k][t] = to_bf16(gelu4(z + b1[t]));
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < kFwdTiles; ++k) {
      f32x4 y = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        f32x4 z = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
        for (int t = 0; t < 4; ++t)
          z = mfma(w2[u][t], h[k][t], z);
        y += gelu4(z + b2[u]) * w3[u];
      }
      const float v = head_sum(y) + b3;
      const uint32_t r = row0 + k * 16u + lr;
      if (lq == 0 && r < n) {
        out[r] = v * m.outScale;
        if (packed)
          packed[r].w = v * m.outScale;
      }
    }
  }
}

// Q[row][c] held as lane (row = lr, c = 4 lq + j) -> lane (c = lr, row = 4 lq + j): a product
// with the identity, exact (one term of each sum is not zero).
__device__ __forceinline__ bf16x4 transpose16(bf16x4 q, bf16x4 identity)
{
  return to_bf16(mfma(q, identity, f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }));
}

// Forward + backward of the mean squared error over a batch.  A wave carries a tile of 16
// rows from the inputs to the last gradient in registers (the two products that contract
// over rows read tiles transposed by transpose16) and adds up every gradient over its tiles;
// a workgroup's waves put their sums side by side in LDS, and the workgroup writes their sum as
// one partial gradient (its squared errors as entry kMlpParams), which k_mlp_update or
// k_mlp_sum adds up in order, so a batch's gradient repeats bit for bit.  Bound by the one wave
// a SIMD that the sums leave room for (300 registers).  65,536 rows: 27 us, and 5 us for
// k_mlp_update; a 64-row wave with its tile in 58 KB of LDS (two waves a CU) and 4.9 M atomics
// on 4,801 words took 78 us, and 10 us for the step and the operand copies apart.
constexpr uint32_t kTrainWaves = 4;
constexpr uint32_t kW1Pitch = 20, kW2Pitch = 68;  // shorts per row in LDS: 16 rows' 8-byte reads on distinct banks
__global__ __launch_bounds__(64 * kTrainWaves) void k_mlp_train(const float* __restrict__ feat,
                                                                const float* __restrict__ target,
                                                                const uint32_t* __restrict__ perm,
                                                                uint32_t n, float invBatch, MlpDev m,
                                                                float* __restrict__ partial)
{
  __shared__ __align__(16) short sw1[64 * kW1Pitch], sw2t[64 * kW2Pitch], sw2[64 * kW2Pitch];
  __shared__ __align__(16) float sb1[64], sb2[64], sw3[64];
  __shared__ float sums[kTrainWaves][kMlpPartial];
  const uint32_t l = threadIdx.x & 63u, lr = l % 16u, lq = l / 16u, w = threadIdx.x >> 6;
  for (uint32_t i = 4u * threadIdx.x; i < 64u * 64u; i += 4u * blockDim.x) {
    const uint32_t at = (i >> 6) * kW2Pitch + (i & 63u);
    *reinterpret_cast<bf16x4*>(sw2t + at) = ld4(m.w2t + i);
    *reinterpret_cast<bf16x4*>(sw2 + at) = ld4(m.w2 + i);
  }
  if (4u * threadIdx.x < 64u * 16u) {
    const uint32_t i = 4u * threadIdx.x;
    *reinterpret_cast<bf16x4*>(sw1 + (i >> 4) * kW1Pitch + (i & 15u)) = ld4(m.w1t + i);
  }
  if (threadIdx.x < 64u) {
    sb1[threadIdx.x] = m.p[kMlpB1 + threadIdx.x];
    sb2[threadIdx.x] = m.p[kMlpB2 + threadIdx.x];
    sw3[threadIdx.x] = m.p[kMlpW3 + threadIdx.x];
  }
  __syncthreads();
  const f32x4 zero = { 0.0f, 0.0f, 0.0f, 0.0f };
  const InputScale inputs(m, lq);
  const float b3 = m.p[kMlpB3];
  const auto four = [&](const float* p, int t) { return *reinterpret_cast<const f32x4*>(p + t * 16 + 4 * lq); };
  bf16x4 identity;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    identity[j] = 4u * lq + j == lr ? (short)0x3f80 : (short)0;
  f32x4 dW2[4][4], dW1[4], db1[4], db2[4], dw3[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    dW1[t] = db1[t] = db2[t] = dw3[t] = zero;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      dW2[t][u] = zero;
  }
  float db3 = 0.0f, se = 0.0f;
  const uint32_t tiles = (n + 15u) / 16u;
  for (uint32_t tile = blockIdx.x * kTrainWaves + w; tile < tiles; tile += gridDim.x * kTrainWaves) {
    // the weights stay in LDS: hoisted out of the loop they would spill the gradient sums
    asm volatile("" ::: "memory");
    const uint32_t row = tile * 16u + lr;
    const bool valid = row < n;
    const uint32_t src = valid ? (perm ? perm[row] : row) : 0u;
    const float goal = valid ? target[src] / m.outScale : 0.0f;
    const bf16x4 x = inputs(feat, src, valid, lq);
    bf16x4 h[4], d2[4];
    f32x4 g1[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x4 z = mfma(ld4(sw1 + (t * 16 + lr) * kW1Pitch + 4 * lq), x, zero) + four(sb1, t);
      h[t] = to_bf16(gelu4(z));
      g1[t] = gelu_grad4(z);
    }
    f32x4 a2[4], g2[4], y = zero;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f32x4 z = zero;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        z = mfma(ld4(sw2t + (u * 16 + lr) * kW2Pitch + t * 16 + 4 * lq), h[t], z);
      z += four(sb2, u);
      a2[u] = gelu4(z);
      g2[u] = gelu_grad4(z);
      y += a2[u] * four(sw3, u);
    }
    const float e = valid ? head_sum(y) + b3 - goal : 0.0f;
    const float dy = 2.0f * e * invBatch;
    if (lq == 0) {  // the four lanes of a row hold the same error
      se += e * e;
      db3 += dy;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const f32x4 dz = (dy * four(sw3, u)) * g2[u];
      dw3[u] += a2[u] * dy;
      db2[u] += dz;
      d2[u] = to_bf16(dz);
    }
    bf16x4 hT[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      hT[t] = transpose16(h[t], identity);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bf16x4 dT = transpose16(d2[u], identity);
#pragma unroll
      for (int t = 0; t < 4; ++t)  // dW2[k][n] = sum over rows of h1[row][k] dz2[row][n]
        dW2[t][u] = mfma(hT[t], dT, dW2[t][u]);
    }
    const bf16x4 xT = transpose16(x, identity);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 dh = zero;  // dh1[k][row] = sum over n of W2[k][n] dz2[row][n]
#pragma unroll
      for (int u = 0; u < 4; ++u)
        dh = mfma(ld4(sw2 + (t * 16 + lr) * kW2Pitch + u * 16 + 4 * lq), d2[u], dh);
      const f32x4 dz = dh * g1[t];
      db1[t] += dz;
      // dW1[k][n] = sum over rows of x[row][k] dz1[row][n]
      dW1[t] = mfma(xT, transpose16(to_bf16(dz), identity), dW1[t]);
    }
  }
  // sums over the tile's rows
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        db1[t][j] += __shfl_xor(db1[t][j], o, 64);
        db2[t][j] += __shfl_xor(db2[t][j], o, 64);
        dw3[t][j] += __shfl_xor(dw3[t][j], o, 64);
      }
    se += __shfl_xor(se, o, 64);
    db3 += __shfl_xor(db3, o, 64);
  }
  float* const own = sums[w];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t k = t * 16 + 4 * lq + j;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        own[kMlpW2 + k * 64 + u * 16 + lr] = dW2[t][u][j];
      if (lq < 2)
        own[kMlpW1 + (4 * lq + j) * 64 + t * 16 + lr] = dW1[t][j];
      if (lr == 0) {
        own[kMlpB1 + k] = db1[t][j];
        own[kMlpB2 + k] = db2[t][j];
        own[kMlpW3 + k] = dw3[t][j];
      }
    }
  if (l == 0) {
    own[kMlpB3] = db3;
    own[kMlpParams] = se;
  }
  __syncthreads();
  float* const mine = partial + (size_t)blockIdx.x * kMlpPartial;
  for (uint32_t i = threadIdx.x; i <= (uint32_t)kMlpParams; i += blockDim.x) {
    float v = sums[0][i];
#pragma unroll
    for (uint32_t k = 1; k < kTrainWaves; ++k)
      v += sums[k][i];
    mine[i] = v;
  }
}

// Sum of entry i of `blocks` partial gradients, 16 slices of a 1024-thread block at a time in
// a fixed order; threads of slice 0 hold it (64 entries per block).
constexpr uint32_t kSumSlices = 16;
__device__ __forceinline__ float sum_partials(const float* __restrict__ partial, uint32_t blocks,
                                              uint32_t i)
{
  __shared__ float s[kSumSlices][64];
  const uint32_t c = threadIdx.x & 63u, slice = threadIdx.x >> 6;
  float v = 0.0f;
#pragma unroll 4
  for (uint32_t b = slice; b < blocks; b += kSumSlices)
    v += partial[(size_t)b * kMlpPartial + i];
  s[slice][c] = v;
  __syncthreads();
  if (slice == 0)
    for (uint32_t k = 1; k < kSumSlices; ++k)
      v += s[k][c];
  return v;
}

// The batch's gradient and squared-error sum.
__global__ __launch_bounds__(64 * kSumSlices) void k_mlp_sum(const float* __restrict__ partial, uint32_t blocks,
                                                             float* __restrict__ grad, float* __restrict__ loss)
{
  const uint32_t i = blockIdx.x * 64u + (threadIdx.x & 63u);  // kMlpPartial covers every i
  const float g = sum_partials(partial, blocks, i);
  if (threadIdx.x >= 64u)
    return;
  if (i < (uint32_t)kMlpParams)
    grad[i] = g;
  else if (i == (uint32_t)kMlpParams)
    loss[0] = g;
}

// Adam on the fp32 master parameters with the summed gradient, the bf16 operand copies of the
// parameters it moved, and the batch's squared errors added to loss: one launch.
__global__ __launch_bounds__(64 * kSumSlices) void k_mlp_update(const float* __restrict__ partial,
                                                                uint32_t blocks, float* __restrict__ p,
                                                                float* __restrict__ m1, float* __restrict__ m2,
                                                                float* __restrict__ loss, float lr, float b1,
                                                                float b2, float eps, float c1, float c2, MlpDev m)
{
  const uint32_t i = blockIdx.x * 64u + (threadIdx.x & 63u);
  const float g = sum_partials(partial, blocks, i);
  if (threadIdx.x >= 64u || i > (uint32_t)kMlpParams)
    return;
  if (i == (uint32_t)kMlpParams) {
    loss[0] += g;
    return;
  }
  const float a = b1 * m1[i] + (1.0f - b1) * g;
  const float v = b2 * m2[i] + (1.0f - b2) * g * g;
  m1[i] = a;
  m2[i] = v;
  const float q = p[i] - lr * (a / c1) / (sqrtf(v / c2) + eps);
  p[i] = q;
  if (i < (uint32_t)kMlpB1) {
    m.w1tMut[(i % 64u) * 16u + i / 64u] = f2bf(q);
  } else if (i >= (uint32_t)kMlpW2 && i < (uint32_t)kMlpB2) {
    const uint32_t k = (i - kMlpW2) / 64u, u = (i - kMlpW2) % 64u;
    m.w2tMut[u * 64u + k] = f2bf(q);
    m.w2Mut[k * 64u + u] = f2bf(q);
  }
}

// Rebuild the operand copies from the master parameters.
__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ p, MlpDev m)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 64u * 16u) {  // w1t[n][k], k padded
    const uint32_t nn = i / 16u, k = i % 16u;
    m.w1tMut[i] = k < 8u ? f2bf(p[kMlpW1 + k * 64u + nn]) : (short)0;
  }
  if (i < 64u * 64u) {
    const uint32_t a = i / 64u, b = i % 64u;
    m.w2tMut[i] = f2bf(p[kMlpW2 + b * 64u + a]);  // w2t[n = a][k = b]
    m.w2Mut[i] = f2bf(p[kMlpW2 + a * 64u + b]);   // w2[k = a][n = b]
  }
}

__global__ void k_zero(float* __restrict__ p, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = 0.0f;
}

__global__ void k_affine_perm(uint32_t* __restrict__ perm, uint32_t n, uint32_t a, uint32_t c)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    perm[i] = (uint32_t)(((uint64_t)a * i + c) % n);
}

inline uint32_t blocks_for(uint32_t n, uint32_t b) { return (n + b - 1u) / b; }

}  // namespace

void launch_mlp_forward(const float* feat, uint32_t n, const MlpDev& m, float* out, hipStream_t s,
                        float4* packed)
{
  if (n == 0)
    return;
  // at most four workgroups a CU: a wave's weights are loaded once for all its rows
  const uint32_t blocks = blocks_for(n, 16u * kFwdTiles * 4u);
  hipLaunchKernelGGL(k_mlp_forward, dim3(blocks < 1024u ? blocks : 1024u), dim3(256), 0, s, feat, n, m, out,
                     packed);
}

// One workgroup a CU at most, so the partial gradients stay few; small batches spread their
// tiles over as many workgroups as have four.
static uint32_t train_blocks(uint32_t n)
{
  const uint32_t b = blocks_for(n, 16u * kTrainWaves);
  return b < kMlpMaxBlocks ? b : kMlpMaxBlocks;
}

void launch_mlp_train(const float* feat, const float* target, const uint32_t* perm, uint32_t n,
                      const MlpDev& m, float* partial, hipStream_t s)
{
  if (n == 0)
    return;
  hipLaunchKernelGGL(k_mlp_train, dim3(train_blocks(n)), dim3(64 * kTrainWaves), 0, s, feat, target,
                     perm, n, 1.0f / (float)n, m, partial);
}

void launch_mlp_sum(const float* partial, uint32_t n, float* grad, float* loss, hipStream_t s)
{
  if (n == 0)
    return;
  hipLaunchKernelGGL(k_mlp_sum, dim3(kMlpPartial / 64), dim3(64 * kSumSlices), 0, s, partial,
                     train_blocks(n), grad, loss);
}

void launch_mlp_update(const float* partial, uint32_t n, float* p, float* m1, float* m2, float* loss,
                       float lr, int step, const MlpDev& m, hipStream_t s)
{
  if (n == 0)
    return;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_mlp_update, dim3(kMlpPartial / 64), dim3(64 * kSumSlices), 0, s, partial,
                     train_blocks(n), p, m1, m2, loss, lr, b1, b2, 1e-8f, c1, c2, m);
}

void launch_mlp_pack(const float* p, const MlpDev& m, hipStream_t s)
{
  hipLaunchKernelGGL(k_mlp_pack, dim3(blocks_for(64 * 64, 256)), dim3(256), 0, s, p, m);
}

void launch_zero(float* p, uint32_t n, hipStream_t s)
{
  if (n)
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, n);
}

void launch_affine_perm(uint32_t* perm, uint32_t n, uint32_t a, uint32_t c, hipStream_t s)
{
  if (n)
    hipLaunchKernelGGL(k_affine_perm, dim3(blocks_for(n, 256)), dim3(256), 0, s, perm, n, a, c);
}

}  // namespace rtp
