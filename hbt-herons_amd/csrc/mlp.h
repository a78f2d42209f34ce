// Per-particle bound-set classifier for the learned warm start: an
// 8 -> 64 -> 64 -> 1 MLP with ReLU hidden layers and a logistic output.
// Parameters are kept as FP32 master weights for the optimiser and rounded to
// BF16 for every forward/backward pass (accumulation in FP32).
//
// Flat parameter layout: W1[64][8] | b1[64] | W2[64][64] | b2[64] | w3[64] | b3.
#pragma once
#include "common.h"

namespace hbtx
{
#define MLP_IN 8
#define MLP_H 64
#define MLP_OFF_W1 0
#define MLP_OFF_B1 (MLP_OFF_W1 + MLP_H * MLP_IN)
#define MLP_OFF_W2 (MLP_OFF_B1 + MLP_H)
#define MLP_OFF_B2 (MLP_OFF_W2 + MLP_H * MLP_H)
#define MLP_OFF_W3 (MLP_OFF_B2 + MLP_H)
#define MLP_OFF_B3 (MLP_OFF_W3 + MLP_H)
#define MLP_NPAR (MLP_OFF_B3 + 1)

// round-to-nearest-even FP32 -> BF16 bits
HBTX_HD uint16_t f32_to_bf16(float f)
{
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u)
    return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
HBTX_HD float bf16_to_f32(uint16_t b)
{
  return __uint_as_float((uint32_t)b << 16);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

HBTX_DEV __bf16 bf16_bits(uint16_t b)
{
  return __builtin_bit_cast(__bf16, b);
}

// Inference on the matrix cores (v_mfma_f32_32x32x16_bf16): one wave evaluates 32
// samples per step, neurons as matrix rows and samples as columns.
//   layer 1: H1^T[64 x 32] = W1[64 x 8] X^T, with X split into bf16 hi + lo parts
//            placed in the two K halves (so the product keeps FP32 accuracy);
//   layer 2: H2^T[64 x 32] = W2[64 x 64] relu(H1^T + b1), H1 again split hi + lo;
//   layer 3: z = w3 . relu(H2^T + b2) + b3 on the vector units.
// Lane l holds output column l % 32 and rows 8*(r/4) + 4*(l/32) + r%4 of a 32 x 32
// accumulator block (r = 0..15); a lane's layer-1 rows are exactly the K entries
// it supplies to layer 2, with the K order of both operands permuted alike.
// groups (may be null): the 32-particle groups to evaluate (particles 32 g .. 32 g + 31
// for g = groups[0 .. ngroups)); null evaluates every particle.
__global__ __launch_bounds__(256) void k_mlp_forward(const float *__restrict__ w, const uint16_t *__restrict__ wb,
                                                     const float *__restrict__ X, int64_t n,
                                                     float *__restrict__ logit, const int32_t *__restrict__ groups,
                                                     int64_t ngroups)
{
  const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
  bf16x8 a1[2];
  bf16x8 a2[2][4];
  float b1v[32], b2v[32], w3v[32];
#pragma unroll
  for (int mb = 0; mb < 2; mb++)
  {
    const int row = 32 * mb + c;
#pragma unroll
    for (int s = 0; s < 8; s++)
      a1[mb][s] = bf16_bits(wb[MLP_OFF_W1 + row * MLP_IN + s]);
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
      for (int s = 0; s < 8; s++)
        a2[mb][kb][s] = bf16_bits(wb[MLP_OFF_W2 + row * MLP_H + 8 * (2 * kb + s / 4) + 4 * h + (s & 3)]);
#pragma unroll
    for (int r = 0; r < 16; r++)
    {
      const int i = 32 * mb + 8 * (r / 4) + 4 * h + (r & 3);
      b1v[16 * mb + r] = w[MLP_OFF_B1 + i];
      b2v[16 * mb + r] = w[MLP_OFF_B2 + i];
      w3v[16 * mb + r] = w[MLP_OFF_W3 + i];
    }
  }
  const float b3 = w[MLP_OFF_B3];
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x / HBTX_WAVE) + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / HBTX_WAVE);
  const int64_t G = groups ? ngroups : (n + 31) / 32;
  for (int64_t gi = wave; gi < G; gi += nwaves)
  {
    const int64_t g = groups ? (int64_t)groups[gi] : gi;
    const int64_t j = g * 32 + c;
    float x[8];
    if (j < n)
    {
      const float4 u0 = reinterpret_cast<const float4 *>(X + j * MLP_IN)[0];
      const float4 u1 = reinterpret_cast<const float4 *>(X + j * MLP_IN)[1];
      x[0] = u0.x, x[1] = u0.y, x[2] = u0.z, x[3] = u0.w, x[4] = u1.x, x[5] = u1.y, x[6] = u1.z, x[7] = u1.w;
    }
    else
    {
#pragma unroll
      for (int s = 0; s < 8; s++)
        x[s] = 0.f;
    }
    bf16x8 bx;
#pragma unroll
    for (int s = 0; s < 8; s++)
    {
      const __bf16 hi = (__bf16)x[s];
      bx[s] = h ? (__bf16)(x[s] - (float)hi) : hi;
    }
    f32x16 zero;
#pragma unroll
    for (int r = 0; r < 16; r++)
      zero[r] = 0.f;
    bf16x8 bh[4], bl[4];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
    {
      const f32x16 d1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1[mb], bx, zero, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; r++)
      {
        const float v = fmaxf(d1[r] + b1v[16 * mb + r], 0.f);
        const int q = 4 * mb + r / 4, kb = q >> 1, s = 4 * (q & 1) + (r & 3);
        const __bf16 hi = (__bf16)v;
        bh[kb][s] = hi;
        bl[kb][s] = (__bf16)(v - (float)hi);
      }
    }
    float z = 0.f;
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
    {
      f32x16 d2 = zero;
#pragma unroll
      for (int kb = 0; kb < 4; kb++)
      {
        d2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2[mb][kb], bh[kb], d2, 0, 0, 0);
        d2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2[mb][kb], bl[kb], d2, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; r++)
        z += w3v[16 * mb + r] * fmaxf(d2[r] + b2v[16 * mb + r], 0.f);
    }
    z += __shfl_xor(z, 32, HBTX_WAVE);
    if (h == 0 && j < n)
      logit[j] = z + b3;
  }
}

inline int mlp_forward_blocks(int64_t n)
{
  const int64_t groups = (n + 31) / 32;
  return (int)std::max<int64_t>(1, std::min<int64_t>((groups + 3) / 4, 4096));
}

// Forward and backward of the network on the FP32 matrix instructions
// (v_mfma_f32_32x32x2_f32): a wave takes 32 samples at a time, neurons as matrix
// rows and samples as columns, as k_mlp_forward does, with every product and sum
// in FP32.
//   H1^T[64 x 32] = W1 X^T + b1,  H2^T = W2 relu(H1^T) + b2,  dH1^T = W2^T dH2^T:
//     a lane's accumulator rows are the K entries it supplies to the next product;
//   dW2[64 x 64] = dH2^T[64 x 32] H1[32 x 64],  dW1 = dH1^T X:  K is the sample, so
//     dH2, H1 and dH1 pass through the wave's own LDS to become operands.
// The weight gradients stay in the accumulators over all of a wave's samples, and a
// block's four waves add theirs in order at the end, so that a block leaves one
// partial gradient.  (One sample a lane on the vector units, a partial gradient per
// 128 samples: 1009 us for 400,000 samples, and 888 us to add 3126 partials.)
#define MLP_TILE 32
#define MLP_WAVES 4
#define MLP_BLOCK (MLP_WAVES * HBTX_WAVE)
#define MLP_LD (MLP_H + 1)
struct MlpLds
{
  float w2[MLP_H * MLP_LD];
  float w1[MLP_H * (MLP_IN + 1)];
  float b1[MLP_H], b2[MLP_H], w3[MLP_H];
  union
  {
    struct
    {
      float d[MLP_TILE * MLP_LD]; // dH2, then dH1: [sample][neuron]
      float h[MLP_TILE * MLP_LD]; // H1
      float x[MLP_TILE * (MLP_IN + 1)];
    } wave[MLP_WAVES];
    float grad[MLP_NPAR + 3]; // the block's sum, once every sample is done
  };
  double loss[MLP_WAVES];
};

__global__ __launch_bounds__(MLP_BLOCK, 1) void k_mlp_grad(const float *__restrict__ w, const float *__restrict__ X,
                                                           const uint8_t *__restrict__ y,
                                                           const int32_t *__restrict__ idx, int64_t nbatch,
                                                           float inv_batch, float *__restrict__ partial,
                                                           double *__restrict__ loss_partial)
{
  __shared__ MlpLds L;
  const int tid = threadIdx.x, wv = uniform(tid / HBTX_WAVE), lane = lane_id(), h = lane >> 5, c = lane & 31;
  for (int i = tid; i < MLP_H * MLP_H; i += MLP_BLOCK)
    L.w2[(i / MLP_H) * MLP_LD + i % MLP_H] = w[MLP_OFF_W2 + i];
  for (int i = tid; i < MLP_H * MLP_IN; i += MLP_BLOCK)
    L.w1[(i / MLP_IN) * (MLP_IN + 1) + i % MLP_IN] = w[MLP_OFF_W1 + i];
  for (int i = tid; i < MLP_H; i += MLP_BLOCK)
  {
    L.b1[i] = w[MLP_OFF_B1 + i];
    L.b2[i] = w[MLP_OFF_B2 + i];
    L.w3[i] = w[MLP_OFF_W3 + i];
  }
  const float b3 = w[MLP_OFF_B3];
  __syncthreads();
  auto &T = L.wave[wv];
  // accumulator register r of row block mb: neuron (row) 32 mb + 8 (r / 4) + 4 h + r % 4
  auto row = [&](int mb, int r) { return 32 * mb + 8 * (r / 4) + 4 * h + (r & 3); };
  f32x16 gw2[2][2], gw1[2];
  float gw3[2][16], gb2[2] = {0.f, 0.f}, gb1[2] = {0.f, 0.f}, gb3 = 0.f;
  double loss = 0.0;
#pragma unroll
  for (int mb = 0; mb < 2; mb++)
#pragma unroll
    for (int r = 0; r < 16; r++)
    {
      gw2[mb][0][r] = gw2[mb][1][r] = gw1[mb][r] = 0.f;
      gw3[mb][r] = 0.f;
    }
  const int64_t ntile = (nbatch + MLP_TILE - 1) / MLP_TILE;
  for (int64_t t = (int64_t)blockIdx.x * MLP_WAVES + wv; t < ntile; t += (int64_t)gridDim.x * MLP_WAVES)
  {
    const int64_t k = t * MLP_TILE + c;
    const bool valid = k < nbatch;
    const int64_t at = valid ? (idx ? (int64_t)idx[k] : k) : 0;
    float x[MLP_IN];
    {
      const float4 u0 = reinterpret_cast<const float4 *>(X + at * MLP_IN)[0];
      const float4 u1 = reinterpret_cast<const float4 *>(X + at * MLP_IN)[1];
      const float xs[MLP_IN] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int f = 0; f < MLP_IN; f++)
        x[f] = valid ? xs[f] : 0.f;
    }
    const float yy = valid ? (float)y[at] : 0.f;
    f32x16 h1[2], h2[2];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
    {
#pragma unroll
      for (int r = 0; r < 16; r++)
        h1[mb][r] = L.b1[row(mb, r)];
#pragma unroll
      for (int s = 0; s < MLP_IN / 2; s++)
        h1[mb] = __builtin_amdgcn_mfma_f32_32x32x2f32(L.w1[(32 * mb + c) * (MLP_IN + 1) + 2 * s + h],
                                                      h ? x[2 * s + 1] : x[2 * s], h1[mb], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; r++)
      {
        h1[mb][r] = fmaxf(h1[mb][r], 0.f);
        h2[mb][r] = L.b2[row(mb, r)];
      }
    }
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
          h2[mb] = __builtin_amdgcn_mfma_f32_32x32x2f32(L.w2[(32 * mb + c) * MLP_LD + row(kb, r)], h1[kb][r], h2[mb],
                                                        0, 0, 0);
    float z = 0.f;
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
      {
        h2[mb][r] = fmaxf(h2[mb][r], 0.f);
        z += L.w3[row(mb, r)] * h2[mb][r];
      }
    z += __shfl_xor(z, 32, HBTX_WAVE);
    z += b3;
    const float sig = 1.f / (1.f + __expf(-z));
    const float dz = valid ? (sig - yy) * inv_batch : 0.f;
    // binary cross-entropy with logits: softplus(z) - y z (a sample's two lanes hold the same)
    if (valid && h == 0)
    {
      loss += (double)(fmaxf(z, 0.f) + log1pf(__expf(-fabsf(z))) - yy * z);
      gb3 += dz;
    }
    f32x16 d1[2];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
      {
        const int j = row(mb, r);
        gw3[mb][r] += dz * h2[mb][r];
        h2[mb][r] = (h2[mb][r] > 0.f) ? dz * L.w3[j] : 0.f; // dH2 from here on
        d1[mb][r] = 0.f;
        T.d[c * MLP_LD + j] = h2[mb][r];
        T.h[c * MLP_LD + j] = h1[mb][r];
      }
    if (h == 0)
#pragma unroll
      for (int f = 0; f < MLP_IN; f++)
        T.x[c * (MLP_IN + 1) + f] = x[f];
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
          d1[mb] = __builtin_amdgcn_mfma_f32_32x32x2f32(L.w2[row(kb, r) * MLP_LD + 32 * mb + c], h2[kb][r], d1[mb],
                                                        0, 0, 0);
    wave_lds_sync();
#pragma unroll
    for (int s2 = 0; s2 < MLP_TILE / 2; s2++)
    {
      const int s = 2 * s2 + h;
      const float a0 = T.d[s * MLP_LD + c], a1 = T.d[s * MLP_LD + 32 + c];
      const float e0 = T.h[s * MLP_LD + c], e1 = T.h[s * MLP_LD + 32 + c];
      gb2[0] += a0;
      gb2[1] += a1;
      gw2[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, e0, gw2[0][0], 0, 0, 0);
      gw2[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, e1, gw2[0][1], 0, 0, 0);
      gw2[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, e0, gw2[1][0], 0, 0, 0);
      gw2[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, e1, gw2[1][1], 0, 0, 0);
    }
    wave_lds_sync();
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        T.d[c * MLP_LD + row(mb, r)] = (h1[mb][r] > 0.f) ? d1[mb][r] : 0.f;
    wave_lds_sync();
#pragma unroll
    for (int s2 = 0; s2 < MLP_TILE / 2; s2++)
    {
      const int s = 2 * s2 + h;
      const float a0 = T.d[s * MLP_LD + c], a1 = T.d[s * MLP_LD + 32 + c];
      const float e = (c < MLP_IN) ? T.x[s * (MLP_IN + 1) + min(c, MLP_IN)] : 0.f;
      gb1[0] += a0;
      gb1[1] += a1;
      gw1[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, e, gw1[0], 0, 0, 0);
      gw1[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, e, gw1[1], 0, 0, 0);
    }
    wave_lds_sync(); // the next samples' rows go where these were read
  }
  // sums over the lanes that share a value
#pragma unroll
  for (int mb = 0; mb < 2; mb++)
  {
    gb2[mb] += __shfl_xor(gb2[mb], 32, HBTX_WAVE);
    gb1[mb] += __shfl_xor(gb1[mb], 32, HBTX_WAVE);
#pragma unroll
    for (int r = 0; r < 16; r++)
#pragma unroll
      for (int d = 1; d < 32; d <<= 1)
        gw3[mb][r] += __shfl_xor(gw3[mb][r], d, HBTX_WAVE);
  }
#pragma unroll
  for (int d = 1; d < HBTX_WAVE; d <<= 1)
  {
    gb3 += __shfl_xor(gb3, d, HBTX_WAVE);
    loss += __shfl_xor(loss, d, HBTX_WAVE);
  }
  if (lane == 0)
    L.loss[wv] = loss;
  __syncthreads(); // (the waves' tiles are done: their LDS becomes the block's sum)
  for (int q = tid; q < MLP_NPAR; q += MLP_BLOCK)
    L.grad[q] = 0.f;
  for (int k = 0; k < MLP_WAVES; k++)
  {
    __syncthreads();
    if (wv != k)
      continue;
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
    {
#pragma unroll
      for (int r = 0; r < 16; r++)
      {
        const int j = row(mb, r);
        L.grad[MLP_OFF_W2 + j * MLP_H + c] += gw2[mb][0][r];
        L.grad[MLP_OFF_W2 + j * MLP_H + 32 + c] += gw2[mb][1][r];
        if (c < MLP_IN)
          L.grad[MLP_OFF_W1 + j * MLP_IN + c] += gw1[mb][r];
        if (c == 0)
          L.grad[MLP_OFF_W3 + j] += gw3[mb][r];
      }
      if (h == 0)
      {
        L.grad[MLP_OFF_B2 + 32 * mb + c] += gb2[mb];
        L.grad[MLP_OFF_B1 + 32 * mb + c] += gb1[mb];
      }
    }
    if (lane == 0)
      L.grad[MLP_OFF_B3] += gb3;
  }
  __syncthreads();
  for (int q = tid; q < MLP_NPAR; q += MLP_BLOCK)
    partial[(int64_t)blockIdx.x * MLP_NPAR + q] = L.grad[q];
  if (tid == 0)
  {
    double l = 0.0;
    for (int k = 0; k < MLP_WAVES; k++)
      l += L.loss[k];
    loss_partial[blockIdx.x] = l;
  }
}

// Blocks of the gradient: one a CU, no more than there are samples for.
inline int mlp_grad_blocks(int64_t nbatch, int num_cu)
{
  const int64_t tiles = (nbatch + MLP_TILE - 1) / MLP_TILE;
  return (int)std::max<int64_t>(1, std::min<int64_t>(num_cu, (tiles + MLP_WAVES - 1) / MLP_WAVES));
}

// Sum of the block partials in a fixed order: a block takes 64 parameters, each of
// its four waves a quarter of the partials, eight loads at a time.
__global__ __launch_bounds__(256) void k_mlp_reduce(const float *__restrict__ partial, int nblocks,
                                                    float *__restrict__ grad, const double *__restrict__ loss_partial,
                                                    double *__restrict__ loss)
{
  __shared__ float part[4][HBTX_WAVE];
  const int g = threadIdx.x / HBTX_WAVE, lane = lane_id();
  const int q = blockIdx.x * HBTX_WAVE + lane;
  const int b0 = nblocks * g / 4, b1 = nblocks * (g + 1) / 4;
  float acc = 0.f;
  if (q < MLP_NPAR)
  {
    int b = b0;
    for (; b + 8 <= b1; b += 8)
    {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; k++)
        v[k] = partial[(int64_t)(b + k) * MLP_NPAR + q];
#pragma unroll
      for (int k = 0; k < 8; k++)
        acc += v[k];
    }
    for (; b < b1; b++)
      acc += partial[(int64_t)b * MLP_NPAR + q];
  }
  part[g][lane] = acc;
  __syncthreads();
  if (g == 0 && q < MLP_NPAR)
    grad[q] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
  if (blockIdx.x == 0 && g == 1)
  {
    double l = 0.0;
    for (int b = lane; b < nblocks; b += HBTX_WAVE)
      l += loss_partial[b];
#pragma unroll
    for (int d = 1; d < HBTX_WAVE; d <<= 1)
      l += __shfl_xor(l, d, HBTX_WAVE);
    if (lane == 0)
      *loss = l;
  }
}

// Adam step on the FP32 master weights, then the BF16 working copy.
__global__ void k_mlp_adam(float *__restrict__ master, float *__restrict__ m, float *__restrict__ v,
                           const float *__restrict__ grad, float *__restrict__ wf, uint16_t *__restrict__ wb, float lr,
                           float b1, float b2, float eps, float c1, float c2)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= MLP_NPAR)
    return;
  const float g = grad[q];
  const float mq = b1 * m[q] + (1.f - b1) * g;
  const float vq = b2 * v[q] + (1.f - b2) * g * g;
  m[q] = mq;
  v[q] = vq;
  const float w = master[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
  master[q] = w;
  const uint16_t b = f32_to_bf16(w);
  wb[q] = b;
  wf[q] = bf16_to_f32(b);
}

__global__ void k_mlp_round(const float *__restrict__ master, float *__restrict__ wf, uint16_t *__restrict__ wb)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= MLP_NPAR)
    return;
  const uint16_t b = f32_to_bf16(master[q]);
  wb[q] = b;
  wf[q] = bf16_to_f32(b);
}

} // namespace hbtx
