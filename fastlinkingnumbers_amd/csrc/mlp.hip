// Learned opening criterion: a 12-64-64-1 hard-swish MLP on matrix cores.
//
// The network predicts log10 of the far-field error of a node pair from 12
// dimensionless features (see mlp_features in bh.hip).  Parameters are FP32
// masters (W1[64x12] b1[64] W2[64x64] b2[64] w3[64] b3, 5,057 floats).  The
// activation is hard-swish, h(z) = z min(max(z/6 + 1/2, 0), 1): the
// logistic of SiLU costs two quarter-rate transcendental instructions per
// activation (2^x and a reciprocal), which bounded inference, while
// hard-swish is one packed FP16 FMA with the clamp bit and one packed
// multiply per two activations.
//
// Training: inputs normalised by the training mean/std, padded from 12 to 32
// features; every matrix product of the forward and backward pass runs on
// v_mfma_f32_16x16x32_bf16 tiles of 16 rows with FP32 accumulation, the
// biases, activations and output layer in FP32.  Inference (below) runs on
// FP16 operands, v_mfma_f32_16x16x32_f16.
//
// MFMA 16x16x32 fragments (one wave): lane l supplies A[l%16][8*(l/16)+j] and
// B[8*(l/16)+j][l%16] for j = 0..7 and receives C[4*(l/16)+i][l%16], i=0..3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>

#include "bh_types.h"
#include "flk_internal.h"
#include "mlp_infer.h"

namespace flk {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int H = 64;       // hidden width
constexpr int KP = 32;      // padded input width
constexpr int OFF_W1 = 0, OFF_B1 = 768, OFF_W2 = 832, OFF_B2 = 4928, OFF_W3 = 4992, OFF_B3 = 5056;

// Hard-swish in FP32 (training) and its derivative: 1/2 + z/3 on (-3, 3),
// 0 at and below -3, 1 at and above 3.
__device__ __forceinline__ float hswish(float z) {
  return z * fminf(fmaxf(fmaf(z, 1.0f / 6.0f, 0.5f), 0.f), 1.f);
}
__device__ __forceinline__ float dhswish(float z) {
  return z <= -3.f ? 0.f : (z < 3.f ? fmaf(z, 1.0f / 3.0f, 0.5f) : 1.f);
}

struct WaveLds {          // per-wave staging, bf16 row-major tiles of 16 rows
  __bf16 x[16][KP];
  __bf16 h1[16][H];
  __bf16 dz2[16][H];
  __bf16 dz1[16][H];
  float y[16];
  float dy[16];
};
struct BlockLds {
  __bf16 w1[H][KP];       // W1 padded, row = output neuron
  __bf16 w2[H][H];
  float b1[H], b2[H], w3[H];
  float b3;
  float mean[FLK_MLP_NFEAT], istd[FLK_MLP_NFEAT];
  WaveLds wv[4];
};

__device__ __forceinline__ bf16x8 a_frag(const __bf16 *m, int ld, int k0) {
  const int l = threadIdx.x & 63;
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = m[(l % 16) * ld + k0 + 8 * (l / 16) + j];
  return v;
}

// Loads the weights into LDS (bf16 copies are made here from FP32 masters),
// every global load of a thread in flight at once.  256 threads.
__device__ void load_weights(BlockLds &L, const float *__restrict__ P, const float *__restrict__ norm) {
  static_assert(FLK_MLP_NFEAT % 4 == 0 && FLK_MLP_NFEAT * H / 4 <= 256 && OFF_W2 % 4 == 0, "whole float4 rows");
  constexpr int kRow = FLK_MLP_NFEAT / 4;  // float4s of a row of W1
  const int t = threadIdx.x;
  const float4 *w1 = reinterpret_cast<const float4 *>(P + OFF_W1), *w2 = reinterpret_cast<const float4 *>(P + OFF_W2);
  float4 v2[H * H / 1024], v1{};
#pragma unroll
  for (int q = 0; q < H * H / 1024; ++q) v2[q] = w2[t + 256 * q];
  if (t < kRow * H) v1 = w1[t];
  // the biases and W3 (a thread each), and the normalisation
  const int j = t & (H - 1);
  const float b = t < H ? P[OFF_B1 + j] : t < 2 * H ? P[OFF_B2 + j] : t < 3 * H ? P[OFF_W3 + j] : t == 3 * H ? P[OFF_B3] : 0.f;
  const float nm = t < 2 * FLK_MLP_NFEAT ? norm[t] : 1.f;
#pragma unroll
  for (int q = 0; q < H * H / 1024; ++q) {
    __bf16 *d = &L.w2[0][0] + 4 * (t + 256 * q);
    d[0] = (__bf16)v2[q].x; d[1] = (__bf16)v2[q].y; d[2] = (__bf16)v2[q].z; d[3] = (__bf16)v2[q].w;
  }
  if (t < kRow * H) {
    __bf16 *d = &L.w1[t / kRow][4 * (t % kRow)];
    d[0] = (__bf16)v1.x; d[1] = (__bf16)v1.y; d[2] = (__bf16)v1.z; d[3] = (__bf16)v1.w;
  }
  for (int k = t; k < H * (KP - FLK_MLP_NFEAT); k += 256)
    L.w1[k / (KP - FLK_MLP_NFEAT)][FLK_MLP_NFEAT + k % (KP - FLK_MLP_NFEAT)] = (__bf16)0.0f;
  if (t < H) L.b1[j] = b;
  else if (t < 2 * H) L.b2[j] = b;
  else if (t < 3 * H) L.w3[j] = b;
  else if (t == 3 * H) L.b3 = b;
  if (t < FLK_MLP_NFEAT) L.mean[t] = nm;
  else if (t < 2 * FLK_MLP_NFEAT) L.istd[t - FLK_MLP_NFEAT] = 1.0f / nm;
  __syncthreads();
}

// Forward pass of 16 rows held in W.x: returns Z1, Z2 fragments (C layout,
// 4 column blocks) and writes W.h1 (bf16) and W.y.
__device__ void forward16(const BlockLds &L, WaveLds &W, f32x4 (&z1)[4], f32x4 (&z2)[4]) {
  const int l = threadIdx.x & 63;
  const bf16x8 ax = a_frag(&W.x[0][0], KP, 0);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    bf16x8 b;
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = L.w1[nb * 16 + l % 16][8 * (l / 16) + j];
    f32x4 acc = {0, 0, 0, 0};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ax, b, acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] += L.b1[nb * 16 + l % 16];
      W.h1[4 * (l / 16) + i][nb * 16 + l % 16] = (__bf16)hswish(acc[i]);
    }
    z1[nb] = acc;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const bf16x8 ah0 = a_frag(&W.h1[0][0], H, 0), ah1 = a_frag(&W.h1[0][0], H, 32);
  float part[4] = {0, 0, 0, 0};
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    bf16x8 b0, b1;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      b0[j] = L.w2[nb * 16 + l % 16][8 * (l / 16) + j];
      b1[j] = L.w2[nb * 16 + l % 16][32 + 8 * (l / 16) + j];
    }
    f32x4 acc = {0, 0, 0, 0};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah0, b0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah1, b1, acc, 0, 0, 0);
    const float w3 = L.w3[nb * 16 + l % 16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] += L.b2[nb * 16 + l % 16];
      part[i] += w3 * hswish(acc[i]);
    }
    z2[nb] = acc;
  }
  // output layer: sum the 64 columns (16 lanes x 4 blocks) of each row
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) part[i] += __shfl_xor(part[i], o, 64);
  }
  if (l % 16 == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) W.y[4 * (l / 16) + i] = part[i] + L.b3;
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// 16 rows of a wave: lane l holds features 3 (l / 16) to + 2 of row l % 16, and
// the row's target.
struct WaveRows {
  float x[3], t;
};
__device__ __forceinline__ WaveRows load_rows(const float *__restrict__ x, const float *__restrict__ t,
                                              const int64_t *__restrict__ idx, int64_t r0, int64_t n) {
  static_assert(FLK_MLP_NFEAT == 12, "three features a lane");
  const int l = threadIdx.x & 63;
  WaveRows v{{0.f, 0.f, 0.f}, 0.f};
  if (r0 + l % 16 < n) {
    const int64_t row = idx ? idx[r0 + l % 16] : r0 + l % 16;
    const float *p = x + row * FLK_MLP_NFEAT + 3 * (l / 16);
    v = WaveRows{{p[0], p[1], p[2]}, t[row]};
  }
  return v;
}

// Stages the rows (those at or past n are zero) normalised into W.x, whose
// columns past the features are zero already.
__device__ __forceinline__ void stage_x(const BlockLds &L, WaveLds &W, const WaveRows &v, int64_t r0, int64_t n) {
  const int l = threadIdx.x & 63, i0 = 3 * (l / 16);
  const bool live = r0 + l % 16 < n;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    W.x[l % 16][i0 + k] = (__bf16)(live ? (v.x[k] - L.mean[i0 + k]) * L.istd[i0 + k] : 0.f);
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

__global__ __launch_bounds__(256) void mlp_forward_kernel(const float *__restrict__ P,
                                                          const float *__restrict__ norm,
                                                          const float *__restrict__ x, int64_t n,
                                                          float *__restrict__ y) {
  __shared__ InferLds L;
  InferRegs R;
  load_infer(P, norm, R, L);
  const int l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t r0 = wave * 16; r0 < n; r0 += nwaves * 16) {
    const int64_t row = r0 + c;
    f16x8 bx;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int f = 8 * g + j;
      const float v =
          (row < n && f < FLK_MLP_NFEAT) ? (x[row * FLK_MLP_NFEAT + f] - L.mean[f]) * L.istd[f] : 0.f;
      bx[j] = (_Float16)v;
    }
    const float yv = infer_tile(RegWeights{R}, L, bx);
    if (g == 0 && row < n) y[row] = yv;
  }
}

// A block's sums: every gradient, then the squared error.
constexpr int kSums = FLK_MLP_NPARAM + 1;

// Forward + backward of the mean squared error over rows idx[0..n) (or 0..n):
// d(loss)/d(params) and the summed squared error, one set of kSums per block in
// `part`, the waves' added in LDS in order.  inv_n = 1 / total rows.
// Bound by latency (a wave has one to a few 16-row tiles): FP32 atomics of every
// wave on the 5,057 gradients took 56 us for 8,192 rows.
__global__ __launch_bounds__(256) void mlp_grad_kernel(const float *__restrict__ P,
                                                       const float *__restrict__ norm,
                                                       const float *__restrict__ x,
                                                       const float *__restrict__ t,
                                                       const int64_t *__restrict__ idx, int64_t n,
                                                       float inv_n, float *__restrict__ part) {
  __shared__ union {
    BlockLds L;
    float sums[2][kSums];
  } lds;
  BlockLds &L = lds.L;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  WaveLds &W = L.wv[w];
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  const int64_t row0 = ((int64_t)blockIdx.x * 4 + w) * 16;
  WaveRows rows = load_rows(x, t, idx, row0, n);  // in flight beside the weights
  for (int k = l; k < 16 * (KP - FLK_MLP_NFEAT); k += 64)
    W.x[k / (KP - FLK_MLP_NFEAT)][FLK_MLP_NFEAT + k % (KP - FLK_MLP_NFEAT)] = (__bf16)0.0f;
  load_weights(L, P, norm);
  // per-lane gradient accumulators in C layout
  f32x4 gW2[4][4], gW1[4];  // gW2[mb][nb]: rows mb*16.. (output j), cols nb*16.. (input k)
  for (int a = 0; a < 4; ++a) {
    gW1[a] = f32x4{0, 0, 0, 0};
    for (int b = 0; b < 4; ++b) gW2[a][b] = f32x4{0, 0, 0, 0};
  }
  float gb2[4] = {0, 0, 0, 0}, gw3[4] = {0, 0, 0, 0}, gb3 = 0, lsum = 0;
  float gb1v[4] = {0, 0, 0, 0};
  for (int64_t r0 = row0; r0 < n; r0 += nwaves * 16) {
    stage_x(L, W, rows, r0, n);
    const float target = rows.t;
    rows = load_rows(x, t, idx, r0 + nwaves * 16, n);
    f32x4 z1[4], z2[4];
    forward16(L, W, z1, z2);
    if (l < 16) {
      float dy = 0.f;
      if (r0 + l < n) {
        const float e = W.y[l] - target;
        lsum += e * e;
        dy = 2.0f * e * inv_n;
      }
      W.dy[l] = dy;
      gb3 += dy;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // dZ2 = dy w3 * h'(z2); dw3 += dy * h2; db2 += dZ2
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const int col = nb * 16 + l % 16;
      const float w3 = L.w3[col];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * (l / 16) + i;
        const float dy = W.dy[row];
        const float z = z2[nb][i];
        gw3[nb] += dy * hswish(z);
        const float d = dy * w3 * dhswish(z);
        gb2[nb] += d;
        W.dz2[row][col] = (__bf16)d;
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // dH1 = dZ2 W2 ; dZ1 = dH1 * h'(z1)
    {
      const bf16x8 a0 = a_frag(&W.dz2[0][0], H, 0), a1 = a_frag(&W.dz2[0][0], H, 32);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        bf16x8 b0, b1;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          b0[j] = L.w2[8 * (l / 16) + j][nb * 16 + l % 16];
          b1[j] = L.w2[32 + 8 * (l / 16) + j][nb * 16 + l % 16];
        }
        f32x4 acc = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float d = acc[i] * dhswish(z1[nb][i]);
          gb1v[nb] += d;
          W.dz1[4 * (l / 16) + i][nb * 16 + l % 16] = (__bf16)d;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // weight gradients over the 16 rows (K padded to 32 with zeros):
    // dW2[j][k] += sum_r dZ2[r][j] H1[r][k];  dW1[j][i] += sum_r dZ1[r][j] X[r][i]
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      bf16x8 a2, a1;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int r = 8 * (l / 16) + j;
        a2[j] = r < 16 ? W.dz2[r][mb * 16 + l % 16] : (__bf16)0.0f;
        a1[j] = r < 16 ? W.dz1[r][mb * 16 + l % 16] : (__bf16)0.0f;
      }
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        bf16x8 b;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int r = 8 * (l / 16) + j;
          b[j] = r < 16 ? W.h1[r][nb * 16 + l % 16] : (__bf16)0.0f;
        }
        gW2[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b, gW2[mb][nb], 0, 0, 0);
      }
      bf16x8 bx;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int r = 8 * (l / 16) + j;
        bx[j] = r < 16 ? W.x[r][l % 16] : (__bf16)0.0f;
      }
      gW1[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bx, gW1[mb], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  }
  // bias / w3 sums: reduce over the 4 row groups (lane bits 4,5)
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    gb2[nb] += __shfl_xor(gb2[nb], 16, 64);
    gb2[nb] += __shfl_xor(gb2[nb], 32, 64);
    gw3[nb] += __shfl_xor(gw3[nb], 16, 64);
    gw3[nb] += __shfl_xor(gw3[nb], 32, 64);
    gb1v[nb] += __shfl_xor(gb1v[nb], 16, 64);
    gb1v[nb] += __shfl_xor(gb1v[nb], 32, 64);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    gb3 += __shfl_xor(gb3, o, 64);
    lsum += __shfl_xor(lsum, o, 64);
  }
  // waves 0 and 1 write their sums, waves 2 and 3 add to them; C layout: row =
  // 4*(l/16)+i within block mb, col = l%16 within nb
  auto flush = [&](float *dst, auto put) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = mb * 16 + 4 * (l / 16) + i;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) put(dst[OFF_W2 + j * H + nb * 16 + l % 16], gW2[mb][nb][i]);
        if (l % 16 < FLK_MLP_NFEAT) put(dst[OFF_W1 + j * FLK_MLP_NFEAT + l % 16], gW1[mb][i]);
      }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
      if (l < 16) {
        put(dst[OFF_B2 + nb * 16 + l], gb2[nb]);
        put(dst[OFF_W3 + nb * 16 + l], gw3[nb]);
        put(dst[OFF_B1 + nb * 16 + l], gb1v[nb]);
      }
    if (l == 0) {
      put(dst[OFF_B3], gb3);
      put(dst[FLK_MLP_NPARAM], lsum);
    }
  };
  __syncthreads();
  if (w < 2) flush(lds.sums[w], [](float &d, float v) { d = v; });
  __syncthreads();
  if (w >= 2) flush(lds.sums[w - 2], [](float &d, float v) { d += v; });
  __syncthreads();
  for (int k = threadIdx.x; k < kSums; k += 256)
    part[(int64_t)blockIdx.x * kSums + k] = lds.sums[0][k] + lds.sums[1][k];
}

// The blocks' sums added, 64 parameters a block, a quarter of the sums a wave;
// then either the gradient itself (grad) or an Adam step (FP32 masters; m, v
// moments, zero before the first step; bias-corrected).  The squared error goes
// to, or with `more` is added to, *loss.
constexpr int kStepBlocks = (kSums + 63) / 64;
__global__ __launch_bounds__(256) void mlp_step_kernel(const float *__restrict__ part, int nparts,
                                                       float *__restrict__ grad, float *__restrict__ P,
                                                       float *__restrict__ m, float *__restrict__ v, int first,
                                                       float lr, float b1t, float b2t, float *__restrict__ loss,
                                                       int more) {
  __shared__ float sums[4][64];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, t = blockIdx.x * 64 + l;
  float s = 0.f;
  if (t < kSums) {
    const float *p = part + t;
    int k = w;
    for (; k + 28 < nparts; k += 32) {  // eight loads in flight
      float u[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) u[i] = p[(int64_t)(k + 4 * i) * kSums];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += u[i];
    }
    for (; k < nparts; k += 4) s += p[(int64_t)k * kSums];
  }
  sums[w][l] = s;
  __syncthreads();
  if (w || t >= kSums) return;
  const float g = (sums[0][l] + sums[1][l]) + (sums[2][l] + sums[3][l]);
  if (t == FLK_MLP_NPARAM) {
    *loss = more ? *loss + g : g;
  } else if (grad) {
    grad[t] = g;
  } else {
    const float b1 = 0.9f, b2 = 0.999f;
    const float mt = (first ? 0.f : b1 * m[t]) + (1 - b1) * g, vt = (first ? 0.f : b2 * v[t]) + (1 - b2) * g * g;
    m[t] = mt;
    v[t] = vt;
    const float mh = mt / (1 - b1t), vh = vt / (1 - b2t);
    P[t] -= lr * mh / (sqrtf(vh) + 1e-8f);
  }
}

// The level kernel's LDS image of the network, one wave.
__global__ __launch_bounds__(64) void mlp_pack_image(const float *__restrict__ P, const float *__restrict__ norm,
                                                     InferImage *__restrict__ img) {
  InferRegs R;
  load_infer(P, norm, R, img->L);
  infer_w_store(R, img->W);
}

}  // namespace

// ---------------------------------------------------------------- host side
// The weights from the host masters to the device, and the level kernel's
// image of them packed from those.
void mlp_upload(flk_ctx *ctx) {
  MlpState &M = ctx->mlp;
  if (!M.loaded) throw Error(FLK_ERR_STATE, "no MLP weights loaded (flk_mlp_set_weights)");
  M.d_params.reserve(sizeof(float) * FLK_MLP_NPARAM);
  M.d_norm.reserve(sizeof(float) * 2 * FLK_MLP_NFEAT);
  FLK_HIP(hipMemcpyAsync(M.d_params.ptr, M.params.data(), sizeof(float) * FLK_MLP_NPARAM,
                         hipMemcpyHostToDevice, ctx->stream));
  FLK_HIP(hipMemcpyAsync(M.d_norm.ptr, M.norm.data(), sizeof(float) * 2 * FLK_MLP_NFEAT,
                         hipMemcpyHostToDevice, ctx->stream));
  M.d_image.reserve(sizeof(InferImage));
  hipLaunchKernelGGL(mlp_pack_image, dim3(1), dim3(64), 0, ctx->stream, M.d_params.as<float>(),
                     M.d_norm.as<float>(), M.d_image.as<InferImage>());
  FLK_HIP(hipGetLastError());
}

void mlp_forward(flk_ctx *ctx, const float *x, int64_t n, float *y) {
  if (n <= 0) return;
  mlp_upload(ctx);
  hipStream_t s = ctx->stream;
  DevBuf dx, dy;
  dx.reserve(sizeof(float) * FLK_MLP_NFEAT * n);
  dy.reserve(sizeof(float) * n);
  FLK_HIP(hipMemcpyAsync(dx.ptr, x, sizeof(float) * FLK_MLP_NFEAT * n, hipMemcpyHostToDevice, s));
  const int blocks = (int)std::min<int64_t>((n + 63) / 64, 8 * std::max(1, ctx->num_cus));
  hipLaunchKernelGGL(mlp_forward_kernel, dim3(blocks), dim3(256), 0, s, ctx->mlp.d_params.as<float>(),
                     ctx->mlp.d_norm.as<float>(), dx.as<float>(), n, dy.as<float>());
  FLK_HIP(hipGetLastError());
  FLK_HIP(hipMemcpyAsync(y, dy.ptr, sizeof(float) * n, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
}

void mlp_forward_device(flk_ctx *ctx, const float *dx, int64_t n, float *dy) {
  const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n + 63) / 64, 8 * std::max(1, ctx->num_cus)));
  hipLaunchKernelGGL(mlp_forward_kernel, dim3(blocks), dim3(256), 0, ctx->stream,
                     ctx->mlp.d_params.as<float>(), ctx->mlp.d_norm.as<float>(), dx, n, dy);
  FLK_HIP(hipGetLastError());
}

namespace {

// Sets of more than this are given back after the call: their upload takes
// many times what allocating them does.
constexpr size_t kKeptBytes = size_t(64) << 20;
void give_back(MlpScratch &D) {
  for (DevBuf *b : {&D.x, &D.t, &D.idx})
    if (b->bytes > kKeptBytes) b->release();
}

// One set of gradients of the n rows at idx (or the first n): the blocks' sums
// into D.part; returns their number.  More blocks than are resident would add
// sets to read without adding waves.
int enqueue_gradient(flk_ctx *ctx, const float *x, const float *t, const int64_t *idx, int64_t n) {
  MlpScratch &D = ctx->mlp.scratch;
  const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n + 63) / 64, 2 * std::max(1, ctx->num_cus)));
  D.part.reserve(sizeof(float) * kSums * blocks);
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(blocks), dim3(256), 0, ctx->stream, ctx->mlp.d_params.as<float>(),
                     ctx->mlp.d_norm.as<float>(), x, t, idx, n, 1.0f / (float)std::max<int64_t>(n, 1),
                     D.part.as<float>());
  FLK_HIP(hipGetLastError());
  return blocks;
}

}  // namespace

float mlp_gradient(flk_ctx *ctx, const float *x, const float *y, int64_t n, float *grad) {
  mlp_upload(ctx);
  hipStream_t s = ctx->stream;
  MlpScratch &D = ctx->mlp.scratch;
  D.x.reserve(sizeof(float) * FLK_MLP_NFEAT * std::max<int64_t>(n, 1));
  D.t.reserve(sizeof(float) * std::max<int64_t>(n, 1));
  D.m.reserve(sizeof(float) * FLK_MLP_NPARAM);
  D.loss.reserve(sizeof(float));
  if (n) {
    FLK_HIP(hipMemcpyAsync(D.x.ptr, x, sizeof(float) * FLK_MLP_NFEAT * n, hipMemcpyHostToDevice, s));
    FLK_HIP(hipMemcpyAsync(D.t.ptr, y, sizeof(float) * n, hipMemcpyHostToDevice, s));
  }
  const int parts = enqueue_gradient(ctx, D.x.as<float>(), D.t.as<float>(), nullptr, n);
  hipLaunchKernelGGL(mlp_step_kernel, dim3(kStepBlocks), dim3(256), 0, s, (const float *)D.part.as<float>(), parts,
                     D.m.as<float>(), (float *)nullptr, (float *)nullptr, (float *)nullptr, 0, 0.f, 0.f, 0.f,
                     D.loss.as<float>(), 0);
  FLK_HIP(hipGetLastError());
  float loss = 0;
  FLK_HIP(hipMemcpyAsync(grad, D.m.ptr, sizeof(float) * FLK_MLP_NPARAM, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipMemcpyAsync(&loss, D.loss.ptr, sizeof(float), hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  give_back(D);
  return loss / (float)std::max<int64_t>(n, 1);
}

float mlp_train(flk_ctx *ctx, const float *x, const float *y, int64_t n, int epochs, int batch,
                float lr, uint64_t seed) {
  if (n <= 0 || epochs <= 0 || batch <= 0) throw Error(FLK_ERR_ARG, "empty training set");
  mlp_upload(ctx);
  hipStream_t s = ctx->stream;
  MlpScratch &D = ctx->mlp.scratch;
  D.x.reserve(sizeof(float) * FLK_MLP_NFEAT * n);
  D.t.reserve(sizeof(float) * n);
  D.m.reserve(sizeof(float) * FLK_MLP_NPARAM);
  D.v.reserve(sizeof(float) * FLK_MLP_NPARAM);
  D.loss.reserve(sizeof(float));
  D.idx.reserve(sizeof(int64_t) * n);
  FLK_HIP(hipMemcpyAsync(D.x.ptr, x, sizeof(float) * FLK_MLP_NFEAT * n, hipMemcpyHostToDevice, s));
  FLK_HIP(hipMemcpyAsync(D.t.ptr, y, sizeof(float) * n, hipMemcpyHostToDevice, s));
  std::vector<int64_t> perm(n);
  for (int64_t k = 0; k < n; ++k) perm[k] = k;
  std::mt19937_64 rng(seed);
  float b1t = 1.f, b2t = 1.f, last = 0.f;
  for (int e = 0; e < epochs; ++e) {
    for (int64_t k = n - 1; k > 0; --k) std::swap(perm[k], perm[rng() % (uint64_t)(k + 1)]);
    FLK_HIP(hipMemcpyAsync(D.idx.ptr, perm.data(), sizeof(int64_t) * n, hipMemcpyHostToDevice, s));
    for (int64_t b0 = 0; b0 < n; b0 += batch) {
      const int parts = enqueue_gradient(ctx, D.x.as<float>(), D.t.as<float>(), D.idx.as<int64_t>() + b0,
                                         std::min<int64_t>(batch, n - b0));
      b1t *= 0.9f;
      b2t *= 0.999f;
      hipLaunchKernelGGL(mlp_step_kernel, dim3(kStepBlocks), dim3(256), 0, s, (const float *)D.part.as<float>(),
                         parts, (float *)nullptr, ctx->mlp.d_params.as<float>(), D.m.as<float>(), D.v.as<float>(),
                         (int)(e == 0 && b0 == 0), lr, b1t, b2t, D.loss.as<float>(), (int)(b0 > 0));
      FLK_HIP(hipGetLastError());
    }
    FLK_HIP(hipMemcpyAsync(&last, D.loss.ptr, sizeof(float), hipMemcpyDeviceToHost, s));
    FLK_HIP(hipStreamSynchronize(s));
    last /= (float)n;
  }
  FLK_HIP(hipMemcpyAsync(ctx->mlp.params.data(), ctx->mlp.d_params.ptr, sizeof(float) * FLK_MLP_NPARAM,
                         hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  give_back(D);
  return last;
}

}  // namespace flk

#define FLK_GUARD(ctx, ...)                 \
  try {                                     \
    __VA_ARGS__                             \
  } catch (const flk::Error &e) {           \
    if (ctx) (ctx)->err = e.msg;            \
    return e.code;                          \
  } catch (const std::exception &e) {       \
    if (ctx) (ctx)->err = e.what();         \
    return FLK_ERR_STATE;                   \
  }

extern "C" {

int32_t flk_mlp_set_weights(flk_ctx *ctx, const float *params, const float *norm24) {
  if (!ctx || !params || !norm24) return FLK_ERR_ARG;
  for (int k = 0; k < FLK_MLP_NFEAT; ++k)
    if (!(norm24[FLK_MLP_NFEAT + k] > 0)) {
      ctx->err = "feature std must be positive";
      return FLK_ERR_ARG;
    }
  ctx->mlp.params.assign(params, params + FLK_MLP_NPARAM);
  ctx->mlp.norm.assign(norm24, norm24 + 2 * FLK_MLP_NFEAT);
  ctx->mlp.loaded = true;
  return FLK_OK;
}

int32_t flk_mlp_get_weights(const flk_ctx *ctx, float *params, float *norm24) {
  if (!ctx || !params || !norm24) return FLK_ERR_ARG;
  if (!ctx->mlp.loaded) return FLK_ERR_STATE;
  std::copy(ctx->mlp.params.begin(), ctx->mlp.params.end(), params);
  std::copy(ctx->mlp.norm.begin(), ctx->mlp.norm.end(), norm24);
  return FLK_OK;
}

int32_t flk_mlp_forward(flk_ctx *ctx, const float *x, int64_t n, float *y) {
  if (!ctx || n < 0 || (n > 0 && (!x || !y))) return FLK_ERR_ARG;
  FLK_GUARD(ctx, {
    FLK_HIP(hipSetDevice(ctx->device));
    flk::mlp_forward(ctx, x, n, y);
    return FLK_OK;
  })
}

int32_t flk_mlp_gradient(flk_ctx *ctx, const float *x, const float *y, int64_t n, float *grad,
                         float *loss) {
  if (!ctx || n < 0 || !grad || (n > 0 && (!x || !y))) return FLK_ERR_ARG;
  FLK_GUARD(ctx, {
    FLK_HIP(hipSetDevice(ctx->device));
    const float l = flk::mlp_gradient(ctx, x, y, n, grad);
    if (loss) *loss = l;
    return FLK_OK;
  })
}

int32_t flk_mlp_train(flk_ctx *ctx, const float *x, const float *y, int64_t n, int32_t epochs,
                      int32_t batch, float lr, uint64_t seed, float *final_loss) {
  if (!ctx || n <= 0 || !x || !y) return FLK_ERR_ARG;
  FLK_GUARD(ctx, {
    FLK_HIP(hipSetDevice(ctx->device));
    const float l = flk::mlp_train(ctx, x, y, n, epochs, batch, lr, seed);
    if (final_loss) *final_loss = l;
    return FLK_OK;
  })
}

int32_t flk_mlp_samples(flk_ctx *ctx, int32_t a, int32_t b, int64_t cap, uint64_t seed, float *x,
                        float *y, int64_t *count) {
  if (!ctx || !count || cap < 0 || (cap > 0 && (!x || !y))) return FLK_ERR_ARG;
  FLK_GUARD(ctx, {
    FLK_HIP(hipSetDevice(ctx->device));
    if (a < 0 || b < 0 || a >= ctx->curves.ncurves || b >= ctx->curves.ncurves)
      throw flk::Error(FLK_ERR_ARG, "curve index out of range");
    *count = flk::mlp_samples(ctx, a, b, cap, seed, x, y);
    return FLK_OK;
  })
}

}  // extern "C"
