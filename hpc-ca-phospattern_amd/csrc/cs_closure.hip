/*
 * cs_closure.hip -- training and inference of the learned closure's
 * network (cs_mlp_*): forward and backward passes on bfloat16 matrix-core
 * products with FP32 accumulation, fixed-order gradient reductions, Adam.
 *
 * The reference has no learned part.  The network corrects the
 * coarse-grid calcium that channel gating reads (evaluate_RyR_
 * stochastically, boundaryfluxes.c:295-359, reads the cleft voxel's
 * concentration); its inputs and labels come from paired fine/coarse
 * runs of the same dyads, and its use inside an ensemble's gating step
 * lives in cs_batch.hip.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <vector>

#include "csparks.h"
#include "cs_device.h"
#include "cs_mlp.h"

namespace {

constexpr int LROW = 40;                   /* LDS row of 32 samples, padded */
constexpr uint64_t IDX_CHUNK = 1u << 22;   /* indices staged in pinned memory at a time */
constexpr int UPD_GROUPS = 16;             /* wavefronts of a k_mlp_update block */

/* FP32 master parameters -> the device image: pre-permuted bfloat16
 * operands of both layers, biases, bfloat16-rounded output weights.  One
 * block; thread k fills element k of the image. */
__global__ void __launch_bounds__(256) k_mlp_pack(const float* __restrict__ p, MlpDev* __restrict__ P)
{
  for (int k = threadIdx.x; k < NSEG * 64 * 8; k += blockDim.x) {
    const int seg = k / 512, lane = (k / 8) % 64, j = k % 8, g = lane / 32, l = lane % 32;
    float w;
    if (seg < SEG_L2F) {
      const int m = (seg - SEG_L1) / 2, c = (seg - SEG_L1) % 2;
      w = p[MLP_OFF_W1 + (16 * c + 8 * g + j) * MLP_H + 32 * m + l];
    } else if (seg < SEG_L2B) {
      const int s = seg - SEG_L2F, m = s / 4, mb = (s / 2) % 2, q = s % 2;
      w = p[MLP_OFF_W2 + (32 * mb + mlp_feat(g, 8 * q + j)) * MLP_H + 32 * m + l];
    } else {
      const int s = seg - SEG_L2B, mi = s / 4, mo = (s / 2) % 2, q = s % 2;
      w = p[MLP_OFF_W2 + (32 * mi + l) * MLP_H + 32 * mo + mlp_feat(g, 8 * q + j)];
    }
    P->opnd[seg][lane][j] = __builtin_bit_cast(uint16_t, to_bf16(w));
  }
  for (int k = threadIdx.x; k < MLP_H; k += blockDim.x) {
    P->b1[k] = p[MLP_OFF_B1 + k];
    P->b2[k] = p[MLP_OFF_B2 + k];
    P->w3[k] = (float)to_bf16(p[MLP_OFF_W3 + k]);
  }
  if (threadIdx.x == 0) P->b3 = p[MLP_OFF_B3];
}

/* Normalised FP32 inputs [n][30] -> bfloat16 rows [n][32] (zero padded). */
__global__ void k_mlp_to_bf16(const float* __restrict__ x, uint64_t n, uint16_t* __restrict__ xb)
{
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n * MLP_PAD;
       k += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t s = k / MLP_PAD;
    const int f = (int)(k % MLP_PAD);
    xb[k] = __builtin_bit_cast(uint16_t, to_bf16(f < MLP_IN ? x[s * MLP_IN + f] : 0.0f));
  }
}

/* B operands of input chunk c for sample s of a bfloat16 row array. */
__device__ inline void load_x(const uint16_t* __restrict__ xb, uint64_t s, bool valid, bf16x8 (&x)[2])
{
  const int g = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int c = 0; c < 2; c++) {
    if (valid) x[c] = *reinterpret_cast<const bf16x8*>(xb + s * MLP_PAD + 16 * c + 8 * g);
    else
#pragma unroll
      for (int j = 0; j < 8; j++) x[c][j] = to_bf16(0.0f);
  }
}

/* Inference: y[s] for n samples of bfloat16 rows, 32 per wavefront. */
__global__ void __launch_bounds__(256)
k_mlp_forward(const MlpDev* __restrict__ P, const uint16_t* __restrict__ xb, uint64_t n, float* __restrict__ y)
{
  const int lane = threadIdx.x & 63;
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / 64);
  const uint64_t w0 = (uint64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  for (uint64_t t = w0; t * 32 < n; t += waves) {
    /* reload the weights every round instead of holding them all in
     * registers across the loop */
    asm volatile("" ::: "memory");
    const uint64_t s = t * 32 + (lane & 31);
    bf16x8 x[2];
    load_x(xb, s, s < n, x);
    f32x16 z1[2], z2[2];
    bf16x8 h1b[2][2];
    const float out = mlp_forward(P, [&](int seg) { return mlp_opnd(P, seg, lane); }, x, z1, z2, h1b,
                                  [](int, int, float) {});
    if (lane < 32 && s < n) y[s] = out;
  }
}

/* Forward and backward passes over n samples (rows idx[k] of xb when idx
 * is given, else rows k), 32 samples to a block, writing each block's
 * gradient of L = sum (y - t)^2 / norm into part[block][MLP_NPARAM] and its
 * sum of squared errors into sse[block].
 *
 * Two wavefronts share the samples: wavefront m owns features 32 m .. 32 m
 * + 31 of either layer, as mlp_forward's block m, and hands the other its
 * bfloat16 layer outputs and back-propagated gradients through LDS; the
 * output sum runs through block 0 and then block 1, so every sum keeps
 * mlp_forward's order.  The weight gradients are products over the 32
 * samples, formed on the matrix cores from activations and gradients
 * transposed through LDS.
 *
 * A training batch of 2048 is 64 blocks of one round, so the length of one
 * wavefront's chain of GELU arithmetic and loads is the time: half of it
 * each, the weight operands and tables loaded once into registers at the
 * start instead of through LDS, and each layer's pre-activations kept, so
 * GELU and its derivative share the error function.  A batch of 2048 takes
 * 8.2 us, where one wavefront per 32 samples took 19.0; 200001 samples 75
 * and 99 us. */
__global__ void __launch_bounds__(128)
k_mlp_grad(const MlpDev* __restrict__ P, const uint16_t* __restrict__ xb, const float* __restrict__ tv,
           const uint32_t* __restrict__ idx, uint64_t n, float norm, float* __restrict__ part,
           double* __restrict__ sse)
{
  /* x, h1, h2, g_z2, g_z1 as [feature][sample] bfloat16; g_y per sample */
  __shared__ alignas(16) uint16_t Lx[MLP_PAD][LROW];
  __shared__ alignas(16) uint16_t Lh1[MLP_H][LROW];
  __shared__ alignas(16) uint16_t Lh2[MLP_H][LROW];
  __shared__ alignas(16) uint16_t Lz2[MLP_H][LROW];
  __shared__ alignas(16) uint16_t Lz1[MLP_H][LROW];
  __shared__ bf16x8 Lop[2][2][64];   /* operands in register order: [block][chunk][lane] */
  __shared__ float Lgy[32], Ly[32], Lpart[64];
  const int lane = threadIdx.x & 63, m = threadIdx.x >> 6, g = lane >> 5, l = lane & 31;
  const uint64_t blocks = gridDim.x, wid = blockIdx.x, tiles = (n + 31) / 32;

  bf16x8 w1[2], w2f[2][2], w2b[2][2];
#pragma unroll
  for (int c = 0; c < 2; c++) w1[c] = mlp_opnd(P, SEG_L1 + 2 * m + c, lane);
#pragma unroll
  for (int o = 0; o < 2; o++)
#pragma unroll
    for (int q = 0; q < 2; q++) {
      w2f[o][q] = mlp_opnd(P, SEG_L2F + 4 * m + 2 * o + q, lane);
      w2b[o][q] = mlp_opnd(P, SEG_L2B + 4 * m + 2 * o + q, lane);
    }
  float b1[16], b2[16], w3[16];
  feat_vec(P->b1, m, g, b1);
  feat_vec(P->b2, m, g, b2);
  feat_vec(P->w3, m, g, w3);
  const float b3 = P->b3;

  f32x16 gw1 = f32x16{}, gw2[2] = {f32x16{}, f32x16{}};
  float gb1 = 0.0f, gb2 = 0.0f, gw3 = 0.0f, gb3 = 0.0f;
  double err2 = 0.0;

  for (uint64_t t = wid; t < tiles; t += blocks) {
    const uint64_t k = t * 32 + l;
    const bool valid = k < n;
    const uint64_t s = valid ? (idx ? (uint64_t)idx[k] : k) : 0;
    bf16x8 x[2];
    load_x(xb, s, valid, x);
    const float target = tv[s];
    /* layer 1 */
    f32x16 z1;
#pragma unroll
    for (int r = 0; r < 16; r++) z1[r] = b1[r];
#pragma unroll
    for (int c = 0; c < 2; c++) z1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1[c], x[c], z1, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 2; q++) {
      bf16x8 h;
#pragma unroll
      for (int j = 0; j < 8; j++) h[j] = to_bf16(mlp_gelu(z1[8 * q + j]));
      Lop[m][q][lane] = h;
#pragma unroll
      for (int j = 0; j < 8; j++) Lh1[32 * m + mlp_feat(g, 8 * q + j)][l] = bf16_bits(h, j);
    }
    /* x for the weight gradients, a chunk to each wavefront */
#pragma unroll
    for (int j = 0; j < 8; j++) Lx[16 * m + 8 * g + j][l] = bf16_bits(m ? x[1] : x[0], j);
    __syncthreads();
    /* layer 2 and the output */
    f32x16 z2;
#pragma unroll
    for (int r = 0; r < 16; r++) z2[r] = b2[r];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
      for (int q = 0; q < 2; q++)
        z2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w2f[mb][q], Lop[mb][q][lane], z2, 0, 0, 0);
    float h2[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const __bf16 h = to_bf16(mlp_gelu(z2[r]));
      Lh2[32 * m + mlp_feat(g, r)][l] = __builtin_bit_cast(uint16_t, h);
      h2[r] = (float)h;
    }
    if (m == 0) {
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; r++) sum += w3[r] * h2[r];
      Lpart[lane] = sum;
    }
    __syncthreads();
    if (m == 1) {
      float sum = Lpart[lane];
#pragma unroll
      for (int r = 0; r < 16; r++) sum += w3[r] * h2[r];
      const float y = sum + __shfl_xor(sum, 32, 64) + b3;
      if (g == 0) Ly[l] = y;
    }
    __syncthreads();
    const float y = Ly[l];
    const float gy = valid ? 2.0f * (y - target) / norm : 0.0f;
    if (m == 0 && g == 0) {
      Lgy[l] = gy;
      gb3 += gy;
      if (valid) err2 += (double)(y - target) * (double)(y - target);
    }
    /* g_z2 = w3 g_y gelu'(z2), bfloat16 */
#pragma unroll
    for (int q = 0; q < 2; q++) {
      bf16x8 h;
#pragma unroll
      for (int j = 0; j < 8; j++) h[j] = to_bf16(w3[8 * q + j] * gy * mlp_gelu_grad(z2[8 * q + j]));
      Lop[m][q][lane] = h;
#pragma unroll
      for (int j = 0; j < 8; j++) Lz2[32 * m + mlp_feat(g, 8 * q + j)][l] = bf16_bits(h, j);
    }
    __syncthreads();
    /* g_h1 = W2 g_z2 on the matrix cores, then g_z1 = g_h1 gelu'(z1) */
    f32x16 gh1 = f32x16{};
#pragma unroll
    for (int mo = 0; mo < 2; mo++)
#pragma unroll
      for (int q = 0; q < 2; q++)
        gh1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w2b[mo][q], Lop[mo][q][lane], gh1, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; r++)
      Lz1[32 * m + mlp_feat(g, r)][l] = __builtin_bit_cast(uint16_t, to_bf16(gh1[r] * mlp_gelu_grad(z1[r])));
    __syncthreads();
    /* dW^T[o][i] += sum over the round's samples of g_z[o][s] a[i][s] */
    auto row = [&](const uint16_t (*L)[LROW], int r, int c) {
      return *reinterpret_cast<const bf16x8*>(&L[r][16 * c + 8 * g]);
    };
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const bf16x8 az2 = row(Lz2, 32 * m + l, c);
#pragma unroll
      for (int mi = 0; mi < 2; mi++)
        gw2[mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(az2, row(Lh1, 32 * mi + l, c), gw2[mi], 0, 0, 0);
      gw1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row(Lz1, 32 * m + l, c), row(Lx, l, c), gw1, 0, 0, 0);
    }
    /* lane f: bias gradients (wavefront 0) and the output weight's gradient
     * (wavefront 1) of feature f */
    auto at = [](const uint16_t (*L)[LROW], int f, int j) { return (float)__builtin_bit_cast(__bf16, L[f][j]); };
    float s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    if (m == 0) {
#pragma unroll 8
      for (int j = 0; j < 32; j++) {
        s1 += at(Lz1, lane, j);
        s2 += at(Lz2, lane, j);
      }
    } else {
#pragma unroll 8
      for (int j = 0; j < 32; j++) s3 += at(Lh2, lane, j) * Lgy[j];
    }
    gb1 += s1;
    gb2 += s2;
    gw3 += s3;
    __syncthreads();   /* reads done before the next round writes */
  }

  /* this block's gradient, in the packed parameter order */
  float* o = part + wid * (uint64_t)MLP_NPARAM;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int of = 32 * m + mlp_feat(g, r);
    o[MLP_OFF_W1 + l * MLP_H + of] = gw1[r];
#pragma unroll
    for (int mi = 0; mi < 2; mi++) o[MLP_OFF_W2 + (32 * mi + l) * MLP_H + of] = gw2[mi][r];
  }
  if (m == 1) {
    o[MLP_OFF_W3 + lane] = gw3;
    return;
  }
  o[MLP_OFF_B1 + lane] = gb1;
  o[MLP_OFF_B2 + lane] = gb2;
  for (int off = 16; off > 0; off >>= 1) {
    gb3 += __shfl_xor(gb3, off, 64);
    err2 += __shfl_xor(err2, off, 64);
  }
  if (lane == 0) {
    o[MLP_OFF_B3] = gb3;
    sse[wid] = err2;
  }
}

/* Parameter k's places in the operand image (the inverse of k_mlp_pack's
 * gather): one element for layer 1, a forward and a backward one for layer
 * 2, the tables for the rest. */
__device__ inline void pack_one(MlpDev* __restrict__ P, int k, float w)
{
  const uint16_t b = __builtin_bit_cast(uint16_t, to_bf16(w));
  /* lane group and register of feature f of a 32-block: mlp_feat(g, r) = f */
  auto group = [](int f) { return (f / 4) % 2; };
  auto reg = [](int f) { return 4 * (f / 8) + f % 4; };
  if (k < MLP_OFF_B1) {
    const int i = k / MLP_H, f = k % MLP_H;
    P->opnd[SEG_L1 + 2 * (f / 32) + i / 16][32 * ((i / 8) % 2) + f % 32][i % 8] = b;
  } else if (k < MLP_OFF_W2) {
    P->b1[k - MLP_OFF_B1] = w;
  } else if (k < MLP_OFF_B2) {
    const int i = (k - MLP_OFF_W2) / MLP_H, o = (k - MLP_OFF_W2) % MLP_H;
    const int ri = reg(i % 32), ro = reg(o % 32);
    P->opnd[SEG_L2F + 4 * (o / 32) + 2 * (i / 32) + ri / 8][32 * group(i % 32) + o % 32][ri % 8] = b;
    P->opnd[SEG_L2B + 4 * (i / 32) + 2 * (o / 32) + ro / 8][32 * group(o % 32) + i % 32][ro % 8] = b;
  } else if (k < MLP_OFF_W3) {
    P->b2[k - MLP_OFF_B2] = w;
  } else if (k < MLP_OFF_B3) {
    P->w3[k - MLP_OFF_W3] = (float)to_bf16(w);
  } else {
    P->b3 = w;
  }
}

/* One Adam step (Kingma & Ba 2015): its rates and bias corrections; off
 * for a gradient alone. */
struct AdamStep {
  float lr, b1, b2, eps, c1, c2;
  uint32_t on;
};

/* grad[k] = sum over the blocks' partials, then (adam.on) the Adam
 * step on the FP32 master parameters and the parameter's places in the
 * device image, so a training step is two launches.  A block owns 64
 * parameters and splits their partials over its 16 wavefronts (one row of
 * 256 bytes per load), each summing its rows in order in FP64, the 16 sums
 * in wavefront order: a fixed order, so training is reproducible.  Bound by
 * the latency of a wavefront's loads (nparts / 16 rows): one thread per
 * parameter walking all 768 partials took 222 us, and a batch of 2048 made
 * only 64 of them. */
__global__ void __launch_bounds__(64 * UPD_GROUPS)
k_mlp_update(const float* __restrict__ part, uint32_t nparts, float* __restrict__ grad, const double* __restrict__ sse,
             double* __restrict__ sse_out, float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
             AdamStep adam, MlpDev* __restrict__ P)
{
  __shared__ double sh[UPD_GROUPS][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + lane;
  double acc = 0.0;
  if (k < MLP_NPARAM) {
#pragma unroll 4
    for (uint32_t w = g; w < nparts; w += UPD_GROUPS) acc += part[(uint64_t)w * MLP_NPARAM + k];
  }
  sh[g][lane] = acc;
  __syncthreads();
  if (g == 0 && k < MLP_NPARAM) {
    acc = sh[0][lane];
    for (int q = 1; q < UPD_GROUPS; q++) acc += sh[q][lane];
    const float gk = (float)acc;
    grad[k] = gk;
    if (adam.on) {
      const float mk = adam.b1 * m[k] + (1.0f - adam.b1) * gk;
      const float vk = adam.b2 * v[k] + (1.0f - adam.b2) * gk * gk;
      m[k] = mk;
      v[k] = vk;
      const float w = p[k] - adam.lr * (mk / adam.c1) / (sqrtf(vk / adam.c2) + adam.eps);
      p[k] = w;
      pack_one(P, k, w);
    }
  }
  if (blockIdx.x == 0 && g == 1) {
    double e = 0.0;
    for (uint32_t w = lane; w < nparts; w += 64) e += sse[w];
    for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
    if (lane == 0) *sse_out = e;
  }
}

}  // namespace

struct cs_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  MlpDev* d_dev = nullptr;
  float* d_p = nullptr;       /* FP32 master parameters */
  float* d_m = nullptr;       /* Adam moments */
  float* d_v = nullptr;
  float* d_grad = nullptr;
  float* d_part = nullptr;
  double* d_sse = nullptr;
  double* d_sse_out = nullptr;
  uint32_t grad_blocks = 0;   /* blocks of a gradient launch */
  uint64_t adam_step = 0;
  /* training set */
  uint16_t* d_x = nullptr;
  float* d_t = nullptr;
  uint32_t* d_idx = nullptr;
  uint64_t ndata = 0, cursor = 0;
  std::vector<uint32_t> order;
  uint32_t* h_idx = nullptr;  /* pinned staging of the order's upload (IDX_CHUNK at most) */
  hipEvent_t idx_done = nullptr;
  uint64_t shuffle_state = 0;
  /* scratch of cs_mlp_forward / cs_mlp_grad */
  float* d_xs = nullptr;
  uint16_t* d_xbs = nullptr;
  float* d_ts = nullptr;
  float* d_ys = nullptr;
  uint64_t scratch_n = 0;
  MlpDev host_norm{};         /* normalisation fields (host copy) */
};

namespace {

void free_mlp(cs_mlp* m)
{
  if (!m) return;
  (void)hipSetDevice(m->device);
  void* ptrs[] = {m->d_dev, m->d_p, m->d_m, m->d_v, m->d_grad, m->d_part, m->d_sse, m->d_sse_out, m->d_x, m->d_t,
                  m->d_idx, m->d_xs, m->d_xbs, m->d_ts, m->d_ys};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (m->h_idx) (void)hipHostFree(m->h_idx);
  if (m->idx_done) (void)hipEventDestroy(m->idx_done);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
}

int pack(cs_mlp* m)
{
  hipLaunchKernelGGL(k_mlp_pack, dim3(1), dim3(256), 0, m->stream, m->d_p, m->d_dev);
  HIP_TRY(hipGetLastError());
  return CS_OK;
}

int ensure_scratch(cs_mlp* m, uint64_t n)
{
  if (n <= m->scratch_n) return CS_OK;
  m->scratch_n = 0;   /* until all four are there */
  void** ptrs[] = {(void**)&m->d_xs, (void**)&m->d_xbs, (void**)&m->d_ts, (void**)&m->d_ys};
  for (void** p : ptrs)
    if (*p) { HIP_TRY(hipFree(*p)); *p = nullptr; }
  HIP_TRY(hipMalloc(&m->d_xs, sizeof(float) * n * MLP_IN));
  HIP_TRY(hipMalloc(&m->d_xbs, sizeof(uint16_t) * n * MLP_PAD));
  HIP_TRY(hipMalloc(&m->d_ts, sizeof(float) * n));
  HIP_TRY(hipMalloc(&m->d_ys, sizeof(float) * n));
  m->scratch_n = n;
  return CS_OK;
}

int to_bf16_rows(cs_mlp* m, const float* d_x, uint64_t n, uint16_t* d_xb)
{
  const unsigned blocks = (unsigned)std::min<uint64_t>(4096, (n * MLP_PAD + 255) / 256 + 1);
  hipLaunchKernelGGL(k_mlp_to_bf16, dim3(blocks), dim3(256), 0, m->stream, d_x, n, d_xb);
  HIP_TRY(hipGetLastError());
  return CS_OK;
}

/* Gradient of sum (y - t)^2 / norm over n samples into d_grad, the sum of
 * squared errors into d_sse_out and, with adam.on, the Adam step.  No more
 * blocks than there are rounds of 32 samples: an idle one still writes
 * a partial of zeros that the update then reads (25 KB each). */
int run_grad(cs_mlp* m, const uint16_t* d_xb, const float* d_t, const uint32_t* d_idx, uint64_t n, float norm,
             const AdamStep& adam)
{
  const uint32_t blocks = (uint32_t)std::min<uint64_t>(m->grad_blocks, (n + 31) / 32);
  hipLaunchKernelGGL(k_mlp_grad, dim3(blocks), dim3(128), 0, m->stream, m->d_dev, d_xb, d_t, d_idx, n, norm, m->d_part,
                     m->d_sse);
  hipLaunchKernelGGL(k_mlp_update, dim3((MLP_NPARAM + 63) / 64), dim3(64 * UPD_GROUPS), 0, m->stream, m->d_part, blocks,
                     m->d_grad, m->d_sse, m->d_sse_out, m->d_p, m->d_m, m->d_v, adam, m->d_dev);
  HIP_TRY(hipGetLastError());
  return CS_OK;
}

}  // namespace

extern "C" {

int cs_mlp_create(const float* params, cs_mlp** out)
{
  if (!out || !params) return set_err(CS_EINVAL, "NULL argument");
  *out = nullptr;
  cs_mlp* m = new cs_mlp();
  auto bail = [&](int code) { free_mlp(m); return code; };
  if (hipGetDevice(&m->device) != hipSuccess) return bail(set_err(CS_EDEVICE, "no HIP device"));
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess)
    return bail(set_err(CS_EDEVICE, "hipStreamCreate failed"));
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, m->device) != hipSuccess) return bail(set_err(CS_EDEVICE, "device query failed"));
  m->grad_blocks = (uint32_t)std::max(1, prop.multiProcessorCount) * 3;   /* three blocks per CU */
  if (hipMalloc(&m->d_dev, sizeof(MlpDev)) != hipSuccess || hipMalloc(&m->d_p, sizeof(float) * MLP_NPARAM) != hipSuccess ||
      hipMalloc(&m->d_m, sizeof(float) * MLP_NPARAM) != hipSuccess ||
      hipMalloc(&m->d_v, sizeof(float) * MLP_NPARAM) != hipSuccess ||
      hipMalloc(&m->d_grad, sizeof(float) * MLP_NPARAM) != hipSuccess ||
      hipMalloc(&m->d_part, sizeof(float) * MLP_NPARAM * (size_t)m->grad_blocks) != hipSuccess ||
      hipMalloc(&m->d_sse, sizeof(double) * m->grad_blocks) != hipSuccess ||
      hipMalloc(&m->d_sse_out, sizeof(double)) != hipSuccess)
    return bail(set_err(CS_ENOMEM, "device allocation of the network failed"));
  /* identity normalisation until cs_mlp_set_normalisation */
  MlpDev& h = m->host_norm;
  for (int k = 0; k < MLP_IN; k++) {
    h.in_mean[k] = 0.0f;
    h.in_std[k] = 1.0f;
    h.in_lo[k] = -INFINITY;
    h.in_hi[k] = INFINITY;
  }
  h.out_mean = 0.0f;
  h.out_std = 1.0f;
  h.margin = 0.0f;
  if (hipMemcpyAsync(m->d_dev, &h, sizeof(MlpDev), hipMemcpyHostToDevice, m->stream) != hipSuccess ||
      hipMemcpyAsync(m->d_p, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
      hipMemsetAsync(m->d_m, 0, sizeof(float) * MLP_NPARAM, m->stream) != hipSuccess ||
      hipMemsetAsync(m->d_v, 0, sizeof(float) * MLP_NPARAM, m->stream) != hipSuccess)
    return bail(set_err(CS_EDEVICE, "upload of the network failed"));
  int rc = pack(m);
  if (rc != CS_OK) return bail(rc);
  if (hipStreamSynchronize(m->stream) != hipSuccess) return bail(set_err(CS_EDEVICE, "network setup failed"));
  *out = m;
  return CS_OK;
}

int cs_mlp_destroy(cs_mlp* m)
{
  if (!m) return CS_OK;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  free_mlp(m);
  return CS_OK;
}

int cs_mlp_num_params(void) { return MLP_NPARAM; }

int cs_mlp_get_params(cs_mlp* m, float* params)
{
  if (!m || !params) return set_err(CS_EINVAL, "NULL argument");
  HIP_TRY(hipSetDevice(m->device));
  HIP_TRY(hipMemcpyAsync(params, m->d_p, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return CS_OK;
}

int cs_mlp_set_params(cs_mlp* m, const float* params)
{
  if (!m || !params) return set_err(CS_EINVAL, "NULL argument");
  HIP_TRY(hipSetDevice(m->device));
  HIP_TRY(hipMemcpyAsync(m->d_p, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, m->stream));
  int rc = pack(m);
  if (rc != CS_OK) return rc;
  HIP_TRY(hipStreamSynchronize(m->stream));
  return CS_OK;
}

int cs_mlp_set_normalisation(cs_mlp* m, const float* in_mean, const float* in_std, const float* in_lo,
                             const float* in_hi, float out_mean, float out_std, float margin)
{
  if (!m || !in_mean || !in_std || !in_lo || !in_hi) return set_err(CS_EINVAL, "NULL argument");
  HIP_TRY(hipSetDevice(m->device));
  MlpDev& h = m->host_norm;
  for (int k = 0; k < MLP_IN; k++) {
    if (!(in_std[k] > 0)) return set_err(CS_EINVAL, "in_std[%d] must be positive", k);
    h.in_mean[k] = in_mean[k];
    h.in_std[k] = in_std[k];
    h.in_lo[k] = in_lo[k];
    h.in_hi[k] = in_hi[k];
  }
  if (!(out_std > 0)) return set_err(CS_EINVAL, "out_std must be positive");
  h.out_mean = out_mean;
  h.out_std = out_std;
  h.margin = margin;
  const size_t off = offsetof(MlpDev, in_mean);
  HIP_TRY(hipMemcpyAsync((char*)m->d_dev + off, (const char*)&h + off, sizeof(MlpDev) - off, hipMemcpyHostToDevice,
                         m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return CS_OK;
}

int cs_mlp_forward(cs_mlp* m, const float* x, uint64_t n, float* y)
{
  if (!m || (!x && n) || (!y && n)) return set_err(CS_EINVAL, "NULL argument");
  if (n == 0) return CS_OK;
  HIP_TRY(hipSetDevice(m->device));
  int rc = ensure_scratch(m, n);
  if (rc != CS_OK) return rc;
  HIP_TRY(hipMemcpyAsync(m->d_xs, x, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, m->stream));
  if ((rc = to_bf16_rows(m, m->d_xs, n, m->d_xbs)) != CS_OK) return rc;
  const unsigned blocks = (unsigned)std::min<uint64_t>(2048, (n + 127) / 128);
  hipLaunchKernelGGL(k_mlp_forward, dim3(blocks), dim3(256), 0, m->stream, m->d_dev, m->d_xbs, n, m->d_ys);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(y, m->d_ys, sizeof(float) * n, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return CS_OK;
}

int cs_mlp_grad(cs_mlp* m, const float* x, const float* t, uint64_t n, float* grad, double* loss)
{
  if (!m || !x || !t || !grad) return set_err(CS_EINVAL, "NULL argument");
  if (n == 0) return set_err(CS_EINVAL, "no samples");
  HIP_TRY(hipSetDevice(m->device));
  int rc = ensure_scratch(m, n);
  if (rc != CS_OK) return rc;
  HIP_TRY(hipMemcpyAsync(m->d_xs, x, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, m->stream));
  HIP_TRY(hipMemcpyAsync(m->d_ts, t, sizeof(float) * n, hipMemcpyHostToDevice, m->stream));
  if ((rc = to_bf16_rows(m, m->d_xs, n, m->d_xbs)) != CS_OK) return rc;
  if ((rc = run_grad(m, m->d_xbs, m->d_ts, nullptr, n, (float)n, AdamStep{})) != CS_OK) return rc;
  double sse = 0.0;
  HIP_TRY(hipMemcpyAsync(grad, m->d_grad, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipMemcpyAsync(&sse, m->d_sse_out, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  if (loss) *loss = sse / (double)n;
  return CS_OK;
}

int cs_mlp_set_data(cs_mlp* m, const float* x, const float* t, uint64_t n, uint64_t shuffle_seed)
{
  if (!m || !x || !t) return set_err(CS_EINVAL, "NULL argument");
  if (n == 0 || n > 0xFFFFFFFFull) return set_err(CS_ERANGE, "training set size out of range");
  HIP_TRY(hipSetDevice(m->device));
  void** ptrs[] = {(void**)&m->d_x, (void**)&m->d_t, (void**)&m->d_idx};
  for (void** p : ptrs)
    if (*p) { HIP_TRY(hipFree(*p)); *p = nullptr; }
  m->ndata = 0;
  HIP_TRY(hipStreamSynchronize(m->stream));   /* an order's upload may still read the staging buffer */
  if (m->h_idx) { HIP_TRY(hipHostFree(m->h_idx)); m->h_idx = nullptr; }
  if (!m->idx_done) HIP_TRY(hipEventCreateWithFlags(&m->idx_done, hipEventDisableTiming));
  HIP_TRY(hipHostMalloc((void**)&m->h_idx, sizeof(uint32_t) * std::min(n, IDX_CHUNK), hipHostMallocDefault));
  float* d_xf = nullptr;
  if (hipMalloc(&d_xf, sizeof(float) * n * MLP_IN) != hipSuccess ||
      hipMalloc(&m->d_x, sizeof(uint16_t) * n * MLP_PAD) != hipSuccess ||
      hipMalloc(&m->d_t, sizeof(float) * n) != hipSuccess ||
      hipMalloc(&m->d_idx, sizeof(uint32_t) * n) != hipSuccess) {
    const int rc = set_err(CS_ENOMEM, "device allocation of %llu training samples failed", (unsigned long long)n);
    if (d_xf) (void)hipFree(d_xf);
    for (void** p : ptrs)
      if (*p) { (void)hipFree(*p); *p = nullptr; }
    return rc;
  }
  HIP_TRY(hipMemcpyAsync(d_xf, x, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, m->stream));
  HIP_TRY(hipMemcpyAsync(m->d_t, t, sizeof(float) * n, hipMemcpyHostToDevice, m->stream));
  int rc = to_bf16_rows(m, d_xf, n, m->d_x);
  HIP_TRY(hipStreamSynchronize(m->stream));
  HIP_TRY(hipFree(d_xf));
  if (rc != CS_OK) return rc;
  m->ndata = n;
  m->cursor = n;   /* shuffle before the first batch */
  m->order.resize(n);
  for (uint64_t k = 0; k < n; k++) m->order[k] = (uint32_t)k;
  m->shuffle_state = shuffle_seed * 0x9E3779B97F4A7C15ull + 1;
  return CS_OK;
}

int cs_mlp_train(cs_mlp* m, uint32_t steps, uint32_t batch, float lr, double* last_loss)
{
  if (!m) return set_err(CS_EINVAL, "NULL argument");
  if (!m->ndata) return set_err(CS_EINVAL, "no training set: call cs_mlp_set_data first");
  if (batch < 32 || batch > m->ndata) return set_err(CS_ERANGE, "batch must be in 32..%llu", (unsigned long long)m->ndata);
  HIP_TRY(hipSetDevice(m->device));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (uint32_t st = 0; st < steps; st++) {
    if (m->cursor + batch > m->ndata) {
      /* a new epoch: Fisher-Yates with a 64-bit LCG (31-bit numbers, so the
       * remainder is a 32-bit one), uploaded through pinned memory in stream
       * order: the steps already queued keep the GPU busy meanwhile */
      for (uint64_t k = m->ndata - 1; k > 0; k--) {
        m->shuffle_state = m->shuffle_state * 6364136223846793005ull + 1442695040888963407ull;
        const uint32_t j = (uint32_t)(m->shuffle_state >> 33) % (uint32_t)(k + 1);
        std::swap(m->order[k], m->order[j]);
      }
      for (uint64_t o = 0; o < m->ndata; o += IDX_CHUNK) {
        const uint64_t c = std::min<uint64_t>(IDX_CHUNK, m->ndata - o);
        HIP_TRY(hipEventSynchronize(m->idx_done));   /* the staging buffer is free again */
        memcpy(m->h_idx, m->order.data() + o, sizeof(uint32_t) * c);
        HIP_TRY(hipMemcpyAsync(m->d_idx + o, m->h_idx, sizeof(uint32_t) * c, hipMemcpyHostToDevice, m->stream));
        HIP_TRY(hipEventRecord(m->idx_done, m->stream));
      }
      m->cursor = 0;
    }
    m->adam_step++;
    const AdamStep adam{lr, b1, b2, eps, 1.0f - powf(b1, (float)m->adam_step), 1.0f - powf(b2, (float)m->adam_step),
                        1u};
    const int rc = run_grad(m, m->d_x, m->d_t, m->d_idx + m->cursor, batch, (float)batch, adam);
    if (rc != CS_OK) return rc;
    m->cursor += batch;
  }
  double sse = 0.0;
  HIP_TRY(hipMemcpyAsync(&sse, m->d_sse_out, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  if (last_loss) *last_loss = sse / (double)batch;
  return CS_OK;
}

}  // extern "C"

/* The device image of a network, for the ensemble's closure gating. */
const void* cs_internal_mlp_device(const cs_mlp* m) { return m ? m->d_dev : nullptr; }
