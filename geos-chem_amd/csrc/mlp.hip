// Learned initial step size and stiffness class of a cell: a 40-input MLP
// with three hidden layers of 128 GELU units and 5 outputs (log h0, four
// class logits).  No reference counterpart: the reference starts each cell's
// Rosenbrock integration from RCNTRL(3) = KPPHvalue, the previous step's
// last step size (GeosCore/fullchem_mod.F90:1016-1020), or 1e-5 s cold.  The
// prediction only sets Hstart; the adaptive controller still accepts or
// rejects every step, so the tolerance is met as without it.
//
// Inference: bf16 MFMA (v_mfma_f32_16x16x16_bf16), fp32 accumulation, the
// activations kept in registers between layers by computing each layer
// transposed (units x cells), so one layer's accumulator tile is the next
// layer's B operand.  Training: fp32 MFMA (v_mfma_f32_16x16x4_f32), one
// launch for the forward pass, the loss and the activations' gradients, one
// for the weights' gradients in row chunks, one to add the chunks.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "cell_fields.h"
#include "gckpp_internal.h"
#include "mlp.h"

namespace gckpp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// fp32 -> bf16, round to nearest even (finite inputs; NaN stays NaN).
__device__ __forceinline__ unsigned short to_bf16(float x) {
  unsigned u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// Feature f of a cell, normalised.
__device__ __forceinline__ float mlp_feature(int f, const MlpDesc &d, const double *met,
                                             const double *photol, const double *conc,
                                             const double *hprev, int64_t n, int64_t cell) {
  double v;
  const double hp = hprev ? hprev[cell] : 0.0;
  if (f == 0) v = met[(int64_t)MET_TEMP * n + cell];
  else if (f == 1) v = log10(fmax(met[(int64_t)MET_PRESS * n + cell], 1e-30));
  else if (f == 2) v = log10(fmax(met[(int64_t)MET_NUMDEN * n + cell], 1e-30));
  else if (f == 3) v = met[(int64_t)MET_SUNCOS * n + cell];
  else if (f < 4 + MLP_NJ) v = log10(fmax(photol[(int64_t)d.jslot[f - 4] * n + cell], 0.0) + 1e-20);
  else if (f < 4 + MLP_NJ + MLP_NS)
    v = log10(fmax(conc[(int64_t)d.spc[f - 4 - MLP_NJ] * n + cell], 0.0) + 1.0);
  else if (f == MLP_NIN - 2) v = hp > 0.0 ? log(hp) : 0.0;
  else if (f == MLP_NIN - 1) v = hp > 0.0 ? 1.0 : 0.0;
  else return 0.0f;
  return (float)((v - d.mean[f]) * d.rstd[f]);
}

// X[cell][MLP_F] (fp32, padded features zero).
__global__ __launch_bounds__(256) void k_mlp_features(int64_t n, MlpDesc d, const double *met,
                                                      const double *photol, const double *conc,
                                                      const double *hprev, float *X) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * MLP_F) return;
  int64_t cell = i / MLP_F;
  int f = (int)(i % MLP_F);
  X[i] = mlp_feature(f, d, met, photol, conc, hprev, n, cell);
}

// Packs W[in][out] (fp32, row-major) of one layer into MFMA A-operand tiles of
// W^T: tile (m, c) holds W^T[16m .. 16m+15][16c .. 16c+15]; lane l of the
// tile holds 4 bf16 at W^T[16m + l%16][16c + 4(l/16) + j], j = 0..3.
__global__ void k_mlp_pack(const float *W, int nin, int nout, unsigned short *pk) {
  int kc = nin / 16, mt = nout / 16;
  int i = blockIdx.x * blockDim.x + threadIdx.x;  // (m, c, lane)
  if (i >= mt * kc * 64) return;
  int l = i % 64, c = (i / 64) % kc, m = i / (64 * kc);
  for (int j = 0; j < 4; ++j) {
    int in = 16 * c + 4 * (l / 16) + j, out = 16 * m + l % 16;
    pk[(int64_t)i * 4 + j] = to_bf16(W[(int64_t)in * nout + out]);
  }
}

// One wave per 16 cells.  Lane l works on cell 16t + l%16 and holds rows
// 4(l/16)..4(l/16)+3 of each 16-row tile.
__global__ __launch_bounds__(256) void k_mlp_predict(int64_t n, MlpDesc d, const double *met,
                                                     const double *photol, const double *conc,
                                                     const double *hprev, const bf16x4 *pk,
                                                     const float *params,
                                                     double safety, double hmin, double hmax,
                                                     double *h0, int32_t *cls) {
  const int l = threadIdx.x & 63;
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int g = l >> 4;
  const int64_t cell = tile * 16 + (l & 15);
  const bool valid = cell < n;
  const int64_t cc = valid ? cell : n - 1;  // every lane runs the MFMAs

  bf16x4 b[8];
  f32x4 acc[8];
  // layer 1 input: features 16c + 4g + j
#pragma unroll
  for (int c = 0; c < MLP_F / 16; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      b[c][j] = (short)to_bf16(mlp_feature(16 * c + 4 * g + j, d, met, photol, conc, hprev, n, cc));
  const bf16x4 *pk1 = pk;
  const bf16x4 *pk2 = pk1 + (MLP_H / 16) * (MLP_F / 16) * 64;
  const bf16x4 *pk3 = pk2 + (MLP_H / 16) * (MLP_H / 16) * 64;
  const bf16x4 *pk4 = pk3 + (MLP_H / 16) * (MLP_H / 16) * 64;
  const float *b1 = params + MLP_OFF_B1, *b2 = params + MLP_OFF_B2, *b3 = params + MLP_OFF_B3,
              *b4 = params + MLP_OFF_B4;
  auto layer = [&](const bf16x4 *w, int kc, const float *bias) {
#pragma unroll
    for (int m = 0; m < MLP_H / 16; ++m) {
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < kc; ++c)
        a = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w[(m * kc + c) * 64 + l], b[c], a, 0, 0, 0);
      acc[m] = a;
    }
#pragma unroll
    for (int m = 0; m < MLP_H / 16; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) b[m][j] = (short)to_bf16(gelu(acc[m][j] + bias[16 * m + 4 * g + j]));
  };
  layer(pk1, MLP_F / 16, b1);
  layer(pk2, MLP_H / 16, b2);
  layer(pk3, MLP_H / 16, b3);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < MLP_H / 16; ++c)
    o = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pk4[c * 64 + l], b[c], o, 0, 0, 0);
  // rows 0..3 in lanes 0-15 (log h0, logits 0..2), row 4 in lanes 16-31 (logit 3)
  float logit3 = __shfl(o[0], (l + 16) & 63) + b4[4];
  if (g == 0 && valid) {
    float lh = o[0] + b4[0];
    float z[4] = {o[1] + b4[1], o[2] + b4[2], o[3] + b4[3], logit3};
    int k = 0;
    for (int q = 1; q < 4; ++q)
      if (z[q] > z[k]) k = q;
    double h = exp((double)d.out_mu + (double)d.out_sigma * (double)lh) * safety;
    h = h < hmin ? hmin : (h > hmax ? hmax : h);
    if (h0) h0[cell] = h;
    if (cls) cls[cell] = k;
  }
}

// ---------------------------------------------------------------------------
// fp32 training kernels.
//
// One workgroup takes 16 samples through the network and back.  Every layer is
// computed transposed (units x samples, MFMA tiles of 16 x 16, K = 4 a step);
// its four waves own two of the eight 16-unit tiles each and exchange the
// activations through LDS.  Pre-activations stay in registers; the
// activations A1..A3 and the gradients dZ1..dZ3, dO go to memory once, for the
// weights' gradients.  A 4,096-sample batch is 256 workgroups of about 1,200
// MFMAs; what bounds it is the weights' way from L2 (160 KB forward, 140 KB
// back, a workgroup).  Measured with the two kernels below on 4,096 samples:
// 3,640 us a gradient with one GEMM, GELU or column sum a launch (the weights'
// gradients on four workgroups), 44 us now.
constexpr int kS = 16;            // samples per workgroup
constexpr int kLdA = kS + 1;      // LDS row of one unit

// acc[t] += sum_k A(k)(row) * B(k)(sample): KN values of k, four a step; a(k, t)
// the lane's element of tile t (row l%16, k = 4 step + l/16), b(k) of the
// samples' side.
template <int KN, class FA, class FB>
__device__ __forceinline__ void mma2(f32x4 (&acc)[2], int g, FA a, FB b) {
#pragma unroll 8
  for (int k0 = 0; k0 < KN; k0 += 4) {
    const float bv = b(k0 + g);
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(k0 + g, 0), bv, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(k0 + g, 1), bv, acc[1], 0, 0, 0);
  }
}

// act: A1, A2, A3, dZ1, dZ2, dZ3 ([nb][128] each), then O [nb][16].  Without
// yh (a forward pass) only O is written.
__global__ __launch_bounds__(256) void k_mlp_train(const float *P, int64_t nb, const float *X,
                                                   const float *yh, const int32_t *ycls, float wh,
                                                   float wc, float *act, float *dO, float *lossp) {
  __shared__ float lds[2][MLP_H * kLdA];
  __shared__ float part[4][MLP_O][kS];
  __shared__ float losses[kS];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, g = l >> 4, c = l & 15;
  const int64_t r0 = (int64_t)blockIdx.x * kS, row = r0 + c;
  const bool live = row < nb;
  float *const A[3] = {act, act + nb * MLP_H, act + 2 * nb * MLP_H};
  float *const dZ[3] = {act + 3 * nb * MLP_H, act + 4 * nb * MLP_H, act + 5 * nb * MLP_H};
  float *const O = act + 6 * nb * MLP_H;
  // inputs: lds[0][feature][sample]
  for (int e = threadIdx.x; e < kS * MLP_F; e += 256) {
    const int s = e / MLP_F, f = e % MLP_F;
    lds[0][f * kLdA + s] = r0 + s < nb ? X[(r0 + s) * MLP_F + f] : 0.f;
  }
  __syncthreads();
  f32x4 z[3][2];
  const int offW[3] = {MLP_OFF_W1, MLP_OFF_W2, MLP_OFF_W3}, offB[3] = {MLP_OFF_B1, MLP_OFF_B2, MLP_OFF_B3};
  int cur = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float *W = P + offW[k] + 32 * w + c;
    f32x4 acc[2] = {};
    auto a = [&](int i, int t) { return W[i * MLP_H + 16 * t]; };
    auto b = [&](int i) { return lds[cur][i * kLdA + c]; };
    if (k == 0) mma2<MLP_F>(acc, g, a, b);
    else mma2<MLP_H>(acc, g, a, b);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int u = 32 * w + 16 * t + 4 * g;
      f32x4 h;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        z[k][t][j] = acc[t][j] + P[offB[k] + u + j];
        h[j] = gelu(z[k][t][j]);
        lds[1 - cur][(u + j) * kLdA + c] = h[j];
      }
      if (yh && live) *(f32x4 *)(A[k] + row * MLP_H + u) = h;
    }
    cur = 1 - cur;
    __syncthreads();
  }
  // output layer: wave w takes units 32 w .. 32 w + 31 of the sum
  {
    f32x4 acc = {};
#pragma unroll
    for (int k0 = 0; k0 < 32; k0 += 4) {
      const int u = 32 * w + k0 + g;
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(P[MLP_OFF_W4 + u * MLP_O + c], lds[cur][u * kLdA + c],
                                                 acc, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) part[w][4 * g + j][c] = acc[j];
  }
  __syncthreads();
  if (threadIdx.x < kS) {
    const int s = threadIdx.x;
    float o[MLP_O];
    for (int k = 0; k < MLP_O; ++k)
      o[k] = ((part[0][k][s] + part[1][k][s]) + (part[2][k][s] + part[3][k][s])) + P[MLP_OFF_B4 + k];
    if (r0 + s < nb)
      for (int k = 0; k < MLP_O; ++k) O[(r0 + s) * MLP_O + k] = o[k];
    // L = wh * mean (O0 - yh)^2 + wc * mean CE(softmax(O1..O4), ycls)
    float L = 0.f, d[MLP_O] = {};
    if (yh && r0 + s < nb) {
      const float n = (float)nb, e = o[0] - yh[r0 + s];
      L = wh * e * e / n;
      d[0] = 2.f * wh * e / n;
      float mx = fmaxf(fmaxf(o[1], o[2]), fmaxf(o[3], o[4])), p[4], sum = 0.f;
      for (int k = 0; k < 4; ++k) {
        p[k] = expf(o[1 + k] - mx);
        sum += p[k];
      }
      const int y = ycls[r0 + s];
      float oy = 0.f;
      for (int k = 0; k < 4; ++k) {
        oy = k == y ? o[1 + k] : oy;
        d[1 + k] = wc * (p[k] / sum - (k == y ? 1.f : 0.f)) / n;
      }
      L += wc * (logf(sum) + mx - oy) / n;
      for (int k = 0; k < MLP_O; ++k) dO[(r0 + s) * MLP_O + k] = d[k];
    }
    for (int k = 0; k < MLP_O; ++k) part[0][k][s] = d[k];
    losses[s] = L;
  }
  if (!yh) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    float L = 0.f;
    for (int s = 0; s < kS; ++s) L += losses[s];
    lossp[blockIdx.x] = L;
  }
  // back: dZ = (W dZ_next) * gelu'(Z); the lane's row of W comes in groups of
  // four consecutive k, so step j of a group takes k = 16 q + 4 g + j
#pragma unroll
  for (int k = 2; k >= 0; --k) {
    const int nk = k == 2 ? MLP_O : MLP_H;
    const float *W = P + (k == 2 ? MLP_OFF_W4 : offW[k + 1]) + (32 * w + c) * nk + 4 * g;
    const float *src = k == 2 ? &part[0][0][0] : lds[cur];
    const int ld = k == 2 ? kS : kLdA;
    f32x4 acc[2] = {};
#pragma unroll 4
    for (int q = 0; q < nk; q += 16) {
      const f32x4 a0 = *(const f32x4 *)(W + q), a1 = *(const f32x4 *)(W + 16 * nk + q);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float bv = src[(q + 4 * g + j) * ld + c];
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[j], bv, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[j], bv, acc[1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int u = 32 * w + 16 * t + 4 * g;
      f32x4 d;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d[j] = acc[t][j] * gelu_grad(z[k][t][j]);
        if (k > 0) lds[1 - cur][(u + j) * kLdA + c] = d[j];
      }
      if (live) *(f32x4 *)(dZ[k] + row * MLP_H + u) = d;
    }
    cur = 1 - cur;
    if (k > 0) __syncthreads();
  }
}

// Weights' gradients of one row chunk: dW[in][out] = sum_rows Aprev[row][in]
// dZ[row][out] and db[out] = sum_rows dZ[row][out], a 32 x 32 block of one
// layer a wave (two by two MFMA tiles, the rows straight from L2).  Chunk q
// writes its own copy part[q][MLP_NPARAM]; grid (chunks, 4 waves a workgroup
// over kDwTiles blocks).
constexpr int kDwMax = 64;        // most chunks
struct DwTile { int layer, m0, n0; };
constexpr int kDwTiles = 2 * 4 + 4 * 4 + 4 * 4 + 4;  // 48 x 128, 128 x 128 twice, 128 x 16
__device__ __forceinline__ DwTile dw_tile(int i) {
  if (i < 8) return DwTile{0, 32 * (i / 4), 32 * (i % 4)};
  if (i < 24) return DwTile{1, 32 * ((i - 8) / 4), 32 * ((i - 8) % 4)};
  if (i < 40) return DwTile{2, 32 * ((i - 24) / 4), 32 * ((i - 24) % 4)};
  return DwTile{3, 32 * (i - 40), 0};
}
__global__ __launch_bounds__(256) void k_mlp_dw(int64_t nb, int64_t rows, const float *X,
                                                const float *act, const float *dO, float *part) {
  const int l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  const DwTile T = dw_tile(blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
  const int k = T.layer;
  const int nin = k == 0 ? MLP_F : MLP_H, nout = k == 3 ? MLP_O : MLP_H;
  const float *A = k == 0 ? X : act + (k - 1) * nb * MLP_H;
  const float *D = k == 3 ? dO : act + (3 + k) * nb * MLP_H;
  const int off = k == 0 ? MLP_OFF_W1 : k == 1 ? MLP_OFF_W2 : k == 2 ? MLP_OFF_W3 : MLP_OFF_W4;
  const int64_t b0 = (int64_t)blockIdx.x * rows, b1 = b0 + rows < nb ? b0 + rows : nb;
  const bool m1 = T.m0 + 16 < nin, n1 = T.n0 + 16 < nout;  // the second tiles exist
  f32x4 acc[2][2] = {};
  float bias[2] = {0.f, 0.f};
  // (a second tile that does not exist repeats the first; it is not stored)
  const float *pa = A + (b0 + g) * nin + T.m0 + c, *pd = D + (b0 + g) * nout + T.n0 + c;
  const int sa = m1 ? 16 : 0, sd = n1 ? 16 : 0;
  auto step = [&](float a0, float a1, float d0, float d1) {
    acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, d0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, d1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, d0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, d1, acc[1][1], 0, 0, 0);
    bias[0] += d0;
    bias[1] += d1;
  };
  int64_t r = b0;
#pragma unroll 1
  for (; r + 16 <= b1; r += 16) {  // 16 rows: the loads of four steps, then their products
    float a0[4], a1[4], d0[4], d1[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a0[j] = pa[4 * j * nin];
      a1[j] = pa[4 * j * nin + sa];
      d0[j] = pd[4 * j * nout];
      d1[j] = pd[4 * j * nout + sd];
    }
    pa += 16 * nin;
    pd += 16 * nout;
#pragma unroll
    for (int j = 0; j < 4; ++j) step(a0[j], a1[j], d0[j], d1[j]);
  }
#pragma unroll 1
  for (; r < b1; r += 4) {
    const bool in = r + g < b1;
    step(in ? pa[0] : 0.f, in ? pa[sa] : 0.f, in ? pd[0] : 0.f, in ? pd[sd] : 0.f);
    pa += 4 * nin;
    pd += 4 * nout;
  }
  float *G = part + (int64_t)blockIdx.x * MLP_NPARAM + off;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if ((t == 0 || m1) && (u == 0 || n1))
#pragma unroll
        for (int j = 0; j < 4; ++j)
          G[(T.m0 + 16 * t + 4 * g + j) * nout + T.n0 + 16 * u + c] = acc[t][u][j];
  if (T.m0 == 0) {  // the bias row follows the weights
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float s = bias[u];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (g == 0 && (u == 0 || n1)) G[nin * nout + T.n0 + 16 * u + c] = s;
    }
  }
}
// G = sum of the chunks' copies, in chunk order.
__global__ __launch_bounds__(256) void k_mlp_dw_sum(int chunks, const float *part, float *G) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= MLP_NPARAM) return;
  float s = 0.f;
#pragma unroll 8
  for (int q = 0; q < chunks; ++q) s += part[(int64_t)q * MLP_NPARAM + i];
  G[i] = s;
}

// out[j] = sum_i X[i][j] over nrow rows (one block per column, fixed order).
__global__ __launch_bounds__(256) void k_colsum(int64_t nrow, int ncol, const float *X, float *out) {
  __shared__ float red[256];
  int j = blockIdx.x;
  float s = 0.f;
  for (int64_t i = threadIdx.x; i < nrow; i += 256) s += X[i * ncol + j];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[j] = red[0];
}

__global__ void k_adam(int n, float *p, const float *gr, float *m, float *v, float lr, float b1,
                       float b2, float eps, float c1, float c2) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float g = gr[i];
  float mi = b1 * m[i] + (1.f - b1) * g;
  float vi = b2 * v[i] + (1.f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---------------------------------------------------------------------------
// Host-side launchers (called by the C ABI in capi.hip).
static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

void mlp_pack(const float *params, unsigned short *pk, hipStream_t s) {
  const int layers[4][3] = {{MLP_OFF_W1, MLP_F, MLP_H}, {MLP_OFF_W2, MLP_H, MLP_H},
                            {MLP_OFF_W3, MLP_H, MLP_H}, {MLP_OFF_W4, MLP_H, MLP_O}};
  int64_t off = 0;
  for (auto &L : layers) {
    int tiles = (L[2] / 16) * (L[1] / 16) * 64;
    hipLaunchKernelGGL(k_mlp_pack, dim3(nblk(tiles, 256)), dim3(256), 0, s, params + L[0], L[1], L[2],
                       pk + off * 4);
    off += tiles;
  }
}

void mlp_features(const MlpDesc &d, int64_t n, const double *met, const double *photol,
                  const double *conc, const double *hprev, float *X, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_features, dim3(nblk(n * MLP_F, 256)), dim3(256), 0, s, n, d, met, photol,
                     conc, hprev, X);
}

void mlp_predict(const MlpDesc &d, int64_t n, const double *met, const double *photol,
                 const double *conc, const double *hprev, const unsigned short *pk,
                 const float *params, double safety, double hmin, double hmax, double *h0,
                 int32_t *cls, hipStream_t s) {
  int64_t tiles = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_predict, dim3(nblk(tiles, 4)), dim3(256), 0, s, n, d, met, photol, conc,
                     hprev, (const bf16x4 *)pk, params, safety, hmin, hmax, h0, cls);
}

// fp32 forward of nb rows; O [nb][16] at act + nb * 6 * MLP_H.
void mlp_forward_f32(const float *P, int64_t nb, const float *X, float *act, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_train, dim3(nblk(nb, kS)), dim3(256), 0, s, P, nb, X, nullptr, nullptr, 0.f,
                     0.f, act, nullptr, nullptr);
}

int64_t mlp_loss_parts(int64_t nb) { return (nb + kS - 1) / kS; }
int64_t mlp_dw_floats(int64_t nb) {
  const int64_t q = (nb + 127) / 128;
  return (q < kDwMax ? q : kDwMax) * MLP_NPARAM;
}

// Gradient of the loss w.r.t. every parameter into G[MLP_NPARAM]; lossp gets
// mlp_loss_parts(nb) parts of the loss; scratch dO [nb][16], dw
// [mlp_dw_floats(nb)].  Chunks of 128 rows (32 workgroups of rows for 4,096
// samples, times eleven of blocks), more rows where that would be more than
// kDwMax chunks.
void mlp_grad_f32(const float *P, int64_t nb, const float *X, const float *yh, const int32_t *ycls,
                  float wh, float wc, float *act, float *dO, float *dw, float *G, float *lossp,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_train, dim3(nblk(nb, kS)), dim3(256), 0, s, P, nb, X, yh, ycls, wh, wc, act,
                     dO, lossp);
  int64_t rows = (nb + kDwMax - 1) / kDwMax;
  rows = rows < 128 ? 128 : (rows + 3) / 4 * 4;
  const int chunks = (int)((nb + rows - 1) / rows);
  hipLaunchKernelGGL(k_mlp_dw, dim3((unsigned)chunks, kDwTiles / 4), dim3(256), 0, s, nb, rows, X, act,
                     dO, dw);
  hipLaunchKernelGGL(k_mlp_dw_sum, dim3(nblk(MLP_NPARAM, 256)), dim3(256), 0, s, chunks, dw, G);
}

void mlp_sum(const float *x, int64_t n, float *out, hipStream_t s) {
  hipLaunchKernelGGL(k_colsum, dim3(1), dim3(256), 0, s, n, 1, x, out);
}

void mlp_adam(float *P, const float *G, float *m, float *v, float lr, int step, hipStream_t s) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(nblk(MLP_NPARAM, 256)), dim3(256), 0, s, MLP_NPARAM, P, G, m, v, lr,
                     b1, b2, eps, c1, c2);
}

}  // namespace gckpp

namespace gckpp {

// ---------------------------------------------------------------------------
// Stable counting sort of cells by class, costliest class (3) first: the
// queue order of the persistent solver.  hist[b*4 + k] = cells of class k in
// block b; one workgroup turns the counts into start offsets; each block
// then writes its cells in order.
__global__ __launch_bounds__(256) void k_class_hist(int64_t n, const int32_t *cls, int32_t *hist) {
  __shared__ int32_t cnt[4];
  if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
  __syncthreads();
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) atomicAdd(&cnt[3 - min(max(cls[i], 0), 3)], 1);
  __syncthreads();
  if (threadIdx.x < 4) hist[(int64_t)blockIdx.x * 4 + threadIdx.x] = cnt[threadIdx.x];
}

// In place: hist[b*4+k] <- start of block b's class-k cells in the output.
// Thread t owns the contiguous blocks [t*per, (t+1)*per): key by key, the
// start of its first block is the totals of all earlier keys plus the
// totals of key k over the blocks of threads before it.
__global__ __launch_bounds__(256) void k_class_scan(int64_t nb, int32_t *hist) {
  __shared__ int32_t tot[4][256];
  __shared__ int32_t base[4];
  const int64_t per = (nb + 255) / 256;
  const int64_t b0 = (int64_t)threadIdx.x * per;
  const int64_t b1 = b0 + per < nb ? b0 + per : nb;
  for (int k = 0; k < 4; ++k) {
    int32_t s = 0;
    for (int64_t b = b0; b < b1; ++b) s += hist[b * 4 + k];
    tot[k][threadIdx.x] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t run = 0;
    for (int k = 0; k < 4; ++k) {
      base[k] = run;
      for (int t = 0; t < 256; ++t) run += tot[k][t];
    }
  }
  __syncthreads();
  for (int k = 0; k < 4; ++k) {
    int32_t run = base[k];
    for (int t = 0; t < (int)threadIdx.x; ++t) run += tot[k][t];
    for (int64_t b = b0; b < b1; ++b) {
      int32_t c = hist[b * 4 + k];
      hist[b * 4 + k] = run;
      run += c;
    }
  }
}

__global__ __launch_bounds__(256) void k_class_scatter(int64_t n, const int32_t *cls,
                                                       const int32_t *start, int32_t *order) {
  __shared__ int32_t key[256];
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int k = i < n ? 3 - min(max(cls[i], 0), 3) : 4;
  key[threadIdx.x] = k;
  __syncthreads();
  if (i < n) {
    int32_t r = 0;  // rank among the earlier cells of this block with the same key
    for (int t = 0; t < (int)threadIdx.x; ++t) r += key[t] == k;
    order[start[(int64_t)blockIdx.x * 4 + k] + r] = (int32_t)i;
  }
}

void order_by_class(int64_t n, const int32_t *cls, int32_t *order, int32_t *scratch, hipStream_t s) {
  int64_t nb = (n + 255) / 256;
  hipLaunchKernelGGL(k_class_hist, dim3((unsigned)nb), dim3(256), 0, s, n, cls, scratch);
  hipLaunchKernelGGL(k_class_scan, dim3(1), dim3(256), 0, s, nb, scratch);
  hipLaunchKernelGGL(k_class_scatter, dim3((unsigned)nb), dim3(256), 0, s, n, cls, scratch, order);
}

// ---------------------------------------------------------------------------
// Stable counting sort of cells by predicted initial step size, smallest
// (the stiffest, costliest cells) first: key = one of H0_BINS bins of
// log10(h0) over [1e-5 s, 1200 s] (a quarter decade each); h0 <= 0 or not
// finite (no prediction) sorts last.  Same three passes as the class sort,
// over the keys stored in the scratch.
constexpr int H0_BINS = 32;
__global__ __launch_bounds__(256) void k_h0_key(int64_t n, const double *h0, int32_t *key) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double h = h0[i];
  int k = H0_BINS - 1;
  if (h > 0.0 && h < INFINITY) {
    const double x = (log10(h) + 5.0) * (H0_BINS / (5.0 + log10(1200.0)));
    k = x < 0.0 ? 0 : (x >= (double)(H0_BINS - 1) ? H0_BINS - 1 : (int)x);
  }
  key[i] = k;
}
__global__ __launch_bounds__(256) void k_key_hist(int64_t n, const int32_t *key, int32_t *hist) {
  __shared__ int32_t cnt[H0_BINS];
  if (threadIdx.x < H0_BINS) cnt[threadIdx.x] = 0;
  __syncthreads();
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) atomicAdd(&cnt[key[i]], 1);
  __syncthreads();
  if (threadIdx.x < H0_BINS) hist[(int64_t)blockIdx.x * H0_BINS + threadIdx.x] = cnt[threadIdx.x];
}
// In place: hist[b*K+k] <- start of block b's key-k cells (as k_class_scan).
__global__ __launch_bounds__(256) void k_key_scan(int64_t nb, int32_t *hist) {
  __shared__ int32_t tot[H0_BINS][256];
  __shared__ int32_t base[H0_BINS];
  const int64_t per = (nb + 255) / 256;
  const int64_t b0 = (int64_t)threadIdx.x * per;
  const int64_t b1 = b0 + per < nb ? b0 + per : nb;
  for (int k = 0; k < H0_BINS; ++k) {
    int32_t s = 0;
    for (int64_t b = b0; b < b1; ++b) s += hist[b * H0_BINS + k];
    tot[k][threadIdx.x] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t run = 0;
    for (int k = 0; k < H0_BINS; ++k) {
      base[k] = run;
      for (int t = 0; t < 256; ++t) run += tot[k][t];
    }
  }
  __syncthreads();
  for (int k = 0; k < H0_BINS; ++k) {
    int32_t run = base[k];
    for (int t = 0; t < (int)threadIdx.x; ++t) run += tot[k][t];
    for (int64_t b = b0; b < b1; ++b) {
      int32_t c = hist[b * H0_BINS + k];
      hist[b * H0_BINS + k] = run;
      run += c;
    }
  }
}
__global__ __launch_bounds__(256) void k_key_scatter(int64_t n, const int32_t *key,
                                                     const int32_t *start, int32_t *order) {
  __shared__ int32_t ks[256];
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int k = i < n ? key[i] : H0_BINS;
  ks[threadIdx.x] = k;
  __syncthreads();
  if (i < n) {
    int32_t r = 0;  // rank among the earlier cells of this block with the same key
    for (int t = 0; t < (int)threadIdx.x; ++t) r += ks[t] == k;
    order[start[(int64_t)blockIdx.x * H0_BINS + k] + r] = (int32_t)i;
  }
}

int64_t order_by_h0_scratch(int64_t n) { return n + (int64_t)H0_BINS * ((n + 255) / 256); }

void order_by_h0(int64_t n, const double *h0, int32_t *order, int32_t *scratch, hipStream_t s) {
  int64_t nb = (n + 255) / 256;
  int32_t *key = scratch, *hist = scratch + n;
  hipLaunchKernelGGL(k_h0_key, dim3((unsigned)nb), dim3(256), 0, s, n, h0, key);
  hipLaunchKernelGGL(k_key_hist, dim3((unsigned)nb), dim3(256), 0, s, n, key, hist);
  hipLaunchKernelGGL(k_key_scan, dim3(1), dim3(256), 0, s, nb, hist);
  hipLaunchKernelGGL(k_key_scatter, dim3((unsigned)nb), dim3(256), 0, s, n, key, hist, order);
}

}  // namespace gckpp
