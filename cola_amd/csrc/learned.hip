// Learned low-rank preconditioner: a per-point MLP (din -> 128 -> 128 -> dout, GELU),
// its training kernels, and the small dense algebra that turns its output into a
// Woodbury factor; plus the rank-r pivoted Cholesky comparator and the dense RBF
// kernel-matrix builder.
//
//   mlp_fwd      one block = 16 points; the three layers run back to back on MFMA with the
//                hidden activations in LDS, optional pre-activation save for the
//                backward pass                                [latency, ~50k flop/point]
//   mlp_bwd      64 points per chunk on MFMA; per-chunk partial parameter gradients in the
//                flat parameter layout, summed over chunks in index order (FP64)
//   gram         C = X^T Y for tall-skinny X, Y (FP64 accumulation, fixed order)
//   rows_gemm    Y = alpha X W + beta Y for tall-skinny X and a small W (LDS-staged)
//   spd_inv      batched Cholesky of small SPD matrices (k <= 64) with jitter,
//                triangular inverse, full inverse                          [latency]
//   energy       the captured-energy loss and its two small gradient factors
//   pivchol      greedy (largest residual diagonal) pivoted Cholesky, Harbrecht,
//                Peters & Schneider (2012): one column kernel per rank step with a
//                fused block argmax of the updated diagonal              [HBM]
//   rbf_dense    K_ij = exp(-|p_i - p_j|^2 / (2 l^2)), exactly symmetric,
//                optional bf16 copy                                         [HBM write]
//   dense_f64acc Y = scale A X + shift X with fp32 A and fp64 vectors/accumulation
//                (refinement residuals of dense systems)                   [HBM]
#include "common.hpp"

using namespace ck;

namespace {

constexpr int kH = 128;     // hidden width
constexpr int kMaxIn = 8;   // input dimension limit
constexpr int kMaxOut = 128;
constexpr int kRows = 64;   // points per block

struct MlpLayout {
  int64_t w1, b1, w2, b2, w3, b3, total;
};

__host__ __device__ inline MlpLayout mlp_layout(int din, int dout) {
  MlpLayout L;
  L.w1 = 0;
  L.b1 = L.w1 + (int64_t)din * kH;
  L.w2 = L.b1 + kH;
  L.b2 = L.w2 + (int64_t)kH * kH;
  L.w3 = L.b2 + kH;
  L.b3 = L.w3 + (int64_t)kH * dout;
  L.total = L.b3 + dout;
  return L;
}

// exact (erf) GELU and its derivative Phi(z) + z phi(z)
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  const float cdf = 0.5f * (1.f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return fmaf(z, pdf, cdf);
}

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ floatx4 mfma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Every sum of the network runs over k in index order, each term added by one fma: an MFMA adds its four
// products that way (lane group g = lane / 16 holds the g-th), so step (c, e) takes k = 16 c + 4 e + g.
// A lane's operands of four steps e are one float4 when they are kept with k at place(k).
// The features' rounding errors reach the gradient multiplied by the condition number of a Gram matrix;
// in another order (16 c + 4 g + e) the gradient moved by up to 4e-4 of itself.
__device__ __forceinline__ int place(int k) { return (k & ~15) | (k & 3) << 2 | (k >> 2 & 3); }

// v[e] of lane group g exchanged with v[g] of lane group e: the operands of four steps from a float4 at 4 g
__device__ __forceinline__ void transpose4(floatx4& v) {
  uint32_t r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = __float_as_uint(v[e]);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto t = __builtin_amdgcn_permlane32_swap(r[e], r[e + 2], false, false);
    r[e] = t[0];
    r[e + 2] = t[1];
  }
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    const auto t = __builtin_amdgcn_permlane16_swap(r[e], r[e + 1], false, false);
    v[e] = __uint_as_float(t[0]);
    v[e + 1] = __uint_as_float(t[1]);
  }
}

// entries p[0 .. 3], those from index `left` on replaced by the last valid one
__device__ __forceinline__ floatx4 load4(const float* __restrict__ p, int left) {
  if (left >= 4) return *reinterpret_cast<const f4u*>(p);
  floatx4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = p[min(e, left - 1)];
  return v;
}

// ------------------------------------------------------------------ MLP forward
// One block: 16 points, four waves of 32 hidden units; all three layers on
// v_mfma_f32_16x16x4f32, bias first and then the inputs in order.  The activations are kept by place(),
// so a lane's operand is a float4 of its row in LDS; the weights come straight from
// memory, every one of them issued before the first layer runs.  The accumulator holds four
// consecutive points of one unit: the saved pre-activations, stored by unit, are 16-byte stores.
// Latency bound at the training size (1024 points): 16 points per block make 64 blocks there, where
// 64 made 16, and with 64 points on the matrix units larger sets run no faster either (16384 points 22.6
// against 27.0 us, 131072 123 against 124: the weights a block reads come from L2).  The activations are
// rolled loops over LDS: a launch runs its code once, from cold instruction caches.  1024 points: 40.4
// us with 64 points per block on the vector units, now 8.6; 16384: 46.8 -> 20.2 us.
constexpr int kFwdRows = 16;

template <bool SAVE>
__global__ __launch_bounds__(256) void mlp_fwd_kernel(int n, int din, int dout, const float* __restrict__ X,
                                                      int64_t ldx, const float* __restrict__ prm,
                                                      float* __restrict__ G, int64_t gsr, int64_t gsc,
                                                      float* __restrict__ Z1, float* __restrict__ Z2, int64_t ldz) {
  constexpr int kP = kH + 4;  // row pitch: 16-byte aligned, rows four banks apart
  __shared__ __align__(16) float h[2][kFwdRows][kP];
  const MlpLayout L = mlp_layout(din, dout);
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), g = lane >> 4, li = lane & 15;
  const int p0 = blockIdx.x * kFwdRows;
  const int u0 = 32 * w + li;  // this lane's unit of the wave's first tile, the second's is u0 + 16
  // layer 1 (din <= 8: k = 4 s + g), biases, W2, the wave's first tile of W3
  float x1[2], w1[2][2], b1[2], b2[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int d = 4 * s + g, dc = min(d, din - 1);
    x1[s] = X[(int64_t)min(p0 + li, n - 1) * ldx + dc];
#pragma unroll
    for (int u = 0; u < 2; ++u) w1[u][s] = prm[L.w1 + dc * kH + u0 + 16 * u];
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    b1[u] = prm[L.b1 + u0 + 16 * u];
    b2[u] = prm[L.b2 + u0 + 16 * u];
  }
  float w2[2][32], w3[32];
  const float* w2p = prm + L.w2 + g * kH + u0;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int u = 0; u < 2; ++u) w2[u][4 * c + e] = w2p[(16 * c + 4 * e) * kH + 16 * u];
  int o = 16 * w + li;  // this lane's output
  float b3;
  auto load_w3 = [&]() {
    const float* w3p = prm + L.w3 + (int64_t)g * dout + min(o, dout - 1);
    b3 = prm[L.b3 + min(o, dout - 1)];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) w3[4 * c + e] = w3p[(16 * c + 4 * e) * dout];
  };
  load_w3();
  __builtin_amdgcn_sched_barrier(0);
  // z: pre-activations of the wave's 32 units; saved, activated in place in LDS
  const int hu = 32 * w + place(li);
  auto activate = [&](const floatx4 (&z)[2], float* __restrict__ Z, int buf) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const floatx4 v = z[u];
      if (SAVE) {
        float* d = Z + (int64_t)(u0 + 16 * u) * ldz + p0 + 4 * g;
        const int left = n - (p0 + 4 * g);
        if (left >= 4)
          *reinterpret_cast<f4u*>(d) = v;
        else
          for (int q = 0; q < left; ++q) d[q] = q == 0 ? v[0] : q == 1 ? v[1] : v[2];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) h[buf][4 * g + q][hu + 16 * u] = v[q];
    }
    // each lane activates the entries it wrote: no barrier
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      float* q = &h[buf][4 * g + (i & 3)][hu + 4 * (i & 4)];
      *q = gelu(*q);
    }
  };
  floatx4 z[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) z[u] = floatx4{b1[u], b1[u], b1[u], b1[u]};
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool in = 4 * s + g < din;
      z[u] = mfma(in ? x1[s] : 0.f, in ? w1[u][s] : 0.f, z[u]);
    }
  activate(z, Z1, 0);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u) z[u] = floatx4{b2[u], b2[u], b2[u], b2[u]};
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const floatx4 a = *reinterpret_cast<const floatx4*>(&h[0][li][16 * c + 4 * g]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int u = 0; u < 2; ++u) z[u] = mfma(a[e], w2[u][4 * c + e], z[u]);
  }
  activate(z, Z2, 1);
  __syncthreads();
#pragma unroll 1
  for (; o - li < dout; o += 64) {
    floatx4 y = {b3, b3, b3, b3};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const floatx4 a = *reinterpret_cast<const floatx4*>(&h[1][li][16 * c + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) y = mfma(a[e], w3[4 * c + e], y);
    }
    if (o < dout) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t row = p0 + 4 * g + q;
        if (row < n) G[row * gsr + (int64_t)o * gsc] = y[q];
      }
    }
    if (o - li + 64 < dout) {
      o += 64;
      load_w3();
      o -= 64;
    }
  }
}

// ----------------------------------------------------------------- MLP backward
// Given dL/dG for a chunk of 64 points, writes that chunk's contribution to every parameter gradient
// (flat layout) into part[blockIdx.x * total + ...].  Eight waves; the five products
//   dH2 = dG W3^T, dW3 = h2^T dG, dH1 = dZ2 W2^T, dW2 = h1^T dZ2 (and dW1 = X^T dZ1 on the vector units)
// run on v_mfma_f32_16x16x4f32 in the order of the forward pass: every operand is a float4
// along the sum (by place()), so dG and dZ2 are kept both by point and by column.  dZ2 is formed whole; everything
// that follows is done for 32 hidden units at a time, quarter blockIdx.y, + gridDim.y, ... -- few chunks
// are spread over up to four blocks each.  Latency bound at the training size (1024 points): 119.4 us
// with a chunk per block on the vector units, now 22 us; 16384 points, the sum over chunks included: 184 -> 109 us.
constexpr int kBP = kH + 4;     // pitch of rows by point
constexpr int kBT = kRows + 4;  // pitch of rows by column
constexpr int kBQ = 32;         // hidden units per quarter

__global__ __launch_bounds__(512) void mlp_bwd_kernel(int n, int din, int dout, const float* __restrict__ X,
                                                      int64_t ldx, const float* __restrict__ prm,
                                                      const float* __restrict__ Z1, const float* __restrict__ Z2,
                                                      int64_t ldz, const float* __restrict__ dG, int64_t dsr,
                                                      int64_t dsc, float* __restrict__ part) {
  __shared__ __align__(16) float Dg[kRows][kBP], DgT[kH][kBT];  // dG, zero past dout and past n
  __shared__ __align__(16) float Dz[kRows][kBP], DzT[kH][kBT];  // dZ2
  __shared__ __align__(16) float Hq[kBQ][kBT], Eq[kBQ][kBT];    // the quarter's h2, then h1; its dZ1 (points as they are)
  __shared__ float xs[kRows][kMaxIn + 1];                       // the points, and 1 for the bias
  const MlpLayout L = mlp_layout(din, dout);
  float* out = part + (int64_t)blockIdx.x * L.total;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), g = lane >> 4, li = lane & 15;
  const int p0 = blockIdx.x * kRows, left = n - p0;  // points of this chunk
  const int nc = (dout + 15) / 16;
  // Z2 at this lane's unit and four points of each row tile: the accumulator's layout
  const int u = 16 * w + li;
  floatx4 z2[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int p = min(16 * r + 4 * g, left - 1);
    z2[r] = load4(Z2 + (int64_t)u * ldz + p0 + p, left - p);
  }
  float w3[8][4];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    if (c < nc) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w3[c][e] = prm[L.w3 + (int64_t)u * dout + min(16 * c + 4 * e + g, dout - 1)];
    }
  for (int e0 = 0; e0 < 16 * nc; e0 += 64) {  // dG: lanes along the points, eight columns per thread
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      v[q] = dG[(int64_t)(p0 + min(lane, left - 1)) * dsr + (int64_t)min(e0 + w + 8 * q, dout - 1) * dsc];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int c = e0 + w + 8 * q;
      const float d = c < dout && lane < left ? v[q] : 0.f;
      Dg[lane][place(c)] = d;
      DgT[c][place(lane)] = d;
    }
  }
  {
    const int d = w;  // kMaxIn == 8 waves
    const float v = X[(int64_t)(p0 + min(lane, left - 1)) * ldx + min(d, din - 1)];
    xs[lane][d] = d < din && lane < left ? v : 0.f;
    if (w == 0) xs[lane][kMaxIn] = 1.f;
  }
  __syncthreads();
  // dZ2 = (dG W3^T) * gelu'(Z2), all 128 units: wave w takes units 16 w .., four row tiles
  {
    floatx4 a[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (c < nc) {
        floatx4 d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = *reinterpret_cast<const floatx4*>(&Dg[16 * r + li][16 * c + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) a[r] = mfma(d[r][e], 16 * c + 4 * e + g < dout ? w3[c][e] : 0.f, a[r]);
      }
    const int up = place(u);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        DzT[u][16 * r + 4 * q + g] = a[r][q];
        Dz[16 * r + 4 * g + q][up] = z2[r][q];
      }
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {  // the entries this lane wrote
      const int p = 16 * (i >> 2) + 4 * g + (i & 3);
      const float v = p < left ? DzT[u][place(p)] * gelu_grad(Dz[p][up]) : 0.f;
      DzT[u][place(p)] = v;
      Dz[p][up] = v;
    }
  }
#pragma unroll 1
  for (int y = blockIdx.y; y < kH / kBQ; y += gridDim.y) {
    const int j0 = kBQ * y;
    // W2 rows of the wave's dH1 tile (row tile w & 3, units j0 + 16 (w >> 2) ..) and Z1 there
    const int j = j0 + 16 * (w >> 2) + li, rt = w & 3, p = min(16 * rt + 4 * g, left - 1);
    floatx4 w2[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) w2[c] = *reinterpret_cast<const floatx4*>(prm + L.w2 + (int64_t)j * kH + 16 * c + 4 * g);
    const floatx4 z1 = load4(Z1 + (int64_t)j * ldz + p0 + p, left - p);
    // h2 of the quarter
    {
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = Z2[(int64_t)(j0 + w + 8 * q) * ldz + p0 + min(lane, left - 1)];
      __syncthreads();  // the previous quarter's Hq and Eq are read
#pragma unroll
      for (int q = 0; q < 4; ++q) Hq[w + 8 * q][place(lane)] = v[q];
#pragma unroll 1
      for (int q = 0; q < 4; ++q) Hq[w + 8 * q][place(lane)] = gelu(Hq[w + 8 * q][place(lane)]);
    }
    __syncthreads();  // Hq, and (first quarter) Dz, DzT
    // dW3[j][c] = sum_p h2[p][j] dG[p][c]
    for (int tile = w; tile < 2 * nc; tile += 8) {
      const int jt = tile & 1, ct = tile >> 1;
      floatx4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const floatx4 hv = *reinterpret_cast<const floatx4*>(&Hq[16 * jt + li][16 * c + 4 * g]);
        const floatx4 dv = *reinterpret_cast<const floatx4*>(&DgT[16 * ct + li][16 * c + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) a = mfma(hv[e], dv[e], a);
      }
      const int col = 16 * ct + li;
      if (col < dout) {
#pragma unroll
        for (int q = 0; q < 4; ++q) out[L.w3 + (int64_t)(j0 + 16 * jt + 4 * g + q) * dout + col] = a[q];
      }
    }
    // db3 (first quarter) and db2 of the quarter: one row of 64 points per thread
    const int nb = kBQ + (y == 0 ? dout : 0);
    if (t < nb) {
      const float* row = t < kBQ ? DzT[j0 + t] : DgT[t - kBQ];
      float s = 0.f;
#pragma unroll 1
      for (int c = 0; c < kRows; c += 16) {
        floatx4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const floatx4*>(row + c + 4 * q);
#pragma unroll
        for (int q = 0; q < 16; ++q) s += v[q & 3][q >> 2];
      }
      out[t < kBQ ? L.b2 + j0 + t : L.b3 + t - kBQ] = s;
    }
    // dH1 tile
    floatx4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const floatx4 d = *reinterpret_cast<const floatx4*>(&Dz[16 * rt + li][16 * c + 4 * g]);
      transpose4(w2[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) a = mfma(d[e], w2[c][e], a);
    }
    __syncthreads();  // h2 is read
    const int jl = 16 * (w >> 2) + li;
    *reinterpret_cast<floatx4*>(&Eq[jl][16 * rt + 4 * g]) = a;
#pragma unroll
    for (int q = 0; q < 4; ++q) Hq[jl][16 * rt + 4 * q + g] = z1[q];
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {  // the entries this lane wrote: dZ1 and h1
      const float z = Hq[jl][16 * rt + 4 * q + g];
      float* e = &Eq[jl][16 * rt + 4 * g + q];
      *e = 16 * rt + 4 * g + q < left ? *e * gelu_grad(z) : 0.f;
      Hq[jl][16 * rt + 4 * q + g] = gelu(z);
    }
    __syncthreads();
    // dW1[d][j] and db1[j] (the point's constant 1): thread (j, d)
    for (int o = t; o < kBQ * (din + 1); o += 512) {
      const int q = o & (kBQ - 1), d = o / kBQ, dc = d < din ? d : kMaxIn;
      float s = 0.f;
#pragma unroll 4
      for (int r = 0; r < kRows; ++r) s = fmaf(xs[r][dc], Eq[q][r], s);
      out[d < din ? L.w1 + (int64_t)d * kH + j0 + q : L.b1 + j0 + q] = s;
    }
    // dW2[j][k] = sum_p h1[p][j] dZ2[p][k]: wave w takes k = 16 w .., both unit tiles
    floatx4 b[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const floatx4 dv = *reinterpret_cast<const floatx4*>(&DzT[u][16 * c + 4 * g]);
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) {
        const floatx4 hv = *reinterpret_cast<const floatx4*>(&Hq[16 * jt + li][16 * c + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) b[jt] = mfma(hv[e], dv[e], b[jt]);
      }
    }
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int q = 0; q < 4; ++q) out[L.w2 + (int64_t)(j0 + 16 * jt + 4 * g + q) * kH + u] = b[jt][q];
  }
}


// grad[p] = scale * sum_b part[b][p] (blocks in index order, FP64)
__global__ __launch_bounds__(256) void grad_reduce_kernel(int nblk, int64_t total, const float* __restrict__ part,
                                                          float scale, float* __restrict__ grad) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= total) return;
  double acc = 0.0;
  for (int b = 0; b < nblk; ++b) acc += (double)part[(int64_t)b * total + p];
  grad[p] = (float)(scale * acc);
}

// torch.optim.Adam update (no weight decay): m, v moments; bc1 = 1 - b1^t, bc2 = 1 - b2^t
__global__ __launch_bounds__(256) void adam_kernel(int64_t count, float* __restrict__ p, const float* __restrict__ gr,
                                                   float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                                   float b2, float eps, float bc1, float bc2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const float gi = gr[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float denom = sqrtf(vi) / sqrtf(bc2) + eps;
  p[i] -= (lr / bc1) * (mi / denom);
}

// ------------------------------------------------------------------ gram C = X^T Y
constexpr int kGramChunk = 64;        // rows staged per pass
constexpr int64_t kGramMaxParts = 1024;  // partials per output entry, at most
// rows per partial: one 64-row chunk per block until n needs more than kGramMaxParts
inline int64_t gram_rows(int64_t n) { return kGramChunk * cdiv(cdiv(n, kGramChunk), kGramMaxParts); }

__global__ __launch_bounds__(256) void gram_partials(int64_t n, int64_t rows, int ka, int kb,
                                                     const float* __restrict__ X, int64_t xsr, int64_t xsc,
                                                     const float* __restrict__ Y, int64_t ysr, int64_t ysc,
                                                     double* __restrict__ part) {
  __shared__ float xs[64][33];
  __shared__ float ys[64][33];
  const int ta = blockIdx.y, tb = blockIdx.z;
  const int al = threadIdx.x >> 3, bq = (threadIdx.x & 7) * 4;
  const int64_t r0 = (int64_t)blockIdx.x * rows;
  const int64_t r1 = r0 + rows < n ? r0 + rows : n;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t rb = r0; rb < r1; rb += kGramChunk) {
    // loads unconditional (indexes clamped) so a chunk's loads issue together
    float vx[8], vy[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = threadIdx.x + 256 * q, rr = e & 63, cc = e >> 6;
      const int64_t i = rb + rr < r1 ? rb + rr : r1 - 1;
      vx[q] = X[i * xsr + (int64_t)min(ta * 32 + cc, ka - 1) * xsc];
      vy[q] = Y[i * ysr + (int64_t)min(tb * 32 + cc, kb - 1) * ysc];
    }
    __syncthreads();  // previous chunk's reads done
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = threadIdx.x + 256 * q, rr = e & 63, cc = e >> 6;
      const bool in = rb + rr < r1;
      xs[rr][cc] = (in && ta * 32 + cc < ka) ? vx[q] : 0.f;
      ys[rr][cc] = (in && tb * 32 + cc < kb) ? vy[q] : 0.f;
    }
    __syncthreads();
    for (int rr = 0; rr < 64; ++rr) {
      const double xv = (double)xs[rr][al];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = fma(xv, (double)ys[rr][bq + q], acc[q]);
    }
  }
  const int ai = ta * 32 + al;
  if (ai >= ka) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int bi = tb * 32 + bq + q;
    if (bi < kb) part[(int64_t)blockIdx.x * ka * kb + (int64_t)ai * kb + bi] = acc[q];
  }
}

__global__ __launch_bounds__(256) void gram_reduce(int nchunks, int64_t count, const double* __restrict__ part,
                                                   double* __restrict__ C) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= count) return;
  double acc = 0.0;
  for (int c0 = 0; c0 < nchunks; c0 += 16) {
    double v[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = part[(int64_t)min(c0 + c, nchunks - 1) * count + idx];  // in flight together
#pragma unroll
    for (int c = 0; c < 16; ++c) acc += c0 + c < nchunks ? v[c] : 0.0;
  }
  C[idx] = acc;
}

// --------------------------------------------------------- rows GEMM Y = a X W + b Y
constexpr int kGemmMax = 128;

// One block: 64 rows x 32 columns, thread (row, 8 columns); the rows of X and the columns of W it needs
// are staged in LDS 64 of the sum at a time.  1024 x 64 x 64: 16.3 us with a row of 32 columns per
// thread and X from global memory (8 blocks), now 8.8 us.
__global__ __launch_bounds__(256) void rows_gemm_kernel(int64_t n, int kin, int kout, const float* __restrict__ X,
                                                        int64_t xsr, int64_t xsc, const float* __restrict__ W,
                                                        float alpha, float beta, float* __restrict__ Y, int64_t ysr,
                                                        int64_t ysc) {
  __shared__ float xs[64][65];
  __shared__ __align__(16) float ws[64][32];
  const int t = threadIdx.x, r = t & 63, cg = (t >> 6) * 8;
  const int64_t i0 = (int64_t)blockIdx.x * 64, i = i0 + r;
  const int c0 = blockIdx.y * 32;
  float acc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = 0.f;
  for (int j0 = 0; j0 < kin; j0 += 64) {
    float xv[16], wv[8];  // clamped indexes: both groups issue together
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int e = t + 256 * q;
      // consecutive threads along the operand's contiguous direction
      const int rr = xsr == 1 ? e & 63 : e >> 6, jj = xsr == 1 ? e >> 6 : e & 63;
      const int64_t row = i0 + rr < n ? i0 + rr : n - 1;
      xv[q] = X[row * xsr + (int64_t)min(j0 + jj, kin - 1) * xsc];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = t + 256 * q, jj = e >> 5, cc = e & 31;
      wv[q] = W[(int64_t)min(j0 + jj, kin - 1) * kout + min(c0 + cc, kout - 1)];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int e = t + 256 * q;
      const int rr = xsr == 1 ? e & 63 : e >> 6, jj = xsr == 1 ? e >> 6 : e & 63;
      xs[rr][jj] = xv[q];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = t + 256 * q;
      ws[e >> 5][e & 31] = wv[q];
    }
    __syncthreads();
    const int jn = kin - j0 < 64 ? kin - j0 : 64;
#pragma unroll 4
    for (int j = 0; j < jn; ++j) {
      const float x = xs[r][j];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = fmaf(x, ws[j][cg + q], acc[q]);
    }
  }
  if (i >= n) return;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (c0 + cg + q < kout) {
      float* y = Y + i * ysr + (int64_t)(c0 + cg + q) * ysc;
      *y = beta == 0.f ? alpha * acc[q] : fmaf(beta, *y, alpha * acc[q]);
    }
  }
}

// ------------------------------------------------------ small SPD: chol, L^-1, A^-1
constexpr int kSpdMax = 64;
constexpr int kSpdPitch = kSpdMax + 2;  // LDS row pitch in doubles: 16-byte aligned pairs, two banks apart

// 1 / p: the hardware's estimate (good to about 2^-26) and three Newton steps; the library's division where
// the estimate could overflow or flush.  And a / p from it: one correction of a r, which by itself carries
// two more roundings than a division.
__device__ __forceinline__ double rcp_f64(double p) {
  if (!(fabs(p) > 1e-290 && fabs(p) < 1e290)) return 1.0 / p;
  double r = __builtin_amdgcn_rcp(p);
  r = fma(r, fma(-p, r, 1.0), r);
  r = fma(r, fma(-p, r, 1.0), r);
  return fma(r, fma(-p, r, 1.0), r);
}
__device__ __forceinline__ double quotient(double a, double p, double r) {
  const double q = a * r;
  return fma(fma(-p, q, a), r, q);
}

// One block per matrix: A + (jitter_abs + jitter_rel * trace(A) / k) I = L L^T.
// linv (required, k x k row-major lower) = L^-1; inv64 / inv32 = A^-1; linvT32 = L^-T.
// status[b] = 0, or j + 1 when the j-th pivot is not positive.
// Latency bound: k dependent pivots.  The factorization runs as L D L^T (L unit lower) and is applied
// to the identity in the same steps, two pivots to a step: columns j, j + 1 of what is left of A and rows
// j, j + 1 of Y = L^-1 are read from a double-buffered LDS row (one barrier, one LDS round trip per
// step), every thread updates its 4 x 4 pieces of A and Y in registers, and the owners of the next two
// columns and rows publish them.  D^-1/2 (the square roots) scales Y's rows once at the end.
// k = 64: 110.8 us with a column per step, two barriers, a square root and a division each; 42.5 us
// with one pivot per step; now 34.6 us (33.1 with products by the reciprocal in place of quotients).
__global__ __launch_bounds__(256) void spd_inv_kernel(int k, const double* __restrict__ A, int64_t lda, int64_t sa,
                                                      double jitter_rel, double jitter_abs, double* __restrict__ linv,
                                                      double* __restrict__ inv64, float* __restrict__ inv32,
                                                      float* __restrict__ linvT32, int* __restrict__ status) {
  __shared__ __align__(16) double Xs[kSpdMax * kSpdPitch];
  __shared__ double2 acol[2][kSpdMax];  // [row i]: A's entries (i, j) and (i, j + 1)
  __shared__ double2 yrow[2][kSpdMax];  // [column c]: Y's entries (j, c) and (j + 1, c)
  __shared__ double piv[kSpdMax];
  __shared__ double red[4];
  const int b = blockIdx.x, t = threadIdx.x, ti = t >> 4, tj = t & 15;
  const int64_t kk = (int64_t)k * k;
  const double* Ab = A + (int64_t)b * sa;
  // piece (u, v): row at(ti, u), column at(tj, v) of the symmetric matrix, neighbouring pairs 32 apart,
  // read from its lower triangle; loads are unconditional (indexes clamped) and issue together
  auto at = [](int q, int u) { return 2 * q + (u & 1) + 32 * (u >> 1); };
  double av[4][4], yv[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = at(ti, u), c = at(tj, v), hi = min(max(i, c), k - 1), lo = min(min(i, c), k - 1);
      av[u][v] = Ab[(int64_t)hi * lda + lo];
    }
  double tr = 0.0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (ti == tj && at(ti, u) < k) tr += av[u][u];
  tr = block_sum<256>(tr, red);
  const double shift = jitter_abs + jitter_rel * tr / k;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const bool diag = ti == tj && u == v;
      // past the order: the identity, which factors to itself
      const bool in = at(ti, u) < k && at(tj, v) < k;
      yv[u][v] = diag ? 1.0 : 0.0;
      av[u][v] = in ? av[u][v] + (diag ? shift : 0.0) : yv[u][v];
    }
  auto publish = [&](int buf, int j) {  // columns and rows j, j + 1 (j even)
    const int q = (j >> 1) & 15;
    const bool hi = j >= 32;
    if (tj == q) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        acol[buf][at(ti, u)] = hi ? make_double2(av[u][2], av[u][3]) : make_double2(av[u][0], av[u][1]);
    }
    if (ti == q) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        yrow[buf][at(tj, v)] = hi ? make_double2(yv[2][v], yv[3][v]) : make_double2(yv[0][v], yv[1][v]);
    }
  };
  publish(0, 0);
  int bad = 0;
#pragma unroll 1
  for (int j = 0; j < k; j += 2) {
    const int cur = (j >> 1) & 1;
    __syncthreads();
    const double2 c0 = acol[cur][j], c1 = acol[cur][j + 1];  // (a_jj, .), (a_j+1,j, a_j+1,j+1)
    double2 ai[4], ac[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ai[u] = acol[cur][at(ti, u)];
      ac[u] = acol[cur][at(tj, u)];
      y[u] = yrow[cur][at(tj, u)];
    }
    const double p0 = c0.x, r0 = rcp_f64(p0), l = quotient(c1.x, p0, r0), p1 = fma(-l, c1.x, c1.y);
    // uniform: every thread reads the same two pivots
    if (!(p0 > 0.0)) {
      bad = j + 1;
      break;
    }
    if (!(p1 > 0.0)) {
      bad = j + 2;
      break;
    }
    if (t == 0) {
      piv[j] = p0;
      piv[j + 1] = p1;
    }
    const double r1 = rcp_f64(p1);
    double b1[4], y1[4];  // column j + 1 and row j + 1 after pivot j
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      b1[v] = fma(-l, ac[v].x, ac[v].y);
      y1[v] = fma(-l, y[v].x, y[v].y);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = at(ti, u);
      const double f0 = i > j ? -quotient(ai[u].x, p0, r0) : 0.0;                            // rows up to j are final
      const double f1 = i > j + 1 ? -quotient(fma(-l, ai[u].x, ai[u].y), p1, r1) : 0.0;  // ... up to j + 1
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        av[u][v] = fma(f1, b1[v], fma(f0, ac[v].x, av[u][v]));
        yv[u][v] = fma(f1, y1[v], fma(f0, y[v].x, yv[u][v]));
      }
    }
    if (j + 2 < k) publish(cur ^ 1, j + 2);
  }
  if (t == 0) status[b] = bad;
  if (bad) return;
  __syncthreads();
  // X = L^-1 = D^-1/2 Y
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = at(ti, u);
    const double d = i < k ? 1.0 / sqrt(piv[i]) : 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = at(tj, v);
      Xs[i * kSpdPitch + c] = c <= i && i < k ? yv[u][v] * d : 0.0;
    }
  }
  __syncthreads();
  double* Li = linv + (int64_t)b * kk;
  for (int e = t; e < k * k; e += 256) {
    const int r = e / k, cc = e % k;
    Li[e] = Xs[r * kSpdPitch + cc];
    if (linvT32) linvT32[(int64_t)b * kk + e] = (float)Xs[cc * kSpdPitch + r];
  }
  if (inv64 || inv32) {
    // S^-1 = X^T X: thread owns the 4 x 4 block at rows r0.., columns c0..; rows q below the block's
    // first nonzero add exact zeros and are skipped
    const int r0 = 4 * ti, c0 = 4 * tj;
    if (r0 < k && c0 < k) {
      double acc[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) acc[u][w] = 0.0;
#pragma unroll 4
      for (int q = r0 > c0 ? r0 : c0; q < k; ++q) {
        const double* xr = Xs + q * kSpdPitch + r0;
        const double* xc = Xs + q * kSpdPitch + c0;
        const double2 ra = *reinterpret_cast<const double2*>(xr), rb = *reinterpret_cast<const double2*>(xr + 2);
        const double2 ca = *reinterpret_cast<const double2*>(xc), cb = *reinterpret_cast<const double2*>(xc + 2);
        const double rv[4] = {ra.x, ra.y, rb.x, rb.y}, cv[4] = {ca.x, ca.y, cb.x, cb.y};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int w = 0; w < 4; ++w) acc[u][w] = fma(rv[u], cv[w], acc[u][w]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (r0 + u >= k || c0 + w >= k) continue;
          const int64_t e = (int64_t)b * kk + (r0 + u) * k + c0 + w;
          if (inv64) inv64[e] = acc[u][w];
          if (inv32) inv32[e] = (float)acc[u][w];
        }
    }
  }
}

// ------------------------------------------------------------- captured-energy loss
// With S^-1 (k x k), T = U^T G (m x k) and weights w (m): P = T S^-1,
//   f  = sum_i w_i sum_a P[i][a] T[i][a] / sum w      (= tr(S^-1 G^T U W U^T G) / sum w)
//   C1 = -(2 / sum w) diag(w) P          (m x k)  so that  dL/dG = U C1 + G C2
//   C2 =  (2 / sum w) P^T diag(w) P      (k x k)  for the loss L = 1 - f
// One block: two 64^3 products in FP64 from zero-padded LDS tiles, T transposed, each thread a 4 x 4
// block, so a step of the sum is four 16-byte broadcasts against sixteen fmas.  P overwrites S^-1
// once every thread has read it.  k = m = 64: 48.8 us with scalar LDS reads whose rows shared a bank,
// now 13.3 us.
__global__ __launch_bounds__(256) void energy_kernel(int k, int m, const double* __restrict__ Sinv,
                                                     const double* __restrict__ T, const double* __restrict__ w,
                                                     float* __restrict__ C1, float* __restrict__ C2,
                                                     double* __restrict__ loss) {
  __shared__ __align__(16) double Tt[kSpdMax * kSpdPitch];  // T^T: [q][i]
  __shared__ __align__(16) double Ss[kSpdMax * kSpdPitch];  // S^-1 rebuilt symmetric from its lower triangle; P
  __shared__ double ws[kSpdMax];
  __shared__ double red[4];
  const int t = threadIdx.x, ti = t >> 4, tj = t & 15;
  {
    double vt[16], vs[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int e = t + 256 * q, i = e >> 6, j = e & 63;
      const int hi = min(max(i, j), k - 1), lo = min(min(i, j), k - 1);
      vt[q] = T[min(i, m - 1) * k + min(j, k - 1)];
      vs[q] = Sinv[hi * k + lo];
    }
    const double wv = w[min(t, m - 1)];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int e = t + 256 * q, i = e >> 6, j = e & 63;
      Tt[j * kSpdPitch + i] = i < m && j < k ? vt[q] : 0.0;
      Ss[i * kSpdPitch + j] = i < k && j < k ? vs[q] : 0.0;
    }
    if (t < kSpdMax) ws[t] = t < m ? wv : 0.0;
  }
  __syncthreads();
  const double wsum = block_sum<256>(t < m ? ws[t] : 0.0, red);
  const double c = 2.0 / wsum;
  auto load4 = [](const double* p, double (&o)[4]) {
    const double2 x = *reinterpret_cast<const double2*>(p), y = *reinterpret_cast<const double2*>(p + 2);
    o[0] = x.x;
    o[1] = x.y;
    o[2] = y.x;
    o[3] = y.y;
  };
  const int i0 = 4 * ti, a0 = 4 * tj;
  double pv[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) pv[u][v] = 0.0;
#pragma unroll 4
  for (int q = 0; q < k; ++q) {
    double tv[4], sv[4];
    load4(Tt + q * kSpdPitch + i0, tv);
    load4(Ss + q * kSpdPitch + a0, sv);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) pv[u][v] = fma(tv[u], sv[v], pv[u][v]);
  }
  double f = 0.0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + u, a = a0 + v;
      if (i < m && a < k) {
        C1[i * k + a] = (float)(-c * ws[i] * pv[u][v]);
        f = fma(ws[i] * pv[u][v], Tt[a * kSpdPitch + i], f);
      }
    }
  f = block_sum<256>(f, red);  // its barriers also order every read of Ss before the writes below
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) Ss[(i0 + u) * kSpdPitch + a0 + v] = pv[u][v];
  __syncthreads();
  // C2[a][b] = c sum_r (w_r P[r][a]) P[r][b]: thread owns the 4 x 4 block at (i0, a0)
  double acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = 0.0;
#pragma unroll 4
  for (int r = 0; r < m; ++r) {
    double pa[4], pb[4];
    load4(Ss + r * kSpdPitch + i0, pa);
    load4(Ss + r * kSpdPitch + a0, pb);
    const double wr = ws[r];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[u][v] = fma(wr * pa[u], pb[v], acc[u][v]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (i0 + u < k && a0 + v < k) C2[(i0 + u) * k + a0 + v] = (float)(c * acc[u][v]);
  if (t == 0) loss[0] = 1.0 - f / wsum;
}

// ------------------------------------------------------------ pivoted Cholesky
constexpr int kPcRows = 1024;  // rows per block (4 per thread)

__device__ __forceinline__ bool pc_better(float v, int i, float bv, int bi) {
  return v > bv || (v == bv && i < bi);
}

// block argmax of (value, index) with ties to the smaller index; order independent
__device__ __forceinline__ void pc_block_argmax(float v, int i, float* sv, int* si, float* outv, int* outi) {
  for (int off = 32; off >= 1; off >>= 1) {
    const float ov = __shfl_xor(v, off);
    const int oi = __shfl_xor(i, off);
    if (pc_better(ov, oi, v, i)) {
      v = ov;
      i = oi;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sv[wave] = v;
    si[wave] = i;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float bv = sv[0];
    int bi = si[0];
    for (int q = 1; q < 4; ++q)
      if (pc_better(sv[q], si[q], bv, bi)) {
        bv = sv[q];
        bi = si[q];
      }
    *outv = bv;
    *outi = bi;
  }
}

__global__ __launch_bounds__(256) void pc_init_kernel(int n, const float* __restrict__ A, int64_t lda,
                                                      float* __restrict__ d, float* __restrict__ pval,
                                                      int* __restrict__ pidx) {
  __shared__ float sv[4];
  __shared__ int si[4];
  float bv = -INFINITY;
  int bi = 0x7FFFFFFF;
  for (int q = 0; q < kPcRows / 256; ++q) {
    const int i = blockIdx.x * kPcRows + q * 256 + threadIdx.x;
    if (i < n) {
      const float v = A[(int64_t)i * lda + i];
      d[i] = v;
      if (pc_better(v, i, bv, bi)) {
        bv = v;
        bi = i;
      }
    }
  }
  pc_block_argmax(bv, bi, sv, si, pval + blockIdx.x, pidx + blockIdx.x);
}

// pivot j = argmax over the block partials (one wave, fixed order)
__global__ __launch_bounds__(64) void pc_select_kernel(int nparts, const float* __restrict__ pval,
                                                       const int* __restrict__ pidx, int j, int* __restrict__ piv,
                                                       float* __restrict__ dpiv) {
  float bv = -INFINITY;
  int bi = 0x7FFFFFFF;
  for (int p = threadIdx.x; p < nparts; p += 64)
    if (pc_better(pval[p], pidx[p], bv, bi)) {
      bv = pval[p];
      bi = pidx[p];
    }
  for (int off = 32; off >= 1; off >>= 1) {
    const float ov = __shfl_xor(bv, off);
    const int oi = __shfl_xor(bi, off);
    if (pc_better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if (threadIdx.x == 0) {
    piv[j] = bi;
    dpiv[j] = bv;
  }
}

// column j: l_i = (A[p][i] - sum_{q<j} L_q[i] L_q[p]) / sqrt(d_p); d_i -= l_i^2; d_p = 0.
// A pivot with d_p <= 0 (exhausted rank) gives a zero column.
__global__ __launch_bounds__(256) void pc_column_kernel(int n, const float* __restrict__ A, int64_t lda, int j,
                                                        const int* __restrict__ piv,
                                                        const float* __restrict__ dpiv, float* __restrict__ L,
                                                        int64_t ldl, float* __restrict__ d, float* __restrict__ pval,
                                                        int* __restrict__ pidx) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const int p = piv[j];
  const float dp = dpiv[j];
  const bool ok = dp > 0.f && p >= 0 && p < n;
  const float sq = ok ? sqrtf(dp) : 1.f;
  float bv = -INFINITY;
  int bi = 0x7FFFFFFF;
  for (int q = 0; q < kPcRows / 256; ++q) {
    const int i = blockIdx.x * kPcRows + q * 256 + threadIdx.x;
    if (i < n) {
      float l = 0.f;
      if (ok) {
        float acc = A[(int64_t)p * lda + i];
        for (int c = 0; c < j; ++c) acc = fmaf(-L[(int64_t)c * ldl + i], L[(int64_t)c * ldl + p], acc);
        l = acc / sq;
      }
      L[(int64_t)j * ldl + i] = l;
      const float nd = (ok && i == p) ? 0.f : fmaf(-l, l, d[i]);
      d[i] = nd;
      if (pc_better(nd, i, bv, bi)) {
        bv = nd;
        bi = i;
      }
    }
  }
  pc_block_argmax(bv, bi, sv, si, pval + blockIdx.x, pidx + blockIdx.x);
}

// ------------------------------------------------------------------ RBF dense build
__global__ __launch_bounds__(256) void rbf_dense_kernel(int n, int dim, const float* __restrict__ P, int64_t ldp,
                                                        float inv2l2, float* __restrict__ K, int64_t ldk,
                                                        uint16_t* __restrict__ Kb, int64_t ldkb) {
  const int64_t i = blockIdx.x;
  float pi[kMaxIn];
#pragma unroll
  for (int d = 0; d < kMaxIn; ++d) pi[d] = d < dim ? P[i * ldp + d] : 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t j = (int64_t)blockIdx.y * 1024 + q * 256 + threadIdx.x;
    if (j < n) {
      float d2 = 0.f;
#pragma unroll
      for (int d = 0; d < kMaxIn; ++d) {
        if (d < dim) {
          const float df = pi[d] - P[j * ldp + d];
          d2 = fmaf(df, df, d2);
        }
      }
      const float v = expf(-d2 * inv2l2);
      if (K) K[i * ldk + j] = v;
      if (Kb) {
        const uint32_t u = __float_as_uint(v);
        Kb[i * ldkb + j] = (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
      }
    }
  }
}

// ------------------------------------------------------- dense apply, fp64 vectors
constexpr int kF64NB = 8;  // rhs per pass

// Every load is unconditional (rows and columns clamped, the extra terms left out) and
// the x chunk staged once per block for all of its rows: eight waves of four rows share one FP64 copy
// of X[:, c0:c0+512) in LDS; A is streamed with non-temporal 16-byte loads, which need dword
// alignment only, so odd orders and leading dimensions take the same path (12289 x 8: 1616 -> 141 us
// against one column per lane); the last n % 4 columns are added one per lane.
constexpr int kF64Chunk = 512;
constexpr int kF64Waves = 8;
typedef float f64acc_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64acc_d2 __attribute__((ext_vector_type(2), aligned(8)));

__global__ __launch_bounds__(64 * kF64Waves) __attribute__((amdgpu_waves_per_eu(4))) void dense_f64acc_lds_kernel(int n, const float* __restrict__ A,
                                                                         int64_t lda, const double* __restrict__ X,
                                                                         int64_t ldx, double* __restrict__ Y,
                                                                         int64_t ldy, int nb, double scale,
                                                                         double shift) {
  __shared__ double2 xs[kF64NB][kF64Chunk / 2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // rows and their pointers stay scalar
  const int row0 = blockIdx.x * (4 * kF64Waves) + wave * 4;
  double acc[4][kF64NB];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int b = 0; b < kF64NB; ++b) acc[r][b] = 0.0;
  const float* arow[4];  // rows past the last: its copy, never stored
#pragma unroll
  for (int r = 0; r < 4; ++r) arow[r] = A + (int64_t)(row0 + r < n ? row0 + r : n - 1) * lda;
  const int n4 = n & ~3;
  for (int c0 = 0; c0 < n4; c0 += kF64Chunk) {
    const int cn = n4 - c0 < kF64Chunk ? n4 - c0 : kF64Chunk;  // a multiple of 4
    __syncthreads();
    for (int e = threadIdx.x; e < kF64NB * (kF64Chunk / 2); e += 64 * kF64Waves) {
      const int b = e / (kF64Chunk / 2), j2 = e % (kF64Chunk / 2);
      f64acc_d2 v = {0.0, 0.0};
      if (b < nb && 2 * j2 < cn) v = *reinterpret_cast<const f64acc_d2*>(X + (int64_t)b * ldx + c0 + 2 * j2);
      xs[b][j2] = make_double2(v.x, v.y);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kF64Chunk / 256; ++q) {
      const int j = q * 256 + lane * 4;
      const int jc = j < cn ? j : cn - 4;  // clamped: the load stays unconditional
      f64acc_f4 a[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = __builtin_nontemporal_load(reinterpret_cast<const f64acc_f4*>(arow[r] + c0 + jc));
      // no product with zero instead: the row's last entries, read again, need not be finite
      if (j < cn) {
#pragma unroll
        for (int b = 0; b < kF64NB; ++b) {
          const double2 x0 = xs[b][j / 2], x1 = xs[b][j / 2 + 1];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            double t = acc[r][b];
            t = fma((double)a[r][0], x0.x, t);
            t = fma((double)a[r][1], x0.y, t);
            t = fma((double)a[r][2], x1.x, t);
            t = fma((double)a[r][3], x1.y, t);
            acc[r][b] = t;
          }
        }
      }
    }
  }
  if (lane < n - n4) {
#pragma unroll
    for (int b = 0; b < kF64NB; ++b) {
      const double xv = X[(int64_t)(b < nb ? b : 0) * ldx + n4 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r][b] = fma((double)arow[r][n4 + lane], xv, acc[r][b]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int b = 0; b < kF64NB; ++b) {
      const double sum = wave_sum(acc[r][b]);
      const int row = row0 + r;
      if (lane == 0 && row < n && b < nb)
        Y[(int64_t)b * ldy + row] = scale * sum + shift * X[(int64_t)b * ldx + row];
    }
  }
}

}  // namespace

extern "C" {

int64_t ck_mlp_param_count(int32_t din, int32_t dout) {
  if (din < 1 || din > kMaxIn || dout < 1 || dout > kMaxOut) return -1;
  return mlp_layout(din, dout).total;
}

size_t ck_mlp_grad_workspace_bytes(int64_t n, int32_t din, int32_t dout) {
  if (n < 1 || din < 1 || din > kMaxIn || dout < 1 || dout > kMaxOut) return 0;
  return sizeof(float) * (size_t)cdiv(n, kRows) * (size_t)mlp_layout(din, dout).total;
}

int ck_mlp_forward(int64_t n, int32_t din, int32_t dout, const float* X, int64_t ldx, const float* params, float* G,
                   int64_t gsr, int64_t gsc, float* Z1, float* Z2, int64_t ldz, void* stream) {
  if (n < 1 || n > 0x7FFFFFFF || din < 1 || din > kMaxIn || dout < 1 || dout > kMaxOut || !X || !params || !G ||
      ldx < din)
    return CK_ERR_BAD_ARG;
  if ((Z1 == nullptr) != (Z2 == nullptr) || (Z1 && ldz < n)) return CK_ERR_BAD_ARG;
  if (reinterpret_cast<uintptr_t>(params) % 16) return CK_ERR_BAD_ARG;  // weights are staged as float4
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)cdiv(n, kFwdRows));
  if (Z1)
    hipLaunchKernelGGL(mlp_fwd_kernel<true>, grid, dim3(256), 0, s, (int)n, din, dout, X, ldx, params, G, gsr, gsc, Z1,
                       Z2, ldz);
  else
    hipLaunchKernelGGL(mlp_fwd_kernel<false>, grid, dim3(256), 0, s, (int)n, din, dout, X, ldx, params, G, gsr, gsc, Z1,
                       Z2, ldz);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_mlp_backward(int64_t n, int32_t din, int32_t dout, const float* X, int64_t ldx, const float* params,
                    const float* Z1, const float* Z2, int64_t ldz, const float* dG, int64_t dsr, int64_t dsc,
                    float grad_scale, float* grad, void* work, size_t work_bytes, void* stream) {
  if (n < 1 || n > 0x7FFFFFFF || din < 1 || din > kMaxIn || dout < 1 || dout > kMaxOut || !X || !params || !Z1 ||
      !Z2 || !dG || !grad || ldx < din || ldz < n)
    return CK_ERR_BAD_ARG;
  if (reinterpret_cast<uintptr_t>(params) % 16) return CK_ERR_BAD_ARG;  // weights are staged as float4
  if (!work || work_bytes < ck_mlp_grad_workspace_bytes(n, din, dout)) return CK_ERR_WORKSPACE;
  const int nblk = (int)cdiv(n, kRows);
  const int64_t total = mlp_layout(din, dout).total;
  hipStream_t s = (hipStream_t)stream;
  float* part = static_cast<float*>(work);
  const unsigned split = nblk <= 64 ? 4 : nblk <= 128 ? 2 : 1;  // blocks per chunk until they fill the chip
  hipLaunchKernelGGL(mlp_bwd_kernel, dim3(nblk, split), dim3(512), 0, s, (int)n, din, dout, X, ldx, params, Z1, Z2, ldz,
                     dG, dsr, dsc, part);
  hipLaunchKernelGGL(grad_reduce_kernel, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, s, nblk, total,
                     (const float*)part, grad_scale, grad);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_adam_step(int64_t count, float* params, const float* grad, float* m, float* v, float lr, float beta1,
                 float beta2, float eps, int32_t step, void* stream) {
  if (count < 1 || !params || !grad || !m || !v || step < 1) return CK_ERR_BAD_ARG;
  const float bc1 = 1.f - powf(beta1, (float)step);
  const float bc2 = 1.f - powf(beta2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)cdiv(count, 256)), dim3(256), 0, (hipStream_t)stream, count, params,
                     grad, m, v, lr, beta1, beta2, eps, bc1, bc2);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

size_t ck_gram_workspace_bytes(int64_t n, int32_t ka, int32_t kb) {
  if (n < 1 || ka < 1 || kb < 1) return 0;
  return sizeof(double) * (size_t)cdiv(n, gram_rows(n)) * (size_t)ka * (size_t)kb;
}

int ck_gram_f64(int64_t n, int32_t ka, int32_t kb, const float* X, int64_t xsr, int64_t xsc, const float* Y,
                int64_t ysr, int64_t ysc, double* C, void* work, size_t work_bytes, void* stream) {
  if (n < 1 || ka < 1 || kb < 1 || !X || !Y || !C) return CK_ERR_BAD_ARG;
  if (!work || work_bytes < ck_gram_workspace_bytes(n, ka, kb)) return CK_ERR_WORKSPACE;
  const int64_t rows = gram_rows(n);
  const int nch = (int)cdiv(n, rows);
  hipStream_t s = (hipStream_t)stream;
  double* part = static_cast<double*>(work);
  hipLaunchKernelGGL(gram_partials, dim3(nch, (unsigned)cdiv(ka, 32), (unsigned)cdiv(kb, 32)), dim3(256), 0, s, n,
                     rows, ka, kb, X, xsr, xsc, Y, ysr, ysc, part);
  const int64_t count = (int64_t)ka * kb;
  hipLaunchKernelGGL(gram_reduce, dim3((unsigned)cdiv(count, 256)), dim3(256), 0, s, nch, count, (const double*)part,
                     C);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_rows_gemm_f32(int64_t n, int32_t kin, int32_t kout, const float* X, int64_t xsr, int64_t xsc, const float* W,
                     float alpha, float beta, float* Y, int64_t ysr, int64_t ysc, void* stream) {
  if (n < 1 || kin < 1 || kin > kGemmMax || kout < 1 || !X || !W || !Y) return CK_ERR_BAD_ARG;
  hipLaunchKernelGGL(rows_gemm_kernel, dim3((unsigned)cdiv(n, 64), (unsigned)cdiv(kout, 32)), dim3(256), 0,
                     (hipStream_t)stream, n, kin, kout, X, xsr, xsc, W, alpha, beta, Y, ysr, ysc);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_spd_inverse_f64(int32_t batch, int32_t k, const double* A, int64_t lda, int64_t stride, double jitter_rel,
                       double jitter_abs, double* linv, double* inv64, float* inv32, float* linvT32, int32_t* status,
                       void* stream) {
  if (batch < 1 || k < 1 || k > kSpdMax || !A || lda < k || stride < (int64_t)lda * (k - 1) + k || !linv || !status)
    return CK_ERR_BAD_ARG;
  hipLaunchKernelGGL(spd_inv_kernel, dim3(batch), dim3(256), 0, (hipStream_t)stream, k, A, lda, stride, jitter_rel,
                     jitter_abs, linv, inv64, inv32, linvT32, status);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_energy_loss_f64(int32_t k, int32_t m, const double* Sinv, const double* T, const double* w, float* C1,
                       float* C2, double* loss, void* stream) {
  if (k < 1 || k > kSpdMax || m < 1 || m > kSpdMax || !Sinv || !T || !w || !C1 || !C2 || !loss) return CK_ERR_BAD_ARG;
  hipLaunchKernelGGL(energy_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, k, m, Sinv, T, w, C1, C2, loss);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

size_t ck_pivchol_workspace_bytes(int64_t n) {
  if (n < 1) return 0;
  const size_t parts = (size_t)cdiv(n, kPcRows);
  return sizeof(float) * (size_t)n + parts * (sizeof(float) + sizeof(int)) + 16;
}

int ck_pivchol_dense_f32(int64_t n, const float* A, int64_t lda, int32_t rank, float* L, int64_t ldl, int32_t* piv,
                         float* dpiv, void* work, size_t work_bytes, void* stream) {
  if (n < 1 || n > 0x7FFFFFFF || !A || lda < n || rank < 1 || rank > n || !L || ldl < n || !piv || !dpiv)
    return CK_ERR_BAD_ARG;
  if (!work || work_bytes < ck_pivchol_workspace_bytes(n)) return CK_ERR_WORKSPACE;
  const int nparts = (int)cdiv(n, kPcRows);
  float* d = static_cast<float*>(work);
  float* pval = d + n;
  int* pidx = reinterpret_cast<int*>(pval + nparts);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(pc_init_kernel, dim3(nparts), dim3(256), 0, s, (int)n, A, lda, d, pval, pidx);
  for (int j = 0; j < rank; ++j) {
    hipLaunchKernelGGL(pc_select_kernel, dim3(1), dim3(64), 0, s, nparts, (const float*)pval, (const int*)pidx, j,
                       piv, dpiv);
    hipLaunchKernelGGL(pc_column_kernel, dim3(nparts), dim3(256), 0, s, (int)n, A, lda, j, (const int*)piv,
                       (const float*)dpiv, L, ldl, d, pval, pidx);
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_rbf_dense_f32(int64_t n, int32_t dim, const float* P, int64_t ldp, float lengthscale, float* K, int64_t ldk,
                     uint16_t* Kb, int64_t ldkb, void* stream) {
  if (n < 1 || n > 0x7FFFFFFF || dim < 1 || dim > kMaxIn || !P || ldp < dim || !(lengthscale > 0.f) ||
      (!K && !Kb) || (K && ldk < n) || (Kb && ldkb < n))
    return CK_ERR_BAD_ARG;
  if (cdiv(n, 1024) > 65535) return CK_ERR_BAD_ARG;
  const float inv2l2 = 1.f / (2.f * lengthscale * lengthscale);
  hipLaunchKernelGGL(rbf_dense_kernel, dim3((unsigned)n, (unsigned)cdiv(n, 1024)), dim3(256), 0, (hipStream_t)stream,
                     (int)n, dim, P, ldp, inv2l2, K, ldk, Kb, ldkb);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int ck_dense_apply_f64acc(int64_t n, const float* A, int64_t lda, double scale, double shift, int32_t nrhs,
                          const double* X, int64_t ldx, double* Y, int64_t ldy, void* stream) {
  if (n < 1 || n > 0x7FFFFFFF || !A || lda < n || nrhs < 1 || !X || !Y || ldx < n || ldy < n) return CK_ERR_BAD_ARG;
  hipStream_t s = (hipStream_t)stream;
  for (int b0 = 0; b0 < nrhs; b0 += kF64NB) {
    const int nb = nrhs - b0 < kF64NB ? nrhs - b0 : kF64NB;
    hipLaunchKernelGGL(dense_f64acc_lds_kernel, dim3((unsigned)cdiv(n, 4 * kF64Waves)), dim3(64 * kF64Waves), 0, s,
                       (int)n, A, lda, X + (int64_t)b0 * ldx, ldx, Y + (int64_t)b0 * ldy, ldy, nb, scale, shift);
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

}  // extern "C"
