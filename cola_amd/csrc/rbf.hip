// The on-the-fly stationary kernel operator: y = scale * K x + shift * x with
// K_ij = k(|p_i - p_j|), never stored.
//
// Bound by vector issue: an entry costs 2 dim instructions for the squared distance, one
// exponential (and one square root for the Matern families, both quarter rate) and one fma per
// right-hand side, some 25-35 issue slots against no memory traffic to speak of.  So:
//   - dimension and rhs count are template parameters (nothing is padded to 8 of either);
//   - exp is one v_exp_f32 on an argument scaled once: log2(e) and the lengthscale are folded
//     into one constant in FP64, so the argument sees fewer roundings than l, 1/l, sqrt(k)/l * r
//     and the exponential's own range reduction would give it; sqrt is one v_sqrt_f32 (1 ulp).
//     Both take subnormals for zero: four columns at a time are looked over for entries that far
//     out, which then go a longer way together (one maximum an entry, 0 to 5 % of the time);
//   - a lane owns two rows, so a staged point and its x (one or two 16-byte LDS broadcasts) serve
//     two entries; the four waves of a block share the rows and split each staged tile of 256
//     columns, and the columns are also split over blockIdx.y until the grid fills the chip
//     (a workspace holds one partial per column slice, added in slice order).
// Measured, 20000 points in 3-D, Matern 5/2, 4 rhs: 4242 us with one row per lane, 79 blocks and
// the library's expf and sqrtf; now 183 us per call (the transposes and the host included).
#include <type_traits>

#include "common.hpp"
#include "ops_internal.hpp"

using namespace ck;

namespace {

constexpr int kRbfCols = 4;     // columns at a time
constexpr int kRbfTile = 256;   // columns staged per step
constexpr int kRbfRows = 128;   // rows per block: two per lane
constexpr int kRbfMaxDim = 8;
constexpr int kRbfNB = 8;       // rhs per pass
constexpr int kRbfMaxSlices = 32;
// Blocks wanted: twice what the chip holds at once (256 CUs x 8 blocks of four waves), so that the
// last wave of blocks is a small part of the run (case above by wall clock, an earlier form of
// the kernel: 512 blocks 262 us, 1024 240 us, 2048 218 us, 4096 210 us).
constexpr int kRbfBlocks = 4096;

// The stationary kernel of the squared distance d2: FAMILY 0 exp(-d2 / (2 l^2)) (RBF), 1 exp(-r / l)
// (Matern 1/2), 2 (1 + a) exp(-a) with a = sqrt(3) r / l (Matern 3/2), 3 (1 + a + a^2 / 3) exp(-a)
// with a = sqrt(5) r / l (Matern 5/2).  ce: the exponent's factor times -log2(e); ca: a's factor.
template <int FAMILY>
__device__ __forceinline__ float stationary(float d2, float ce, float ca) {
  if (FAMILY == 0) return __builtin_amdgcn_exp2f(ce * d2);
  const float r = __builtin_amdgcn_sqrtf(d2);
  const float e = __builtin_amdgcn_exp2f(ce * r);
  if (FAMILY == 1) return e;
  const float a = ca * r;
  if (FAMILY == 2) return fmaf(a, e, e);
  return fmaf(a, fmaf(a, 1.f / 3.f, 1.f), 1.f) * e;
}

// The same where v_exp_f32 would return zero for a subnormal, or v_sqrt_f32 take one for zero.
template <int FAMILY>
__device__ __forceinline__ float stationary_far(float d2, float ce, float ca) {
  const float r = FAMILY == 0 ? d2 : sqrtf(d2), arg = ce * r, a = ca * r;
  const bool far = arg < -126.f;
  const float e = __builtin_amdgcn_exp2f(far ? arg + 64.f : arg);
  const float f = FAMILY == 0 || FAMILY == 1 ? e
                  : FAMILY == 2              ? fmaf(a, e, e)
                                             : fmaf(a, fmaf(a, 1.f / 3.f, 1.f), 1.f) * e;
  return far ? f * 0x1p-64f : f;
}

// Column slice blockIdx.y of the rows 128 blockIdx.x ..: the finished rows when there is one slice
// (part == nullptr), else part[(slice * NB + b) * n + row].
template <int FAMILY, int DIM, int NB>
__global__ __launch_bounds__(256) void rbf_kernel(int n, int dim, const float* __restrict__ P, int64_t ldp, float ce,
                                                  float ca, const float* __restrict__ X, int64_t ldx,
                                                  float* __restrict__ Y, int64_t ldy, int nbr, float scale,
                                                  float shift, float far2, float* __restrict__ part,
                                                  const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int W = (DIM + NB + 3) / 4 * 4;  // floats per staged column: its point, then its x
  __shared__ float4 tile[kRbfTile * W / 4];
  __shared__ float red[3][NB][kRbfRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i0 = blockIdx.x * kRbfRows + lane, i1 = i0 + 64;
  const int c0 = i0 < n ? i0 : n - 1, c1 = i1 < n ? i1 : n - 1;
  float p0[DIM], p1[DIM], acc0[NB], acc1[NB];
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    p0[d] = d < dim ? P[(int64_t)c0 * ldp + d] : 0.f;
    p1[d] = d < dim ? P[(int64_t)c1 * ldp + d] : 0.f;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) acc0[b] = acc1[b] = 0.f;
  const int T = (n + kRbfTile - 1) / kRbfTile;
  const int t0 = (int)((int64_t)blockIdx.y * T / gridDim.y), t1 = (int)((int64_t)(blockIdx.y + 1) * T / gridDim.y);
  float* flat = reinterpret_cast<float*>(tile);
  // the next tile's column waits in registers while the current one is used
  float pn[DIM], xn[NB];
  auto fetch = [&](int t) {
    const int j = t * kRbfTile + (int)threadIdx.x;
    const int c = j < n ? j : n - 1;  // columns past n are staged but never used
#pragma unroll
    for (int d = 0; d < DIM; ++d) pn[d] = d < dim ? P[(int64_t)c * ldp + d] : 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b) xn[b] = b < nbr ? X[(int64_t)b * ldx + c] : 0.f;
  };
  if (t0 < t1) fetch(t0);
  for (int t = t0; t < t1; ++t) {
    __syncthreads();
#pragma unroll
    for (int d = 0; d < DIM; ++d) flat[threadIdx.x * W + d] = pn[d];
#pragma unroll
    for (int b = 0; b < NB; ++b) flat[threadIdx.x * W + DIM + b] = xn[b];
    __syncthreads();
    if (t + 1 < t1) fetch(t + 1);
    const int left = n - t * kRbfTile - wave * 64;
    const int jn = left < 64 ? left : 64;
    const float4* col = tile + wave * 64 * (W / 4);
    // K columns from jj on; entries whose kernel value is subnormal go the long way, all K together
    auto columns = [&](int jj, auto count) {
      constexpr int K = decltype(count)::value;
      float c[K][W], d0[K], d1[K], most = 0.f;
#pragma unroll
      for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int q = 0; q < W / 4; ++q) {
          const float4 v = col[(jj + k) * (W / 4) + q];
          c[k][4 * q] = v.x;
          c[k][4 * q + 1] = v.y;
          c[k][4 * q + 2] = v.z;
          c[k][4 * q + 3] = v.w;
        }
        d0[k] = d1[k] = 0.f;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const float e0 = p0[d] - c[k][d], e1 = p1[d] - c[k][d];
          d0[k] = fmaf(e0, e0, d0[k]);
          d1[k] = fmaf(e1, e1, d1[k]);
        }
        most = fmaxf(most, fmaxf(d0[k], d1[k]));
      }
      if (__any(most > far2)) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          d0[k] = stationary_far<FAMILY>(d0[k], ce, ca);
          d1[k] = stationary_far<FAMILY>(d1[k], ce, ca);
        }
      } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          d0[k] = stationary<FAMILY>(d0[k], ce, ca);
          d1[k] = stationary<FAMILY>(d1[k], ce, ca);
        }
      }
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          acc0[b] = fmaf(d0[k], c[k][DIM + b], acc0[b]);
          acc1[b] = fmaf(d1[k], c[k][DIM + b], acc1[b]);
        }
    };
    int jj = 0;
    for (; jj + kRbfCols <= jn; jj += kRbfCols) columns(jj, std::integral_constant<int, kRbfCols>());
    for (; jj < jn; ++jj) columns(jj, std::integral_constant<int, 1>());
  }
  if (wave > 0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      red[wave - 1][b][lane] = acc0[b];
      red[wave - 1][b][lane + 64] = acc1[b];
    }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (b >= nbr) break;
    const float s0 = (acc0[b] + red[0][b][lane]) + (red[1][b][lane] + red[2][b][lane]);
    const float s1 = (acc1[b] + red[0][b][lane + 64]) + (red[1][b][lane + 64] + red[2][b][lane + 64]);
    if (part) {
      float* q = part + ((int64_t)blockIdx.y * NB + b) * n;
      if (i0 < n) q[i0] = s0;
      if (i1 < n) q[i1] = s1;
    } else {
      if (i0 < n) Y[(int64_t)b * ldy + i0] = fmaf(shift, X[(int64_t)b * ldx + i0], scale * s0);
      if (i1 < n) Y[(int64_t)b * ldy + i1] = fmaf(shift, X[(int64_t)b * ldx + i1], scale * s1);
    }
  }
}

// y = scale * (the slices' partials, in slice order) + shift * x
__global__ __launch_bounds__(256) void rbf_reduce(int n, int slices, int nb, const float* __restrict__ part,
                                                  const float* __restrict__ X, int64_t ldx, float* __restrict__ Y,
                                                  int64_t ldy, float scale, float shift, const int* __restrict__ done) {
  if (done && *done) return;
  const int i = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
  if (i >= n) return;
  float s = 0.f;
  for (int k0 = 0; k0 < slices; k0 += 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {  // clamped: eight loads in flight, the surplus dropped below
      const int sl = k0 + k < slices ? k0 + k : slices - 1;
      v[k] = part[((int64_t)sl * nb + b) * n + i];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) s += k0 + k < slices ? v[k] : 0.f;
  }
  Y[(int64_t)b * ldy + i] = fmaf(shift, X[(int64_t)b * ldx + i], scale * s);
}

// column slices that fill the chip, at least one staged tile each
inline int rbf_slices(int64_t n) {
  const int64_t rb = cdiv(n, kRbfRows), T = cdiv(n, kRbfTile);
  int64_t s = cdiv(kRbfBlocks, rb);
  if (s > T) s = T;
  if (s > kRbfMaxSlices) s = kRbfMaxSlices;
  return (int)(s < 1 ? 1 : s);
}

template <int FAMILY, int DIM>
void rbf_launch(int nb_t, dim3 grid, hipStream_t s, int n, int dim, const float* P, int64_t ldp, float ce, float ca,
                const float* X, int64_t ldx, float* Y, int64_t ldy, int nbr, float scale, float shift, float far2,
                float* part, const int* done) {
#define CK_RBF(NB_)                                                                                                  \
  hipLaunchKernelGGL((rbf_kernel<FAMILY, DIM, NB_>), grid, dim3(256), 0, s, n, dim, P, ldp, ce, ca, X, ldx, Y, ldy, \
                     nbr, scale, shift, far2, part, done)
  switch (nb_t) {
    case 1: CK_RBF(1); break;
    case 2: CK_RBF(2); break;
    case 4: CK_RBF(4); break;
    default: CK_RBF(8); break;
  }
#undef CK_RBF
}

template <int FAMILY, typename... Args>
void rbf_family(int dim, Args... a) {
  if (dim == 1)
    rbf_launch<FAMILY, 1>(a...);
  else if (dim == 2)
    rbf_launch<FAMILY, 2>(a...);
  else if (dim == 3)
    rbf_launch<FAMILY, 3>(a...);
  else if (dim == 4)
    rbf_launch<FAMILY, 4>(a...);
  else if (dim <= 6)
    rbf_launch<FAMILY, 6>(a...);
  else
    rbf_launch<FAMILY, 8>(a...);
}

}  // namespace

namespace ck {

size_t rbf_workspace_bytes(const ck_op* op, int nrhs) {
  const int S = rbf_slices(op->n);
  return S > 1 ? (size_t)S * (nrhs <= 1 ? 1 : nrhs <= 2 ? 2 : nrhs <= 4 ? 4 : kRbfNB) * op->n * sizeof(float) : 0;
}

// Without (enough) workspace the columns are not split over blocks.
int rbf_apply(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, void* work,
              size_t work_bytes, const int* done, hipStream_t s) {
  if (!op->a || op->dim < 1 || op->dim > kRbfMaxDim || op->lda < op->dim || !(op->aux_f > 0.f) || op->rank < 0 ||
      op->rank > 3)
    return CK_ERR_BAD_ARG;
  const int n = op->n, fam = op->rank;
  const double l = (double)op->aux_f, log2e = 1.4426950408889634;
  const double root = fam == 2 ? sqrt(3.0) : fam == 3 ? sqrt(5.0) : 1.0;
  const float ce = (float)(fam == 0 ? -log2e / (2.0 * l * l) : -log2e * root / l), ca = (float)(root / l);
  // squared distance from which on an exponential may be subnormal (below 2^-126, and a margin for the
  // rounding of either side); all where the distances themselves may be
  const double reach = fam == 0 ? sqrt(125.5 / -(double)ce) : 125.5 / -(double)ce;
  const float far2 = reach < 1e-16 ? -1.f : (float)(reach * reach);
  const float* P = static_cast<const float*>(op->a);
  const int S = rbf_slices(n);
  for (int b0 = 0; b0 < nrhs; b0 += kRbfNB) {
    const int nb = nrhs - b0 < kRbfNB ? nrhs - b0 : kRbfNB;
    const int nb_t = nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8;
    const bool split = S > 1 && work && work_bytes >= (size_t)S * nb_t * n * sizeof(float);
    float* part = split ? static_cast<float*>(work) : nullptr;
    const dim3 grid((unsigned)cdiv(n, kRbfRows), split ? S : 1);
    const float* Xb = X + b0 * ldx;
    float* Yb = Y + b0 * ldy;
    switch (fam) {
      case 0:
        rbf_family<0>(op->dim, nb_t, grid, s, n, (int)op->dim, P, op->lda, ce, ca, Xb, ldx, Yb, ldy, nb, op->scale,
                      op->shift, far2, part, done);
        break;
      case 1:
        rbf_family<1>(op->dim, nb_t, grid, s, n, (int)op->dim, P, op->lda, ce, ca, Xb, ldx, Yb, ldy, nb, op->scale,
                      op->shift, far2, part, done);
        break;
      case 2:
        rbf_family<2>(op->dim, nb_t, grid, s, n, (int)op->dim, P, op->lda, ce, ca, Xb, ldx, Yb, ldy, nb, op->scale,
                      op->shift, far2, part, done);
        break;
      default:
        rbf_family<3>(op->dim, nb_t, grid, s, n, (int)op->dim, P, op->lda, ce, ca, Xb, ldx, Yb, ldy, nb, op->scale,
                      op->shift, far2, part, done);
        break;
    }
    if (split)
      hipLaunchKernelGGL(rbf_reduce, dim3((unsigned)cdiv(n, 256), nb), dim3(256), 0, s, n, S, nb_t, (const float*)part,
                         Xb, ldx, Yb, ldy, op->scale, op->shift, done);
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

}  // namespace ck
