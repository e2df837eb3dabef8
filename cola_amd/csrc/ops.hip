// Operator kernels: y = scale * S x + shift * x on column blocks.
//
//   dense  : each wavefront owns ROWS rows; lanes stride the row in float4 chunks,
//            one DPP wave reduction per (row, rhs).            [HBM / L2 bound]
//   csr    : by the average row: one lane per row up to 8 entries, 4 lanes (8 at eight rhs, 16
//            at one rhs above 64) up to 128, a wave above; rows far longer than their group's
//            share by the whole wave; int32 column indices. [HBM; bound by the gathers where
//            columns scatter]
//   kron   : factors of order <= 64, in kron.hip (64^3) and kron_any.hip.
#include "common.hpp"
#include "ops_internal.hpp"

using namespace ck;

typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

// ============================================================== dense fp32
// Rows and vectors start at any multiple of four bytes: the hardware takes dword-aligned 16-byte
// loads, so an odd order or leading dimension costs one more cache line per kilobyte of row, not
// four times the load instructions.  The last n % 4 columns are added one per lane.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// One or two rhs: x stays in the caches and every wave reads it for itself.
template <int NB, int ROWS>
__global__ __launch_bounds__(256) void dense_f32_kernel(int n, const float* __restrict__ A, int64_t lda,
                                                        const float* __restrict__ X, int64_t ldx, float* __restrict__ Y,
                                                        int64_t ldy, int nbr, float scale, float shift,
                                                        const int* __restrict__ done) {
  if (done && *done) return;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int row0 = wave * ROWS;
  if (row0 >= n) return;
  float acc[ROWS][NB];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = 0.f;
  const int n4 = n & ~3;
  for (int j = lane * 4; j < n4; j += 256) {
    f4u xv[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) xv[b] = *reinterpret_cast<const f4u*>(X + (b < nbr ? b : 0) * ldx + j);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (row0 + r < n) {
        const f4u a = *reinterpret_cast<const f4u*>(A + (int64_t)(row0 + r) * lda + j);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][b] = fmaf(a[e], xv[b][e], acc[r][b]);
      }
    }
  }
  if (lane < n - n4) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (row0 + r < n) {
        const float a = A[(int64_t)(row0 + r) * lda + n4 + lane];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[r][b] = fmaf(a, X[(b < nbr ? b : 0) * ldx + n4 + lane], acc[r][b]);
      }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float s = wave_sum(acc[r][b]);
      const int row = row0 + r;
      if (lane == 0 && b < nbr && row < n) {
        float y = scale * s;
        if (shift != 0.f) y = fmaf(shift, X[b * ldx + row], y);
        Y[b * ldy + row] = y;
      }
    }
  }
}

// Three and more rhs: the eight waves of a block share one copy of X[:, c0 : c0 + 1024) in LDS instead
// of each wave re-reading it from L2, so per block and chunk the traffic is 8 * ROWS rows of A from HBM
// against one NB x 1024 slice of X.  A is streamed with non-temporal loads (it is read once per product
// and would otherwise evict X and the vectors of the surrounding solver from the caches).  The pieces
// of A and of X that a wave holds are replaced by the next chunk's as soon as they are used, so a
// whole chunk of rows is always in flight.  HBM bound at large n; at small n a launch is latency
// and needs blocks: dense_rows(n) rows each, 8, 16 or 32.
// Measured (before -> now): 20001^2, 4 / 8 / 16 rhs 537 -> 270, 580 -> 292, 947 -> 357 us (odd orders took
// 4-byte loads and re-read x per wave); 16384^2 x 8 167 -> 165 us (6.5 TB/s), x 16 251 -> 219 us;
// 2500^2 x 4 15.2 -> 6.6 us, 8192^2 x 8 62 -> 49 us.
constexpr int kDenseChunk = 1024;
constexpr int kDenseWaves = 8;

// With astride != 0 the launch is batched over blockIdx.y: block row b multiplies its own
// matrix (A + b * astride elements) with its own vectors (X + b * xbs, Y + b * ybs).
template <int NB, int ROWS>
__global__ __launch_bounds__(64 * kDenseWaves) __attribute__((amdgpu_waves_per_eu(4))) void dense_f32_lds_kernel(int n, const float* __restrict__ A,
                                                                         int64_t lda, const float* __restrict__ X,
                                                                         int64_t ldx, float* __restrict__ Y,
                                                                         int64_t ldy, int nbr, float scale,
                                                                         float shift, const int* __restrict__ done,
                                                                         int64_t astride, int64_t xbs, int64_t ybs,
                                                                         float* __restrict__ xy_part = nullptr) {
  if (done && *done) return;
  A += blockIdx.y * astride;
  X += blockIdx.y * xbs;
  Y += blockIdx.y * ybs;
  constexpr int Q = kDenseChunk / 256;                               // pieces of a row per lane and chunk
  constexpr int XQ = (NB * (kDenseChunk / 4) + 64 * kDenseWaves - 1) / (64 * kDenseWaves);  // of X per thread
  __shared__ float4 xs[NB][kDenseChunk / 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // rows and their pointers stay scalar
  const int row0 = blockIdx.x * (kDenseWaves * ROWS) + wave * ROWS;
  const int n4 = n & ~3;
  const float* arow[ROWS];  // rows past the last: its copy, never stored
#pragma unroll
  for (int r = 0; r < ROWS; ++r) arow[r] = A + (int64_t)(row0 + r < n ? row0 + r : n - 1) * lda;
  float acc[ROWS][NB];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = 0.f;
  f4u a[Q][ROWS], xn[XQ];
  auto fetch_a = [&](int c0, int q) {
    const int j = c0 + q * 256 + lane * 4, c = j < n4 ? j : n4 - 4;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) a[q][r] = __builtin_nontemporal_load(reinterpret_cast<const f4u*>(arow[r] + c));
  };
  auto fetch_x = [&](int c0) {
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
      const int e = threadIdx.x + 64 * kDenseWaves * q, b = e / (kDenseChunk / 4), j = c0 + 4 * (e % (kDenseChunk / 4));
      xn[q] = *reinterpret_cast<const f4u*>(X + (int64_t)(b < nbr ? b : 0) * ldx + (j < n4 ? j : n4 - 4));
    }
  };
  // 4 rows x 8 rhs have no registers left to hold the next slice of X: it is loaded where it is stored
  constexpr bool XP = ROWS * NB < 32;
  if (n4 > 0) {
    if (XP) fetch_x(0);
#pragma unroll
    for (int q = 0; q < Q; ++q) fetch_a(0, q);
  }
  for (int c0 = 0; c0 < n4; c0 += kDenseChunk) {
    if (!XP) fetch_x(c0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
      const int e = threadIdx.x + 64 * kDenseWaves * q;
      if (e < NB * (kDenseChunk / 4))
        xs[e / (kDenseChunk / 4)][e % (kDenseChunk / 4)] = make_float4(xn[q][0], xn[q][1], xn[q][2], xn[q][3]);
    }
    __syncthreads();
    const bool more = c0 + kDenseChunk < n4;
    if (XP && more) fetch_x(c0 + kDenseChunk);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (c0 + q * 256 + lane * 4 < n4) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const float4 xv = xs[b][q * 64 + lane];
#pragma unroll
          for (int r = 0; r < ROWS; ++r) {
            float t = acc[r][b];
            t = fmaf(a[q][r][0], xv.x, t);
            t = fmaf(a[q][r][1], xv.y, t);
            t = fmaf(a[q][r][2], xv.z, t);
            t = fmaf(a[q][r][3], xv.w, t);
            acc[r][b] = t;
          }
        }
      }
      if (more) fetch_a(c0 + kDenseChunk, q);
    }
  }
  if (lane < n - n4) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float xv = X[(int64_t)(b < nbr ? b : 0) * ldx + n4 + lane];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) acc[r][b] = fmaf(arow[r][n4 + lane], xv, acc[r][b]);
    }
  }
  // lane L < ROWS * NB owns (row0 + L / NB, rhs L % NB): the wave-wide sums give it Y
  const int my_r = lane / NB, my_b = lane % NB;
  const bool mine = lane < ROWS * NB && my_b < nbr && row0 + my_r < n;
  const bool need_x = shift != 0.f || xy_part != nullptr;
  const float my_x = mine && need_x ? X[(int64_t)my_b * ldx + row0 + my_r] : 0.f;
  float my_y = 0.f;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float sum = wave_sum(acc[r][b]);
      my_y = lane == r * NB + b ? sum : my_y;
    }
  }
  my_y *= scale;
  if (shift != 0.f) my_y = fmaf(shift, my_x, my_y);
  if (mine) Y[(int64_t)my_b * ldy + row0 + my_r] = my_y;
  if (xy_part) {
    // per-block partial sums of X . Y (the CG step's p.Ap), rows then waves in index order
    __shared__ float xys[kDenseWaves][ROWS * NB];
    if (lane < ROWS * NB) xys[wave][lane] = mine ? my_x * my_y : 0.f;
    __syncthreads();
    if (threadIdx.x < nbr) {
      float t = 0.f;
      for (int w = 0; w < kDenseWaves; ++w)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) t += xys[w][r * NB + threadIdx.x];
      xy_part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
  }
}

// One launch of up to 8 rhs (16 without partials): dense_rows(n) rows per block, half of them at 16.
void dense_f32_lds(int n, const float* A, int64_t lda, const float* X, int64_t ldx, float* Y, int64_t ldy, int nb,
                   float scale, float shift, const int* done, float* xy_part, hipStream_t s) {
  const int rows = dense_rows(n) / kDenseWaves;
#define CK_DENSE(NB_, ROWS_)                                                                                        \
  hipLaunchKernelGGL((dense_f32_lds_kernel<NB_, ROWS_>), dim3((unsigned)cdiv(n, kDenseWaves * (ROWS_))),            \
                     dim3(64 * kDenseWaves), 0, s, n, A, lda, X, ldx, Y, ldy, nb, scale, shift, done, (int64_t)0,   \
                     (int64_t)0, (int64_t)0, xy_part)
#define CK_DENSE_ROWS(NB_)  \
  do {                      \
    if (rows == 1)          \
      CK_DENSE(NB_, 1);     \
    else if (rows == 2)     \
      CK_DENSE(NB_, 2);     \
    else                    \
      CK_DENSE(NB_, 4);     \
  } while (0)
  if (nb <= 4)
    CK_DENSE_ROWS(4);
  else if (nb <= 8)
    CK_DENSE_ROWS(8);
  else if (rows == 1)
    CK_DENSE(16, 1);
  else
    CK_DENSE(16, 2);
#undef CK_DENSE_ROWS
#undef CK_DENSE
}

// bf16 stored matrix, fp32 vectors and accumulation (vector path; the MFMA
// path for nrhs >= 4 is in mixed.hip).
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

template <int NB, int ROWS>
__global__ __launch_bounds__(256) void dense_bf16_kernel(int n, const uint16_t* __restrict__ A, int64_t lda,
                                                         const float* __restrict__ X, int64_t ldx, float* __restrict__ Y,
                                                         int64_t ldy, int nbr, float scale, float shift,
                                                         const int* __restrict__ done) {
  if (done && *done) return;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  const int row0 = wave * ROWS;
  if (row0 >= n) return;
  float acc[ROWS][NB];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = 0.f;
  // 8 bf16 (16 bytes) per lane per chunk; requires n % 8 == 0 and lda % 8 == 0 (checked by host)
  for (int j = lane * 8; j < n; j += 512) {
    float4 x0[NB], x1[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b < nbr) {
        x0[b] = *reinterpret_cast<const float4*>(X + b * ldx + j);
        x1[b] = *reinterpret_cast<const float4*>(X + b * ldx + j + 4);
      } else {
        x0[b] = x1[b] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (row0 + r < n) {
        const uint4 w = *reinterpret_cast<const uint4*>(A + (int64_t)(row0 + r) * lda + j);
        const float a0 = bf16_lo(w.x), a1 = bf16_hi(w.x), a2 = bf16_lo(w.y), a3 = bf16_hi(w.y);
        const float a4 = bf16_lo(w.z), a5 = bf16_hi(w.z), a6 = bf16_lo(w.w), a7 = bf16_hi(w.w);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          float s = acc[r][b];
          s = fmaf(a0, x0[b].x, s);
          s = fmaf(a1, x0[b].y, s);
          s = fmaf(a2, x0[b].z, s);
          s = fmaf(a3, x0[b].w, s);
          s = fmaf(a4, x1[b].x, s);
          s = fmaf(a5, x1[b].y, s);
          s = fmaf(a6, x1[b].z, s);
          s = fmaf(a7, x1[b].w, s);
          acc[r][b] = s;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float s = wave_sum(acc[r][b]);
      const int row = row0 + r;
      if (lane == 0 && b < nbr && row < n) {
        float y = scale * s;
        if (shift != 0.f) y = fmaf(shift, X[b * ldx + row], y);
        Y[b * ldy + row] = y;
      }
    }
  }
}

// Multi-rhs product of a bf16 matrix, the vector chunk staged in LDS as in dense_f32_lds_kernel and
// each piece of a row loaded again as soon as it is used.  Requires n % 8 == 0 and 16-byte aligned
// rows; lanes take 8 consecutive columns, whose two halves of X lie 64 apart in LDS, so that 16
// lanes read 256 contiguous bytes (side by side they met in the same banks two by two).  Bound by
// HBM up to 4 rhs, by the VALU (9 instructions an entry) and the LDS reads at 8: 24576 x 4 / 8 / 16
// 187 / 240 / 400 us, without the rolling loads and at 4 rows a wave (2 at 16) 225 / 265 / 450;
// 5000 x 4 / 8 13.6 / 20 against 20 / 26; 16384 x 4 / 16 93 / 215 against 91 / 203.
// v_mfma_f32_16x16x32_bf16 with x in three bf16 terms reads 4.2 TB/s where this does 5 to 6.5, takes
// values below 1e-31 for zero and rounds its sums worse (4.9e-7 against 3.6e-7 at 24576).
typedef float f32x2_nt __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_nt __attribute__((ext_vector_type(4)));

template <int NB, int ROWS>
__global__ __launch_bounds__(64 * kDenseWaves) __attribute__((amdgpu_waves_per_eu(4))) void dense_bf16_lds_kernel(
    int n, const uint16_t* __restrict__ A, int64_t lda, const float* __restrict__ X, int64_t ldx,
    float* __restrict__ Y, int64_t ldy, int nbr, float scale, float shift, const int* __restrict__ done) {
  if (done && *done) return;
  constexpr int Q = kDenseChunk / 512;                               // pieces of a row per lane and chunk
  constexpr int XN = NB * (kDenseChunk / 4);                         // float4 of X per chunk
  __shared__ float4 xs[NB][Q][2][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // rows and their pointers stay scalar
  const int row0 = blockIdx.x * (kDenseWaves * ROWS) + wave * ROWS;
  const uint16_t* arow[ROWS];  // rows past the last: its copy, never stored
#pragma unroll
  for (int r = 0; r < ROWS; ++r) arow[r] = A + (int64_t)(row0 + r < n ? row0 + r : n - 1) * lda;
  float acc[ROWS][NB];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = 0.f;
  u32x4_nt a[Q][ROWS];
  auto fetch_a = [&](int c0, int q) {
    const int j = c0 + q * 512 + lane * 8, c = j < n ? j : n - 8;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) a[q][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_nt*>(arow[r] + c));
  };
#pragma unroll
  for (int q = 0; q < Q; ++q) fetch_a(0, q);
  for (int c0 = 0; c0 < n; c0 += kDenseChunk) {
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < XN; e0 += 64 * kDenseWaves) {
      const int e = e0 + threadIdx.x, b = e / (kDenseChunk / 4), j4 = e % (kDenseChunk / 4);
      if (XN % (64 * kDenseWaves) == 0 || e < XN)
        xs[b][j4 / 128][j4 % 2][j4 / 2 % 64] = (b < nbr && c0 + 4 * j4 < n)
                                                   ? *reinterpret_cast<const float4*>(X + (int64_t)b * ldx + c0 + 4 * j4)
                                                   : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    const bool more = c0 + kDenseChunk < n;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (c0 + q * 512 + lane * 8 < n) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const float4 x0 = xs[b][q][0][lane], x1 = xs[b][q][1][lane];
#pragma unroll
          for (int r = 0; r < ROWS; ++r) {
            float t = acc[r][b];
            t = fmaf(bf16_lo(a[q][r][0]), x0.x, t);
            t = fmaf(bf16_hi(a[q][r][0]), x0.y, t);
            t = fmaf(bf16_lo(a[q][r][1]), x0.z, t);
            t = fmaf(bf16_hi(a[q][r][1]), x0.w, t);
            t = fmaf(bf16_lo(a[q][r][2]), x1.x, t);
            t = fmaf(bf16_hi(a[q][r][2]), x1.y, t);
            t = fmaf(bf16_lo(a[q][r][3]), x1.z, t);
            t = fmaf(bf16_hi(a[q][r][3]), x1.w, t);
            acc[r][b] = t;
          }
        }
      }
      if (more) fetch_a(c0 + kDenseChunk, q);
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float sum = wave_sum(acc[r][b]);
      const int row = row0 + r;
      if (lane == 0 && b < nbr && row < n) {
        float y = scale * sum;
        if (shift != 0.f) y = fmaf(shift, X[(int64_t)b * ldx + row], y);
        Y[(int64_t)b * ldy + row] = y;
      }
    }
  }
}

// ---------------------------------------------------------------- symmetric dense fp32
// Y = scale * A X + shift * X for a symmetric A reading only the 128-column strips on and
// above the diagonal: half the matrix bytes of the full product.  The upper part is cut
// into units of 64 rows x 128 columns, strip by strip (strip J: units s = 0 .. 2J+1, rows
// 64s .. 64s+63, columns 128J .. 128J+127; s >= 2J is the diagonal block), and the units are
// split evenly over a persistent grid of three blocks per CU.  Each wave of a block takes
// 16 rows of a unit (lane l: columns 2l, 2l+1 of every row):
//   column sums (K^T x for the rows' x: the block's mirror image below the diagonal) on the
//   VALU, accumulated over the block's consecutive units of one strip in registers and
//   summed over the four waves when the strip ends;
//   row sums (K x for the strip's x) on v_mfma_f32_16x16x4f32 from the wave's own 16 rows
//   staged in LDS (lane = row l % 16, four columns at 4 (l / 16)), written per unit.
// Diagonal units compute row sums over the whole 128 x 128 block and no column sums.
// dense_sym_reduce then adds, per 64 rows, the row sums of every strip to the right and the
// column sums of the rows above, in a fixed order (bit-reproducible).
constexpr int kSymCols = 128;
constexpr int kSymKs4 = 33;  // LDS row stride of a wave's 16 x 128 block in float4 (bank padding)
// persistent blocks: three per CU (a fourth block's 39.9 KB of LDS does not fit beside them;
// a grid sized for four left a tail of a quarter of the blocks: 143 against 126 us at 8 rhs)
constexpr int kSymGrid = 768;
constexpr int kSymNB = 8;    // rhs per pass

__host__ __device__ inline int64_t sym_strip_start(int64_t J) { return J * (J + 1); }
__host__ __device__ inline int64_t sym_units(int64_t nJ) { return sym_strip_start(nJ); }
__host__ __device__ inline int64_t sym_lo(int64_t w, int64_t U, int G) { return w * U / G; }
// block whose unit range holds unit u: the largest w with sym_lo(w) <= u
__host__ __device__ inline int sym_block_of(int64_t u, int64_t U, int G) { return (int)(((u + 1) * G - 1) / U); }
__host__ __device__ inline int sym_strip_of(int64_t u) {
  int64_t J = (int64_t)((sqrt(4.0 * (double)u + 1.0) - 1.0) * 0.5);
  while (sym_strip_start(J + 1) <= u) ++J;
  while (J > 0 && sym_strip_start(J) > u) --J;
  return (int)J;
}
inline int sym_grid(int64_t U) { return (int)(U < kSymGrid ? U : kSymGrid); }
// strips one block's range can touch: interior strips hold >= 4 units each
inline int sym_slots(int64_t U, int G) { return (int)(((U + G - 1) / G + 3) / 4 + 2); }

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// qr: units x NB x 64 row sums; cp: blocks x mslots x NB x 128 column sums
template <int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void dense_sym_kernel(
    int n, const float* __restrict__ A, int64_t lda, const float* __restrict__ X, int64_t ldx, int nbr,
    float* __restrict__ qr, float* __restrict__ cp, int mslots, const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ float4 ks4[4 * 16 * kSymKs4];
  __shared__ float4 xs4[8 * 4 * kSymNB];  // [column block][lane / 16][rhs]: x at 4 consecutive columns
  __shared__ float xis[4][16][kSymNB];    // per wave: x at its 16 rows, rhs fastest
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t U = sym_units(n / kSymCols);
  const int G = gridDim.x, w = blockIdx.x;
  const int64_t lo = sym_lo(w, U, G), hi = sym_lo(w + 1, U, G);
  if (lo >= hi) return;
  const int Jlo = sym_strip_of(lo);
  float* ksw = reinterpret_cast<float*>(ks4 + wv * 16 * kSymKs4);
  const int r16 = lane & 15, g = lane >> 4;
  float accz[2][NB];  // column sums at columns 2 lane, 2 lane + 1
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b) accz[t][b] = 0.f;
  bool have = false;
  int curJ = -1;
  // the unit's rows as loaded and x at (row lane % 16, rhs lane / 16 and lane / 16 + 4); the
  // next unit's loads are issued as soon as the rows are in LDS
  float2 kr[16];
  float xv[2];
  // units are walked in order, so their strips follow from integer compares (no square root
  // per unit)
  auto load_unit = [&](int64_t u, int J) {
    const int64_t s = u - sym_strip_start(J);
    const float* base = A + (64 * s + 16 * wv) * lda + (int64_t)J * kSymCols + 2 * lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x2_nt v = __builtin_nontemporal_load(reinterpret_cast<const f32x2_nt*>(base + i * lda));
      kr[i] = make_float2(v.x, v.y);
    }
    // x at the rows, loaded for every unit (diagonal ones do not use it) and masked where it is
    // used: a load behind a branch, or a select right after it, makes the wave wait for all of
    // its loads -- the next unit's rows included -- before the row-sum phase
    const int64_t r = 64 * s + 16 * wv + r16;
    const int b0 = g < nbr ? g : 0, b1 = g + 4 < nbr ? g + 4 : 0;  // clamped rhs
    xv[0] = X[(int64_t)b0 * ldx + r];
    xv[1] = X[(int64_t)b1 * ldx + r];
  };
  auto flush = [&](int slot) {
    __syncthreads();  // every wave is past its row sums: ks4 is free
    float* red = reinterpret_cast<float*>(ks4);
#pragma unroll
    for (int b = 0; b < NB; ++b)
      *reinterpret_cast<float2*>(red + (wv * NB + b) * kSymCols + 2 * lane) = make_float2(accz[0][b], accz[1][b]);
    __syncthreads();
    if (slot < mslots) {
      for (int e = threadIdx.x; e < NB * kSymCols; e += 256) {
        const int b = e / kSymCols, c = e % kSymCols;
        if (b < nbr)
          cp[((int64_t)(w * mslots + slot) * NB + b) * kSymCols + c] =
              ((red[(0 * NB + b) * kSymCols + c] + red[(1 * NB + b) * kSymCols + c]) +
               red[(2 * NB + b) * kSymCols + c]) + red[(3 * NB + b) * kSymCols + c];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) accz[t][b] = 0.f;
  };
  int J = Jlo;
  load_unit(lo, J);
  for (int64_t u = lo; u < hi; ++u) {
    while (sym_strip_start(J + 1) <= u) ++J;
    const int64_t s = u - sym_strip_start(J);
    const bool diag = s >= 2 * (int64_t)J;
    if (have && (J != curJ || diag)) {
      flush(curJ - Jlo);
      have = false;
    }
    if (J != curJ) {
      __syncthreads();  // the previous strip's x is no longer read
      for (int e = threadIdx.x; e < 8 * 4 * kSymNB; e += 256) {
        const int r = e % kSymNB, gg = (e / kSymNB) % 4, cb = e / (4 * kSymNB);
        xs4[e] = r < nbr ? *reinterpret_cast<const float4*>(X + (int64_t)r * ldx + (int64_t)J * kSymCols + cb * 16 +
                                                             4 * gg)
                         : make_float4(0.f, 0.f, 0.f, 0.f);
      }
      __syncthreads();
      curJ = J;
    }
    if (!diag) {
      // column sums; the rows' x values go through LDS and come back wave-uniform
      if (g < NB) xis[wv][r16][g] = g < nbr ? xv[0] : 0.f;
      if (g + 4 < NB) xis[wv][r16][g + 4] = g + 4 < nbr ? xv[1] : 0.f;
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float xr[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) xr[b] = xis[wv][i][b];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          accz[0][b] = fmaf(kr[i].x, xr[b], accz[0][b]);
          accz[1][b] = fmaf(kr[i].y, xr[b], accz[1][b]);
        }
      }
      have = true;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) *reinterpret_cast<float2*>(ksw + i * 4 * kSymKs4 + 2 * lane) = kr[i];
    wave_lds_sync();
    if (u + 1 < hi) load_unit(u + 1, sym_strip_start(J + 1) <= u + 1 ? J + 1 : J);
    // row sums: D[row][rhs] += K[row][c] x[c][rhs] over the strip's 8 column blocks
    floatx4 d0 = {0.f, 0.f, 0.f, 0.f}, d1 = {0.f, 0.f, 0.f, 0.f};
    const float4* ksr = reinterpret_cast<const float4*>(ksw) + r16 * kSymKs4 + g;
    // column j of D depends only on column j of B: lanes r16 >= 8 read another rhs's x (an
    // unconditional read) and fill columns that are never stored
    const float4* xsr = xs4 + g * kSymNB + (r16 & (kSymNB - 1));
#pragma unroll
    for (int cb = 0; cb < 8; cb += 2) {
      const float4 a0 = ksr[cb * 4];
      const float4 a1 = ksr[(cb + 1) * 4];
      const float4 b0 = xsr[cb * 4 * kSymNB];
      const float4 b1 = xsr[(cb + 1) * 4 * kSymNB];
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.x, b0.x, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.x, b1.x, d1, 0, 0, 0);
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.y, b0.y, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.y, b1.y, d1, 0, 0, 0);
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.z, b0.z, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.z, b1.z, d1, 0, 0, 0);
      d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0.w, b0.w, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1.w, b1.w, d1, 0, 0, 0);
    }
    // lane (g, r16) holds rows 4g .. 4g+3 of the wave's 16 for rhs r16
    if (r16 < nbr)
      *reinterpret_cast<float4*>(qr + (u * NB + r16) * 64 + 16 * wv + 4 * g) =
          make_float4(d0[0] + d1[0], d0[1] + d1[1], d0[2] + d1[2], d0[3] + d1[3]);
    wave_lds_sync();  // the rows are read before the next unit overwrites them
  }
  if (have) flush(curJ - Jlo);
}

// one block per 64 rows (sub-tile s of strip s / 2).  Wave q of eight sums the row sums of
// strips Ji + q, Ji + q + 8, ... (four strips' loads per batch, all rhs at once) and the column
// sums of every eighth block that covered strip Ji above the diagonal; then wave q takes rhs q:
// the eight waves' sums in order, the epilogue and the X . Y partials.
constexpr int kSymRedWaves = 8;
template <int NB>
__global__ __launch_bounds__(64 * kSymRedWaves) void dense_sym_reduce(int n, const float* __restrict__ X, int64_t ldx,
                                                        float* __restrict__ Y, int64_t ldy, int nbr, float scale,
                                                        float shift, const float* __restrict__ qr,
                                                        const float* __restrict__ cp, int mslots, int G,
                                                        const int* __restrict__ done, float* __restrict__ xy_part) {
  if (done && *done) return;
  __shared__ float red[kSymRedWaves][NB][64];
  const int s = blockIdx.x, nJ = n / kSymCols, Ji = s / 2;
  const int64_t U = sym_units(nJ);
  const int il = threadIdx.x & 63, q = threadIdx.x >> 6;
  float acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = 0.f;
  for (int J0 = Ji + q; J0 < nJ; J0 += 4 * kSymRedWaves) {
    float t[4][NB];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int J = J0 + kSymRedWaves * k < nJ ? J0 + kSymRedWaves * k : nJ - 1;  // clamped: unconditional load
      const float* src = qr + (sym_strip_start(J) + s) * NB * 64 + il;
#pragma unroll
      for (int b = 0; b < NB; ++b) t[k][b] = src[b * 64];
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float v0 = J0 < nJ ? t[0][b] : 0.f, v1 = J0 + kSymRedWaves < nJ ? t[1][b] : 0.f;
      const float v2 = J0 + 2 * kSymRedWaves < nJ ? t[2][b] : 0.f;
      const float v3 = J0 + 3 * kSymRedWaves < nJ ? t[3][b] : 0.f;
      acc[b] += (v0 + v1) + (v2 + v3);
    }
  }
  // column sums of the blocks wf + q, wf + q + 4, ... that covered strip Ji above the diagonal
  if (Ji > 0) {
    const int wf = sym_block_of(sym_strip_start(Ji), U, G);
    const int wl = sym_block_of(sym_strip_start(Ji) + 2 * (int64_t)Ji - 1, U, G);
    for (int w = wf + q; w <= wl; w += kSymRedWaves) {
      const int slot = Ji - sym_strip_of(sym_lo(w, U, G));
      const float* src =
          cp + ((int64_t)(w * mslots + (slot < mslots ? slot : 0)) * NB) * kSymCols + 64 * (s % 2) + il;
      float t[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) t[b] = src[b * kSymCols];
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] += slot < mslots ? t[b] : 0.f;
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) red[q][b][il] = acc[b];
  __syncthreads();
  const int64_t row = 64 * (int64_t)s + il;
  for (int b = q; b < NB; b += kSymRedWaves) {
    if (b >= nbr) break;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kSymRedWaves; ++w) sum += red[w][b][il];
    const float x = X[(int64_t)b * ldx + row];
    float y = scale * sum;
    if (shift != 0.f) y = fmaf(shift, x, y);
    Y[(int64_t)b * ldy + row] = y;
    if (xy_part) {
      // two partials of 32 rows each
      float v = x * y;
      v += dpp_f32<0xB1>(v);
      v += dpp_f32<0x4E>(v);
      v += dpp_f32<0x124>(v);
      v += dpp_f32<0x128>(v);
      // read the lanes before the branch: the last add must not move under the lane test
      const float h0 = readlane_f32(v, 0) + readlane_f32(v, 16);
      const float h1 = readlane_f32(v, 32) + readlane_f32(v, 48);
      if (il == 0) {
        // dense_xy_nparts(n) slots, 64 / dense_rows(n) of them per block: what is left over is zero
        const int per = 64 / dense_rows(n);
        float* dst = xy_part + ((int64_t)b * (n / 64) + s) * per;
        dst[0] = h0;
        dst[1] = h1;
        for (int k = 2; k < per; ++k) dst[k] = 0.f;
      }
    }
  }
}

// scratch of the symmetric product, for up to kSymNB rhs per pass
size_t sym_scratch_bytes(int64_t n) {
  const int64_t U = sym_units(n / kSymCols);
  const int G = sym_grid(U);
  const size_t q = (size_t)U * kSymNB * 64 * sizeof(float), c = (size_t)G * sym_slots(U, G) * kSymNB * kSymCols * 4;
  return (q + 255) / 256 * 256 + (c + 255) / 256 * 256;
}

bool sym_eligible(const ck_op* op, const float* X, int64_t ldx, size_t avail) {
  auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int64_t n = op->n;
  return op->kind == CK_OP_DENSE_F32 && (op->flags & CK_OP_SYMMETRIC) && n >= kSymCols && n % kSymCols == 0 &&
         op->lda % 4 == 0 && ldx % 4 == 0 && al16(op->a) && al16(X) && avail >= sym_scratch_bytes(n);
}

// Y = op(X) through the symmetric kernels, in passes of up to eight rhs; scratch is the
// workspace past dense_sym_offset.  xy_part (optional, nrhs <= 8): dense_xy_nparts(n)
// partials of X . Y per rhs.
int dense_sym_apply(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, const int* done,
                    void* scratch, float* xy_part, hipStream_t s) {
  const int n = op->n;
  const int64_t U = sym_units(n / kSymCols);
  const int G = sym_grid(U), ms = sym_slots(U, G);
  const size_t qb = ((size_t)U * kSymNB * 64 * sizeof(float) + 255) / 256 * 256;
  float* qr = static_cast<float*>(scratch);
  float* cp = reinterpret_cast<float*>(static_cast<char*>(scratch) + qb);
  const float* A = static_cast<const float*>(op->a);
  for (int b0 = 0; b0 < nrhs; b0 += kSymNB) {
    const int nb = nrhs - b0 < kSymNB ? nrhs - b0 : kSymNB;
    const float* Xb = X + b0 * ldx;
    float* Yb = Y + b0 * ldy;
    float* xyb = xy_part && nrhs <= kSymNB ? xy_part : nullptr;
#define CK_SYM(NB_)                                                                                              \
  do {                                                                                                           \
    hipLaunchKernelGGL((dense_sym_kernel<NB_>), dim3(G), dim3(256), 0, s, n, A, op->lda, Xb, ldx, nb, qr, cp,  \
                       ms, done);                                                                                \
    hipLaunchKernelGGL((dense_sym_reduce<NB_>), dim3(n / 64), dim3(64 * kSymRedWaves), 0, s, n, Xb, ldx, Yb, ldy, nb, \
                       op->scale, op->shift, (const float*)qr, (const float*)cp, ms, G, done, xyb);              \
  } while (0)
    if (nb <= 1)
      CK_SYM(1);
    else if (nb <= 2)
      CK_SYM(2);
    else if (nb <= 4)
      CK_SYM(4);
    else
      CK_SYM(8);
#undef CK_SYM
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

int dense_dispatch(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, const int* done,
                   void* work, size_t work_bytes, hipStream_t s) {
  const size_t off = dense_sym_offset(op->n, nrhs);
  if (work && work_bytes > off && sym_eligible(op, X, ldx, work_bytes - off))
    return dense_sym_apply(op, nrhs, X, ldx, Y, ldy, done, static_cast<char*>(work) + off, nullptr, s);
  const int n = op->n;
  if (op->kind == CK_OP_DENSE_F32) {
    const float* A = static_cast<const float*>(op->a);
    for (int b0 = 0; b0 < nrhs; b0 += 16) {
      const int nb = nrhs - b0 < 16 ? nrhs - b0 : 16;
      const float* Xb = X + b0 * ldx;
      float* Yb = Y + b0 * ldy;
      if (nb == 1)
        hipLaunchKernelGGL((dense_f32_kernel<1, 1>), dim3((n + 3) / 4), dim3(256), 0, s, n, A, op->lda, Xb, ldx, Yb, ldy,
                           nb, op->scale, op->shift, done);
      else if (nb == 2)
        hipLaunchKernelGGL((dense_f32_kernel<2, 2>), dim3((n + 7) / 8), dim3(256), 0, s, n, A, op->lda, Xb, ldx, Yb, ldy,
                           nb, op->scale, op->shift, done);
      else
        dense_f32_lds(n, A, op->lda, Xb, ldx, Yb, ldy, nb, op->scale, op->shift, done, nullptr, s);
    }
    CK_CHECK_LAUNCH();
    return CK_OK;
  }
  const uint16_t* A = static_cast<const uint16_t*>(op->a);
  auto aligned16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  // uint4 / float4 loads need 16-byte aligned rows and vector starts
  if ((n % 8) || (op->lda % 8) || (ldx % 4) || !aligned16(op->a) || !aligned16(X)) return CK_ERR_UNSUPPORTED;
  for (int b0 = 0; b0 < nrhs; b0 += 16) {
    const int nb = nrhs - b0 < 16 ? nrhs - b0 : 16;
    const float* Xb = X + b0 * ldx;
    float* Yb = Y + b0 * ldy;
#define CK_DENSE_LDS(NB_, ROWS_)                                                                                  \
  hipLaunchKernelGGL((dense_bf16_lds_kernel<NB_, ROWS_>), dim3((unsigned)cdiv(n, kDenseWaves * (ROWS_))),         \
                     dim3(64 * kDenseWaves), 0, s, n, A, op->lda, Xb, ldx, Yb, ldy, nb, op->scale, op->shift, done)
#define CK_DENSE_LAUNCH(NB_, ROWS_)                                                                              \
  hipLaunchKernelGGL((dense_bf16_kernel<NB_, ROWS_>), dim3((unsigned)cdiv(n, 4 * (ROWS_))), dim3(256), 0, s, n, A, \
                     op->lda, Xb, ldx, Yb, ldy, nb, op->scale, op->shift, done)
    // Rows per wave.  A round of resident blocks takes 16384 rows at 4 rows a wave (2 blocks a CU) and
    // 12288 at 2 (3 blocks); the fewer rows' worth of rounds wins: 14336 x 8 84 us at 4 rows, 118 at 2;
    // 18432 x 8 185 and 165.  One row where that fills the chip better: 8192 x 4 24 us, 31 at two rows.
    auto rounds = [&](int64_t cap) { return cdiv(n, cap) * cap; };
    const int rows = n <= (nb <= 4 ? 8192 : 2048) ? 1 : nb <= 8 && rounds(16384) < rounds(12288) ? 4 : 2;
#define CK_DENSE_ROWS(NB_)  \
  do {                      \
    if (rows == 1)          \
      CK_DENSE_LDS(NB_, 1); \
    else if (rows == 2)     \
      CK_DENSE_LDS(NB_, 2); \
    else                    \
      CK_DENSE_LDS(NB_, 4); \
  } while (0)
    // One and two rhs: straight from cache while the 256 MB last level holds the matrix (10000: 31 us, 33
    // staged), staged above it (24576: 246 us, 187 staged).
    const bool cached = 2 * (int64_t)n * op->lda <= (int64_t)256 << 20;
    if (nb == 1 && cached)
      CK_DENSE_LAUNCH(1, 1);
    else if (nb == 2 && cached)
      CK_DENSE_LAUNCH(2, 2);
    else if (nb == 1)
      CK_DENSE_LDS(1, 2);
    else if (nb == 2)
      CK_DENSE_LDS(2, 2);
    else if (nb <= 4)
      CK_DENSE_ROWS(4);
    else if (nb <= 8)
      CK_DENSE_ROWS(8);
    else if (rows == 1)
      CK_DENSE_LDS(16, 1);
    else
      CK_DENSE_LDS(16, 2);
#undef CK_DENSE_ROWS
#undef CK_DENSE_LDS
#undef CK_DENSE_LAUNCH
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

// ============================================================== CSR
// Rows of up to 8 entries on average: one lane per row.  A row of at most eight entries is loaded
// into registers in one batch (column indices and values, then the x gathers of NB vectors), so
// each lane waits for memory twice per NB vectors instead of once per nonzero; the matrix is read
// once for all vectors.  Longer rows go through the same batches NB vectors at a time.  Every row is
// summed k ascending with one fma per nonzero, in both paths, so results do not depend on the path
// or on the vector count.
constexpr int kCsrBatch = 8;

// XY: also xy_part[b * gridDim.x + block] = sum over the block's rows of X[b][row] Y[b][row] (a
// Krylov step's x . Ax from the matvec itself, instead of a separate pass over both vectors).
// The XY launch takes 1024 rows per block, so its partials are as few as a 1024-element tile
// pass would give: every block of the kernel that consumes them reads all of them.
template <int NB, bool XY = false>
__global__ __launch_bounds__(XY ? 1024 : 256) void csr_lane_per_row(int n, const int32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ colind,
                                                        const float* __restrict__ val, const float* __restrict__ X,
                                                        int64_t ldx, float* __restrict__ Y, int64_t ldy, int nrhs,
                                                        float scale, float shift, const int* __restrict__ done,
                                                        float* __restrict__ xy_part) {
  if (done && *done) return;
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (!XY && row >= n) return;
  const int rc = row < n ? row : n - 1;  // XY: rows past n compute a copy of row n - 1 and store nothing
  const int k0 = rowptr[rc], k1 = rowptr[rc + 1];
  const int len = k1 - k0;
  if (len <= kCsrBatch) {
    int c[kCsrBatch];
    float v[kCsrBatch];
#pragma unroll
    for (int i = 0; i < kCsrBatch; ++i) {
      c[i] = i < len ? colind[k0 + i] : rc;
      v[i] = i < len ? val[k0 + i] : 0.f;
    }
    for (int b0 = 0; b0 < nrhs; b0 += NB) {
      float xv[NB][kCsrBatch];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < kCsrBatch; ++i)
          xv[j][i] = (i < len && b0 + j < nrhs) ? X[(int64_t)(b0 + j) * ldx + c[i]] : 0.f;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int b = b0 + j;
        if (b >= nrhs) break;
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < kCsrBatch; ++i)
          if (i < len) acc = fmaf(v[i], xv[j][i], acc);
        float y = scale * acc;
        if (shift != 0.f) y = fmaf(shift, X[(int64_t)b * ldx + rc], y);
        if (!XY || row < n) Y[(int64_t)b * ldy + row] = y;
      }
    }
  } else {
    for (int b0 = 0; b0 < nrhs; b0 += NB) {
      float acc[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j] = 0.f;
      for (int kb = k0; kb < k1; kb += kCsrBatch) {
        int c[kCsrBatch];
        float v[kCsrBatch], xv[NB][kCsrBatch];
#pragma unroll
        for (int i = 0; i < kCsrBatch; ++i) {  // past the row's end: its last entry again, dropped below
          const int k = kb + i < k1 ? kb + i : k1 - 1;
          c[i] = colind[k];
          v[i] = val[k];
        }
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < kCsrBatch; ++i)
            xv[j][i] = X[(int64_t)(b0 + j < nrhs ? b0 + j : b0) * ldx + c[i]];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < kCsrBatch; ++i) acc[j] = kb + i < k1 ? fmaf(v[i], xv[j][i], acc[j]) : acc[j];
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int b = b0 + j;
        if (b >= nrhs) break;
        float y = scale * acc[j];
        if (shift != 0.f) y = fmaf(shift, X[(int64_t)b * ldx + rc], y);
        if (!XY || row < n) Y[(int64_t)b * ldy + row] = y;
      }
    }
  }
  if constexpr (XY) {
    __shared__ float red[16];
    for (int b = 0; b < nrhs; ++b) {
      const float xy = row < n ? X[(int64_t)b * ldx + row] * Y[(int64_t)b * ldy + row] : 0.f;
      const float sum = block_sum<1024>(xy, red);
      if (threadIdx.x == 0) xy_part[(int64_t)b * gridDim.x + blockIdx.x] = sum;
    }
  }
}

// Longer rows: a group of G lanes per row (4, or 8 at eight rhs so that each rhs has a lane to store
// it; a whole wave for rows of more than 128 entries on average).  Lane l of the group takes the
// row's entries l, l + G, ..., U of them per batch: the batch's column indices and values go
// out together, then its gathers of x, so a row costs two dependent memory waits per G * U entries.
// A row of more than kCsrLong batches (a hub among short rows) is taken by the whole wave after its
// other rows: 100 rows of 100000 entries among 400000 of 35 took 2400 / 4740 us at 1 / 4 rhs by their
// groups, 3 to 5 times as long as one wave per row and rhs (684 / 3000); by their waves 411 / 680.
// The sums are added in a fixed order, whether or not xy_part is asked for.
// Bound by the gathers, which land on a cache line of their own where the columns are scattered:
// with several rhs they come from a copy of x with the rhs fastest (csr_interleave, 4-5 us at
// 300000 x 4), one NB-wide load and one line per entry instead of NB.  Measured, 300000 rows of 14.9
// entries, a quarter of them anywhere (36 MB): 1 rhs 69 -> 16 us, 4 rhs 246 -> 32 us (57 without
// the copy), 8 rhs 511 -> 56 us, against one lane per row; 50000 rows of 69 entries anywhere, against one
// wave per row and rhs: 1 rhs 19.2 -> 16.9, 4 rhs 60 -> 27, 8 rhs 117 -> 36 us.  Short regular rows
// (5-point Laplacian, 631000 rows) stay with one lane per row: 7.6 us against 14.6, 4 rhs 12.7
// against 19.4.
constexpr int kCsrLong = 8;  // batches of a group beyond which its wave takes the row

template <int G>
__device__ __forceinline__ float group_sum(float v) {
  if (G == 64) return wave_sum(v);
  v += dpp_f32<0xB1>(v);                // quad_perm [1,0,3,2]
  v += dpp_f32<0x4E>(v);                // quad_perm [2,3,0,1]
  if (G >= 8) v += dpp_f32<0x141>(v);   // row_half_mirror
  if (G >= 16) v += dpp_f32<0x140>(v);  // row_mirror
  return v;
}

// Xt[i * NB + j] = X[j * ldx + i] for the nbr <= NB rhs of a pass, zero beyond them
template <int NB>
__global__ __launch_bounds__(256) void csr_interleave(int n, int nbr, const float* __restrict__ X, int64_t ldx,
                                                      float* __restrict__ Xt, const int* __restrict__ done) {
  if (done && *done) return;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) v[j] = j < nbr ? X[(int64_t)j * ldx + i] : 0.f;
  typedef float vec __attribute__((ext_vector_type(NB < 4 ? NB : 4)));
#pragma unroll
  for (int q = 0; q < NB; q += (NB < 4 ? NB : 4)) {
    vec t;
#pragma unroll
    for (int j = 0; j < (NB < 4 ? NB : 4); ++j) t[j] = v[q + j];
    *reinterpret_cast<vec*>(Xt + (int64_t)i * NB + q) = t;
  }
}

// One pass of nbr <= NB rhs.  Xt: the interleaved x (unused at NB = 1, where X itself is gathered).
template <int G, int NB, int U>
__global__ __launch_bounds__(256) void csr_group_kernel(int n, const int32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ colind,
                                                        const float* __restrict__ val, const float* __restrict__ X,
                                                        int64_t ldx, const float* __restrict__ Xt,
                                                        float* __restrict__ Y, int64_t ldy, int nbr, float scale,
                                                        float shift, int rows, const int* __restrict__ done,
                                                        float* __restrict__ xy_part) {
  static_assert(NB <= G, "one lane of the group stores each rhs");
  if (done && *done) return;
  __shared__ float red[256];
  constexpr int R = 256 / G;  // rows per sweep of the block
  constexpr int V = NB < 4 ? NB : 4;
  typedef float vec __attribute__((ext_vector_type(V)));
  const int l = threadIdx.x % G, g = threadIdx.x / G, lane = threadIdx.x & 63;
  const int row0 = blockIdx.x * rows;
  const bool stores = l < nbr;
  const int lb = stores ? l : 0;  // the rhs this lane stores
  float xy = 0.f;
  for (int r = g; r < rows; r += R) {
    const int row = row0 + r;
    const bool in = row < n;
    const int rc = in ? row : n - 1;
    const int k0 = rowptr[rc], k1 = in ? rowptr[rc + 1] : k0;
    const float xr = X[(int64_t)lb * ldx + rc];
    float acc[NB], odd[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = odd[j] = 0.f;
    // the entries [a, b) from lane `at` of `width`: a batch's products are added on their own, in pairs, and
    // the batches in two chains, so that a lane's sum of 16 or 32 entries errs no more than those of 64 lanes
    auto add = [&](int a, int b, int at, int width) {
      for (int kb = a; kb < b; kb += width * U) {
        int c[U];
        float v[U], x[U][NB];
#pragma unroll
        for (int u = 0; u < U; ++u) {  // past the row's end: its last entry again, dropped below
          const int k = kb + u * width + at, kk = k < b ? k : b - 1;
          c[u] = colind[kk];
          v[u] = val[kk];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (NB == 1) {
            x[u][0] = X[c[u]];
          } else {
#pragma unroll
            for (int q = 0; q < NB; q += V) {
              const vec t = *reinterpret_cast<const vec*>(Xt + (int64_t)c[u] * NB + q);
#pragma unroll
              for (int j = 0; j < V; ++j) x[u][q + j] = t[j];
            }
          }
        }
        // used once, behind a select: the compiler would move the first loads into a branch of their own,
        // another memory wait per batch
#pragma unroll
        for (int u = 0; u < U; ++u) {
          asm("" : "+v"(v[u]));
          if (NB == 1) asm("" : "+v"(x[u][0]));
        }
        float t[U / 2][NB];
#pragma unroll
        for (int u = 0; u < U; u += 2) {
          const bool on0 = kb + u * width + at < b, on1 = kb + (u + 1) * width + at < b;
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const float p = on0 ? v[u] * x[u][j] : 0.f;
            t[u / 2][j] = on1 ? fmaf(v[u + 1], x[u + 1][j], p) : p;
          }
        }
#pragma unroll
        for (int w = U / 4; w >= 1; w /= 2)
#pragma unroll
          for (int u = 0; u < w; ++u)
#pragma unroll
            for (int j = 0; j < NB; ++j) t[u][j] += t[u + w][j];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const float s = odd[j] + t[0][j];
          odd[j] = acc[j];
          acc[j] = s;
        }
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j] += odd[j];
    };
    const bool over = G < 64 && k1 - k0 > kCsrLong * G * U;
    add(k0, over ? k0 : k1, l, G);
    if (G < 64) {  // rows far longer than the others: one at a time by the whole wave
      for (uint64_t left = __ballot(over); left != 0;) {
        const int first = __builtin_ctzll(left);  // lane 0 of a group
        float keep[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          keep[j] = acc[j];
          acc[j] = odd[j] = 0.f;
        }
        add(__builtin_amdgcn_readlane(k0, first), __builtin_amdgcn_readlane(k1, first), lane, 64);
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const float s = wave_sum(acc[j]);
          acc[j] = lane == first ? s : keep[j];
        }
        left &= ~(((1ull << (G % 64)) - 1) << first);
      }
    }
    float mine = 0.f;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const float s = group_sum<G>(acc[j]);
      mine = l == j ? s : mine;
    }
    float y = scale * mine;
    if (shift != 0.f) y = fmaf(shift, xr, y);
    if (stores && in) {
      Y[(int64_t)lb * ldy + row] = y;
      xy = fmaf(xr, y, xy);
    }
  }
  if (xy_part) {
    red[threadIdx.x] = xy;
    __syncthreads();
    if (threadIdx.x < 64) {
      float s = (red[threadIdx.x] + red[threadIdx.x + 64]) + (red[threadIdx.x + 128] + red[threadIdx.x + 192]);
#pragma unroll
      for (int o = G; o < 64; o *= 2) s += __shfl_xor(s, o);
      if ((int)threadIdx.x < nbr) xy_part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = s;
    }
  }
}

inline int csr_pass(int nrhs) { return nrhs <= 1 ? 1 : nrhs <= 2 ? 2 : nrhs <= 4 ? 4 : 8; }
inline size_t csr_xt_bytes(int64_t n, int nrhs) {
  return nrhs > 1 ? (size_t)csr_pass(nrhs) * n * sizeof(float) : 0;
}

int csr_launch(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, void* work,
               size_t work_bytes, const int* done, float* xy_part, hipStream_t s) {
  const int n = op->n;
  if (!op->rowptr || !op->colind || !op->values) return CK_ERR_BAD_ARG;
  if (csr_short_rows(op)) {
    const dim3 grid((unsigned)cdiv(n, xy_part ? 1024 : 256)), blk(xy_part ? 1024 : 256);
#define CK_CSR(NB_)                                                                                                 \
  do {                                                                                                              \
    if (xy_part)                                                                                                    \
      hipLaunchKernelGGL((csr_lane_per_row<NB_, true>), grid, blk, 0, s, n, op->rowptr, op->colind, op->values, X, \
                         ldx, Y, ldy, nrhs, op->scale, op->shift, done, xy_part);                                   \
    else                                                                                                            \
      hipLaunchKernelGGL((csr_lane_per_row<NB_>), grid, blk, 0, s, n, op->rowptr, op->colind, op->values, X, ldx,  \
                         Y, ldy, nrhs, op->scale, op->shift, done, xy_part);                                        \
  } while (0)
    if (nrhs == 1)
      CK_CSR(1);
    else if (nrhs == 2)
      CK_CSR(2);
    else
      CK_CSR(4);
#undef CK_CSR
    CK_CHECK_LAUNCH();
    return CK_OK;
  }
  // One rhs and more than 64 entries a row: 16 lanes a row, one sweep a block (the partials' bound on blocks
  // has no say without partials): 200000 rows of 69 61 us, 73 with 4 lanes, 68 with a wave a row;
  // 150000 of 120 78, 89 and 80.
  const bool wide = nrhs == 1 && !xy_part && !csr_long_rows(op) && (double)op->nnz > 64.0 * (double)n;
  const int rows = wide ? 16 : csr_rows(op);
  const dim3 grid(wide ? (unsigned)cdiv(n, rows) : (unsigned)csr_xy_nparts(op)), blk(256);
  // the interleaved x sits past the partials; without room for it the rhs go one at a time
  const size_t off = csr_xy_bytes(op, nrhs);
  const bool room = work && work_bytes >= off + csr_xt_bytes(n, nrhs);
  float* xt = room ? reinterpret_cast<float*>(static_cast<char*>(work) + off) : nullptr;
  const int step = room ? csr_pass(nrhs) : 1;
  for (int b0 = 0; b0 < nrhs; b0 += step) {
    const int nb = nrhs - b0 < step ? nrhs - b0 : step;
    const float* Xb = X + b0 * ldx;
    float* Yb = Y + b0 * ldy;
    float* xyb = xy_part ? xy_part + (size_t)b0 * grid.x : nullptr;
    const dim3 tg((unsigned)cdiv(n, 256));
#define CK_CSR(G_, NB_, U_)                                                                                        \
  do {                                                                                                             \
    if (NB_ > 1) hipLaunchKernelGGL(csr_interleave<NB_>, tg, blk, 0, s, n, nb, Xb, ldx, xt, done);                  \
    hipLaunchKernelGGL((csr_group_kernel<G_, NB_, U_>), grid, blk, 0, s, n, op->rowptr, op->colind, op->values,    \
                       Xb, ldx, (const float*)xt, Yb, ldy, nb, op->scale, op->shift, rows, done, xyb);             \
  } while (0)
    if (csr_long_rows(op)) {
      if (step == 1)
        CK_CSR(64, 1, 4);
      else if (step == 2)
        CK_CSR(64, 2, 4);
      else if (step == 4)
        CK_CSR(64, 4, 4);
      else
        CK_CSR(64, 8, 2);
    } else {
      if (wide)
        CK_CSR(16, 1, 8);
      else if (step == 1)
        CK_CSR(4, 1, 8);
      else if (step == 2)
        CK_CSR(4, 2, 4);
      else if (step == 4)
        CK_CSR(4, 4, 4);
      else
        CK_CSR(8, 8, 4);
    }
#undef CK_CSR
  }
  CK_CHECK_LAUNCH();
  return CK_OK;
}

}  // namespace

namespace ck {

int csr_apply_xy(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, const int* done,
                 float* xy_part, void* work, size_t work_bytes, hipStream_t s) {
  if (op->kind != CK_OP_CSR_F32 || !xy_part) return CK_ERR_BAD_ARG;
  return csr_launch(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, xy_part, s);
}

}  // namespace ck

namespace {

// ============================================================== diagonal / identity
__global__ __launch_bounds__(256) void diag_kernel(int64_t n, int nrhs, const float* __restrict__ d,
                                                   const float* __restrict__ X, int64_t ldx, float* __restrict__ Y,
                                                   int64_t ldy, float scale, float shift,
                                                   const int* __restrict__ done) {
  if (done && *done) return;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (i >= n || b >= nrhs) return;
  const float x = X[b * ldx + i];
  const float s = d ? d[i] : 1.f;
  Y[b * ldy + i] = fmaf(scale * s, x, shift * x);
}

}  // namespace

// ============================================================== internal API
namespace ck {

// Y = op(X) for a dense fp32 operator with 3..8 rhs on the LDS-staged kernel, writing the
// per-block partial sums of X . Y to xy_part (nrhs x dense_xy_nparts(n), column-major by
// rhs); returns CK_ERR_UNSUPPORTED when the shapes fall outside that kernel
int dense_apply_xy(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, const int* done,
                   float* xy_part, void* work, size_t work_bytes, hipStream_t s) {
  const int n = op->n;
  const size_t off = dense_sym_offset(n, nrhs);
  if (work && work_bytes > off && nrhs >= 1 && nrhs <= 8 && sym_eligible(op, X, ldx, work_bytes - off))
    return dense_sym_apply(op, nrhs, X, ldx, Y, ldy, done, static_cast<char*>(work) + off, xy_part, s);
  if (op->kind != CK_OP_DENSE_F32 || nrhs < 3 || nrhs > 8) return CK_ERR_UNSUPPORTED;
  dense_f32_lds(n, static_cast<const float*>(op->a), op->lda, X, ldx, Y, ldy, nrhs, op->scale, op->shift, done, xy_part,
                s);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

// U of the first pass, then (orders other than 64^3) room for the X . Y partials that a Krylov step
// takes from the second pass's epilogue
size_t kron_workspace_bytes(const ck_op* op, int nrhs) {
  if (op->nfactors != 3) return 0;
  const size_t off = kron_xy_offset(op, nrhs);
  return off == 0 ? (size_t)nrhs * op->n * sizeof(float) : off + (size_t)nrhs * kron_nparts(op) * sizeof(float);
}

size_t kron_xy_offset(const ck_op* op, int nrhs) {
  if (op->fdim[0] == 64 && op->fdim[1] == 64 && op->fdim[2] == 64) return 0;
  return ((size_t)nrhs * op->n * sizeof(float) + 255) / 256 * 256;
}

int kron_dispatch(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, void* work,
                  size_t work_bytes, const int* done, float* partials, int nparts, hipStream_t s) {
  const int d = op->nfactors;
  if (d != 2 && d != 3) return CK_ERR_UNSUPPORTED;
  int64_t prod = 1;
  for (int i = 0; i < d; ++i) {
    if (op->fdim[i] < 1 || op->fdim[i] > 64 || !op->factor[i]) return CK_ERR_UNSUPPORTED;
    prod *= op->fdim[i];
  }
  if (prod != op->n) return CK_ERR_BAD_ARG;
  if (d == 2) {
    if (partials) return CK_ERR_UNSUPPORTED;
    return kron_any_apply(op, nrhs, X, ldx, Y, ldy, nullptr, done, nullptr, 0, s);
  }
  if (work_bytes < (size_t)nrhs * op->n * sizeof(float) || !work) return CK_ERR_WORKSPACE;
  if (kron64_eligible(op, X, ldx, Y, ldy))
    return kron64_apply_f32(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, partials, nparts, s);
  // (64^3 with unaligned vectors or factors: kron_nparts counts kron64_pass_b4's tiles)
  if (partials && (kron_xy_offset(op, nrhs) == 0 || nparts != kron_nparts(op))) return CK_ERR_UNSUPPORTED;
  return kron_any_apply(op, nrhs, X, ldx, Y, ldy, static_cast<float*>(work), done, partials, nparts, s);
}

int kron_nparts(const ck_op* op) {
  if (op->nfactors != 3) return 0;
  const int plane = op->fdim[1] * op->fdim[2];
  return kron_xy_offset(op, 1) == 0 ? plane / 64 : kron_any_nparts(plane);
}

int op_apply_internal(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, void* work,
                      size_t work_bytes, const int* done, hipStream_t s) {
  if (!op || !X || !Y || nrhs < 1 || op->n < 1 || ldx < op->n || ldy < op->n) return CK_ERR_BAD_ARG;
  switch (op->kind) {
    case CK_OP_IDENTITY:
    case CK_OP_DIAG_F32: {
      const float* d = op->kind == CK_OP_DIAG_F32 ? (const float*)op->a : nullptr;
      if (op->kind == CK_OP_DIAG_F32 && !d) return CK_ERR_BAD_ARG;
      dim3 grid((unsigned)cdiv(op->n, 256), nrhs);
      hipLaunchKernelGGL(diag_kernel, grid, dim3(256), 0, s, (int64_t)op->n, nrhs, d, X, ldx, Y, ldy, op->scale,
                         op->shift, done);
      CK_CHECK_LAUNCH();
      return CK_OK;
    }
    case CK_OP_DENSE_F32:
    case CK_OP_DENSE_BF16:
      if (!op->a || op->lda < op->n) return CK_ERR_BAD_ARG;
      return dense_dispatch(op, nrhs, X, ldx, Y, ldy, done, work, work_bytes, s);
    case CK_OP_DENSE_BATCHED_F32: {
      // vector b multiplies matrix b (a + b * nnz elements): independent dense systems of one order
      auto aligned16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
      if (!op->a || op->lda < op->n || op->nnz < (int64_t)op->lda * (op->n - 1) + op->n) return CK_ERR_BAD_ARG;
      if (op->n % 4 || op->lda % 4 || op->nnz % 4 || ldx % 4 || ldy % 4 || !aligned16(op->a) || !aligned16(X))
        return CK_ERR_UNSUPPORTED;
      const int grid = (op->n + kDenseWaves * 4 - 1) / (kDenseWaves * 4);
      hipLaunchKernelGGL((dense_f32_lds_kernel<1, 4>), dim3(grid, nrhs), dim3(64 * kDenseWaves), 0, s, op->n,
                         static_cast<const float*>(op->a), op->lda, X, ldx, Y, ldy, 1, op->scale, op->shift, done,
                         op->nnz, ldx, ldy, nullptr);
      CK_CHECK_LAUNCH();
      return CK_OK;
    }
    case CK_OP_CSR_F32:
      return csr_launch(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, nullptr, s);
    case CK_OP_KRON_F32:
      return kron_dispatch(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, nullptr, 0, s);
    case CK_OP_WOODBURY_INV:
      return woodbury_apply(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, s);
    case CK_OP_RBF_F32:
      return rbf_apply(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, s);
    case CK_OP_KRON_EIG_F32:
      if (!kron64_eligible(op, X, ldx, Y, ldy)) return CK_ERR_UNSUPPORTED;
      return kron64_eig_apply_f32(op, nrhs, X, ldx, Y, ldy, work, work_bytes, done, s);
    default:
      return CK_ERR_UNSUPPORTED;
  }
}

size_t op_workspace_internal(const ck_op* op, int nrhs) {
  if (!op) return 0;
  switch (op->kind) {
    case CK_OP_KRON_F32:
      return kron_workspace_bytes(op, nrhs);
    case CK_OP_WOODBURY_INV:
      return woodbury_workspace_bytes(op, nrhs);
    case CK_OP_KRON_EIG_F32:
      return 2 * (size_t)nrhs * op->n * sizeof(float);
    case CK_OP_DENSE_F32:
      // a symmetric operator's product reads half the matrix through scratch placed past the
      // regions CG's fused steps use (dense_sym_offset)
      if ((op->flags & CK_OP_SYMMETRIC) && op->n >= kSymCols && op->n % kSymCols == 0)
        return dense_sym_offset(op->n, nrhs) + sym_scratch_bytes(op->n);
      // room for the p.Ap partials a CG step takes from the matvec epilogue (dense_apply_xy)
      return (nrhs >= 3 && nrhs <= 8) ? dense_xy_bytes(op->n, nrhs) : 0;
    case CK_OP_RBF_F32:
      return rbf_workspace_bytes(op, nrhs);
    case CK_OP_CSR_F32:
      // the x.Ax partials of csr_apply_xy (CG's p.Ap, Lanczos's v.Av), then the interleaved x
      return csr_xy_bytes(op, nrhs) + (csr_short_rows(op) ? 0 : csr_xt_bytes(op->n, nrhs));
    default:
      return 0;
  }
}

}  // namespace ck

// ============================================================== transpose / dot
namespace {

__global__ __launch_bounds__(256) void transpose_kernel(int64_t n, int nrhs, const float* __restrict__ src,
                                                        int64_t lds_, float* __restrict__ dst, int64_t ldd,
                                                        int to_blocks) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (to_blocks) {
    for (int b = 0; b < nrhs; ++b) dst[b * ldd + i] = src[i * lds_ + b];
  } else {
    for (int b = 0; b < nrhs; ++b) dst[i * ldd + b] = src[b * lds_ + i];
  }
}

__global__ __launch_bounds__(256) void dot_partials_kernel(int64_t n, const float* __restrict__ X, int64_t ldx,
                                                           const float* __restrict__ Y, int64_t ldy,
                                                           double* __restrict__ part, int nparts) {
  __shared__ double red[4];
  const int b = blockIdx.y;
  const int64_t per = cdiv(n, nparts);
  const int64_t i0 = blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
  double acc = 0.0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += blockDim.x)
    acc += (double)X[b * ldx + i] * (double)Y[b * ldy + i];
  acc = block_sum<256>(acc, red);
  if (threadIdx.x == 0) part[b * nparts + blockIdx.x] = acc;
}

__global__ __launch_bounds__(64) void dot_final_kernel(int nparts, const double* __restrict__ part,
                                                       double* __restrict__ out) {
  const int b = blockIdx.x;
  double acc = 0.0;
  for (int i = threadIdx.x; i < nparts; i += 64) acc += part[b * nparts + i];
  acc = wave_sum(acc);
  if (threadIdx.x == 0) out[b] = acc;
}

constexpr int kDotParts = 256;

}  // namespace

extern "C" {

size_t ck_op_workspace_bytes(const ck_op* op, int32_t nrhs) { return ck::op_workspace_internal(op, nrhs); }

int ck_op_apply(const ck_op* op, int32_t nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, void* work,
                size_t work_bytes, void* stream) {
  return ck::op_apply_internal(op, nrhs, X, ldx, Y, ldy, work, work_bytes, nullptr, (hipStream_t)stream);
}

int ck_transpose_f32(int64_t n, int32_t nrhs, const float* src, int64_t lds_, float* dst, int64_t ldd,
                     int32_t to_blocks, void* stream) {
  if (n < 1 || nrhs < 1 || !src || !dst) return CK_ERR_BAD_ARG;
  if (to_blocks ? (lds_ < nrhs || ldd < n) : (lds_ < n || ldd < nrhs)) return CK_ERR_BAD_ARG;
  hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, n, nrhs, src,
                     lds_, dst, ldd, to_blocks);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

size_t ck_dot_workspace_bytes(int64_t n, int32_t nrhs) { return (size_t)nrhs * kDotParts * sizeof(double); }

int ck_dot_f32(int64_t n, int32_t nrhs, const float* X, int64_t ldx, const float* Y, int64_t ldy, double* out,
               void* work, size_t work_bytes, void* stream) {
  if (n < 1 || nrhs < 1 || !X || !Y || !out || ldx < n || ldy < n) return CK_ERR_BAD_ARG;
  if (!work || work_bytes < ck_dot_workspace_bytes(n, nrhs)) return CK_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  double* part = static_cast<double*>(work);
  hipLaunchKernelGGL(dot_partials_kernel, dim3(kDotParts, nrhs), dim3(256), 0, s, n, X, ldx, Y, ldy, part, kDotParts);
  hipLaunchKernelGGL(dot_final_kernel, dim3(nrhs), dim3(64), 0, s, kDotParts, part, out);
  CK_CHECK_LAUNCH();
  return CK_OK;
}

}  // extern "C"
