// Kronecker matvecs with two or three factors of any order up to 64, fp32 on v_mfma_f32_16x16x4f32.
//
// Vector b of a column block is a tensor X[i1][i2][i3].
//   pass A, per slab (b, i1):   U = K2 S K3^T, S = X[b][i1] (n2 x n3)
//   pass B, per 32 columns c of the i2*i3 plane:   Y[:, c] = scale * K1 U[:, c] + shift * X[:, c]
//
// The sum over k of an MFMA is order-free, so step (c, e) of a reduction takes k = 16 c + 4 g + e in
// lane group g = lane / 16 instead of four consecutive k.  That is the accumulator's own layout (item
// e of lane group g of row strip c is row 16 c + 4 g + e), so the n2 x 16 tile of S K3^T that a wave
// accumulates is, as it stands in registers, the second product's operand: the intermediate needs no
// LDS, no transposition and no barrier.  A wave of pass A owns a 16-column tile of a slab (all rows),
// one of pass B 32 columns of the plane, two per lane.  The slab and the factors are staged in LDS
// zero-padded to 64, so that the products' operands are float4 reads whatever the orders; all global
// loads of a block go out before the first is waited for, and chunks of 16 past an order are skipped.
// Latency bound at the sizes of a grid solve (the MFMAs of a 48 x 60 x 50 pass at 8 rhs take 2.6 us
// of the chip): pass A 17.2 -> 10.3 us, pass B 16.9 -> 6.5 us there against scalar LDS operands and a
// factor reloaded for every product, and CG's 4.5 us pass for p . Ap is gone.  63 x 64 x 64, 16 rhs:
// 59.6 -> 32.9 us for both.
#include "common.hpp"
#include "ops_internal.hpp"

using namespace ck;

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
// rows start wherever the orders put them: dword-aligned vector accesses
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ floatx4 mfma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kPitch = 68;  // LDS row pitch: 16-byte aligned rows, conflict-free float4 reads
constexpr int kTile = 64 * kPitch;

// A matrix of R x n (both up to 64, row-major, dense) on its way to a zero-padded 64 x kPitch LDS tile:
// thread t takes columns 4 (t % 16) .. + 3 of rows t / 16 + 16 q.  fetch() only loads (clamped
// addresses, nothing waits on the values); put() shifts a piece that was clamped at the row's end back
// into place, zeroes what lies outside and writes it.
struct Piece {
  floatx4 v[4];
};
__device__ __forceinline__ Piece fetch(const float* __restrict__ M, int R, int n) {
  Piece p;
  const int j = 4 * (threadIdx.x & 15), r0 = threadIdx.x >> 4;
  if (n >= 4) {
    const int jc = j < n - 4 ? j : n - 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 16 * q;
      p.v[q] = *reinterpret_cast<const f4u*>(M + (r < R ? r : R - 1) * n + jc);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 16 * q;
#pragma unroll
      for (int e = 0; e < 4; ++e) p.v[q][e] = M[(r < R ? r : R - 1) * n + (e < n ? e : n - 1)];
    }
  }
  return p;
}
__device__ __forceinline__ void put(float* __restrict__ tile, const Piece& p, int R, int n) {
  const int j = 4 * (threadIdx.x & 15), r0 = threadIdx.x >> 4;
  const int d = n >= 4 && j > n - 4 ? j - (n - 4) : 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = r0 + 16 * q;
    const floatx4 w = p.v[q];
    floatx4 o;
    o[0] = d == 0 ? w[0] : d == 1 ? w[1] : d == 2 ? w[2] : w[3];
    o[1] = d == 0 ? w[1] : d == 1 ? w[2] : w[3];
    o[2] = d == 0 ? w[2] : w[3];
    o[3] = w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = r < R && j + e < n ? o[e] : 0.f;
    *reinterpret_cast<floatx4*>(tile + r * kPitch + j) = o;
  }
}

// Slabs [blockIdx.x * per, + per); slab s is (rhs s / n1, i1 = s % n1), C2 = ceil(n2 / 16).  Wave t owns
// the slab's columns 16 t .. + 15.  LAST (two factors): U is the operator's output,
// scale * U + shift * S.
template <int C2, bool LAST>
__global__ __launch_bounds__(256) void kron_any_pass_a(int slabs, int per, int n1, int n2, int n3,
                                                       const float* __restrict__ K2, const float* __restrict__ K3,
                                                       const float* __restrict__ X, int64_t ldx,
                                                       float* __restrict__ Out, int64_t ldo, float scale, float shift,
                                                       const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ __align__(16) float S[kTile], L2[kTile], L3[kTile];
  const int lane = threadIdx.x & 63, t = threadIdx.x >> 6, g = lane >> 4, li = lane & 15;
  const int C3 = (n3 + 15) / 16, col = 16 * t + li;
  const int s0 = blockIdx.x * per, s1 = s0 + per < slabs ? s0 + per : slabs;
  auto slab = [&](int s) {
    const int b = s / n1;
    return X + (int64_t)b * ldx + (int64_t)(s - b * n1) * n2 * n3;
  };
  Piece ps = fetch(slab(s0), n2, n3);
  {
    const Piece p3 = fetch(K3, n3, n3), p2 = fetch(K2, n2, n2);
    __builtin_amdgcn_sched_barrier(0);  // all twelve loads go out before the first is waited for
    put(L3, p3, n3, n3);
    put(L2, p2, n2, n2);
  }
  for (int s = s0; s < s1; ++s) {
    put(S, ps, n2, n3);
    __syncthreads();
    if (s + 1 < s1) ps = fetch(slab(s + 1), n2, n3);
    if (t < C3) {
      floatx4 T[C2], u[C2];
#pragma unroll
      for (int r = 0; r < C2; ++r) T[r] = u[r] = floatx4{0.f, 0.f, 0.f, 0.f};
      const float* sp = S + li * kPitch + 4 * g;
      const float* p3 = L3 + col * kPitch + 4 * g;
      for (int c = 0; c < C3; ++c) {
        const floatx4 k = *reinterpret_cast<const floatx4*>(p3 + 16 * c);
        floatx4 a[C2];
#pragma unroll
        for (int r = 0; r < C2; ++r) a[r] = *reinterpret_cast<const floatx4*>(sp + 16 * r * kPitch + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < C2; ++r) T[r] = mfma(a[r][e], k[e], T[r]);
      }
      // rows past n2 are 0 times K3: zero for the second product also where K3 is not finite
#pragma unroll
      for (int q = 0; q < 4; ++q) T[C2 - 1][q] = 16 * (C2 - 1) + 4 * g + q < n2 ? T[C2 - 1][q] : 0.f;
      const float* p2 = L2 + li * kPitch + 4 * g;
#pragma unroll
      for (int c = 0; c < C2; ++c) {
        floatx4 a[C2];
#pragma unroll
        for (int r = 0; r < C2; ++r) a[r] = *reinterpret_cast<const floatx4*>(p2 + 16 * r * kPitch + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < C2; ++r) u[r] = mfma(a[r][e], T[c][e], u[r]);
      }
      if (col < n3) {
        const int b = s / n1;
        float* O = Out + (int64_t)b * ldo + (int64_t)(s - b * n1) * n2 * n3 + col;
#pragma unroll
        for (int r = 0; r < C2; ++r)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int row = 16 * r + 4 * g + q;
            if (row < n2) {
              float y = u[r][q];
              if (LAST) {
                y *= scale;
                if (shift != 0.f) y = fmaf(shift, S[row * kPitch + col], y);
              }
              O[row * n3] = y;
            }
          }
      }
    }
    __syncthreads();  // S is read before the next slab overwrites it
  }
}

// two neighbouring entries of a row of `plane` (one, twice, where a row has no second)
__device__ __forceinline__ f2u load_pair(const float* __restrict__ p, int plane) {
  if (plane < 2) {
    f2u v;
    v.x = v.y = p[0];
    return v;
  }
  return *reinterpret_cast<const f2u*>(p);
}

// Block (x, b): columns [128 x, + 128) of rhs b, 32 per wave; C1 = ceil(n1 / 16).  With partials,
// partials[b * nparts + x] = the block's sum of X . Y.
template <int C1>
__global__ __launch_bounds__(256) void kron_any_pass_b(int n1, int plane, const float* __restrict__ K1,
                                                       const float* __restrict__ U, int64_t ldu,
                                                       const float* __restrict__ X, int64_t ldx, float* __restrict__ Y,
                                                       int64_t ldy, float scale, float shift,
                                                       float* __restrict__ partials, int nparts,
                                                       const int* __restrict__ done) {
  if (done && *done) return;
  __shared__ __align__(16) float L1[kTile];
  __shared__ float red[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, li = lane & 15;
  const int b = blockIdx.y, col = blockIdx.x * 128 + 32 * w + 2 * li;
  const float* Ub = U + (int64_t)b * ldu;
  const float* Xb = X + (int64_t)b * ldx;
  float* Yb = Y + (int64_t)b * ldy;
  const Piece p1 = fetch(K1, n1, n1);
  // rows 16 c + 4 g + e of the lane's two columns, clamped like the factor's pieces
  const int cl = plane < 2 ? 0 : col < plane - 1 ? col : plane - 2;
  f2u uv[C1][4], xv[C1][4];
#pragma unroll
  for (int c = 0; c < C1; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = 16 * c + 4 * g + e, o = (k < n1 ? k : n1 - 1) * plane + cl;
      uv[c][e] = load_pair(Ub + o, plane);
      xv[c][e] = load_pair(Xb + o, plane);
    }
  __builtin_amdgcn_sched_barrier(0);
  put(L1, p1, n1, n1);
  __syncthreads();
  const bool swap = cl != col;  // the row's last column came back as the pair's second
  floatx4 y0[C1], y1[C1];
#pragma unroll
  for (int r = 0; r < C1; ++r) y0[r] = y1[r] = floatx4{0.f, 0.f, 0.f, 0.f};
  const float* lp = L1 + li * kPitch + 4 * g;
#pragma unroll
  for (int c = 0; c < C1; ++c) {
    floatx4 a[C1];
#pragma unroll
    for (int r = 0; r < C1; ++r) a[r] = *reinterpret_cast<const floatx4*>(lp + 16 * r * kPitch + 16 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = 16 * c + 4 * g + e < n1;
      const float ux = in ? (swap ? uv[c][e].y : uv[c][e].x) : 0.f, uy = in ? uv[c][e].y : 0.f;
#pragma unroll
      for (int r = 0; r < C1; ++r) {
        y0[r] = mfma(a[r][e], ux, y0[r]);
        y1[r] = mfma(a[r][e], uy, y1[r]);
      }
    }
  }
  float dot = 0.f;
#pragma unroll
  for (int r = 0; r < C1; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 16 * r + 4 * g + q;
      const float x0 = swap ? xv[r][q].y : xv[r][q].x, x1 = xv[r][q].y;
      float a = scale * y0[r][q], c = scale * y1[r][q];
      if (shift != 0.f) {
        a = fmaf(shift, x0, a);
        c = fmaf(shift, x1, c);
      }
      if (row < n1) {
        float* dst = Yb + row * plane + col;
        if (col + 1 < plane) {
          f2u o;
          o.x = a;
          o.y = c;
          *reinterpret_cast<f2u*>(dst) = o;
          dot = fmaf(x0, a, fmaf(x1, c, dot));
        } else if (col < plane) {
          dst[0] = a;
          dot = fmaf(x0, a, dot);
        }
      }
    }
  if (partials) {
    const float s = block_sum<256>(dot, red);
    if (threadIdx.x == 0) partials[(int64_t)b * nparts + blockIdx.x] = s;
  }
}

}  // namespace

namespace ck {

int kron_any_nparts(int plane) { return (plane + 127) / 128; }

int kron_any_apply(const ck_op* op, int nrhs, const float* X, int64_t ldx, float* Y, int64_t ldy, float* U,
                   const int* done, float* partials, int nparts, hipStream_t s) {
  const bool two = op->nfactors == 2;
  const int n1 = two ? 1 : op->fdim[0], n2 = op->fdim[two ? 0 : 1], n3 = op->fdim[two ? 1 : 2];
  const float* K2 = op->factor[two ? 0 : 1];
  const float* K3 = op->factor[two ? 1 : 2];
  // a block keeps its factors for several slabs once there are enough of them to fill the chip (three
  // blocks per CU) that often
  const int slabs = n1 * nrhs;
  int per = slabs / 768;
  per = per < 1 ? 1 : per > 4 ? 4 : per;
  const dim3 grid((unsigned)cdiv(slabs, per));
#define CK_PASS_A(C_, LAST_, O_, LDO_, SC_, SH_)                                                                       \
  hipLaunchKernelGGL((kron_any_pass_a<C_, LAST_>), grid, dim3(256), 0, s, slabs, per, n1, n2, n3, K2, K3, X, ldx, O_, \
                     LDO_, SC_, SH_, done)
#define CK_PASS_A_C(LAST_, O_, LDO_, SC_, SH_)      \
  switch ((n2 + 15) / 16) {                         \
    case 1: CK_PASS_A(1, LAST_, O_, LDO_, SC_, SH_); break;  \
    case 2: CK_PASS_A(2, LAST_, O_, LDO_, SC_, SH_); break;  \
    case 3: CK_PASS_A(3, LAST_, O_, LDO_, SC_, SH_); break;  \
    default: CK_PASS_A(4, LAST_, O_, LDO_, SC_, SH_); break; \
  }
  if (two) {
    CK_PASS_A_C(true, Y, ldy, op->scale, op->shift)
  } else {
    CK_PASS_A_C(false, U, (int64_t)op->n, 1.f, 0.f)
    const dim3 gb((unsigned)kron_any_nparts(n2 * n3), nrhs);
#define CK_PASS_B(C_)                                                                                                 \
  hipLaunchKernelGGL(kron_any_pass_b<C_>, gb, dim3(256), 0, s, n1, n2 * n3, op->factor[0], (const float*)U,          \
                     (int64_t)op->n, X, ldx, Y, ldy, op->scale, op->shift, partials, nparts, done)
    switch ((n1 + 15) / 16) {
      case 1: CK_PASS_B(1); break;
      case 2: CK_PASS_B(2); break;
      case 3: CK_PASS_B(3); break;
      default: CK_PASS_B(4); break;
    }
#undef CK_PASS_B
  }
#undef CK_PASS_A_C
#undef CK_PASS_A
  CK_CHECK_LAUNCH();
  return CK_OK;
}

}  // namespace ck
