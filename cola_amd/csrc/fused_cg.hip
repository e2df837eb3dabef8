// Persistent fused CG: a whole batched CG solve in one launch.
//
// Arithmetic and stopping rule are those of cola/linalg/inverse/cg.py:94-178 (column
// normalisation, threshold tol*||r0|| + tol, safe division at 1e-40, frozen columns), the
// loop of cola/utils/torch_tqdm.py:86-90 runs inside the kernel.  Scope: dense operators
// (y = scale*A x + shift*x) whose solves are launch- and latency-bound, with no
// preconditioner or a diagonal one, 1 to 8 columns.
//
// A stays in registers for the whole solve.  A workgroup is 8 waves of 512 threads; lane
// (b, i) = (lane / 4, lane % 4) of a wave keeps rows 4q + i, q < Q, at columns 64c + 4b .. + 3
// of its KC chunks of 64, loaded once with 16-byte loads (4 Q KC registers of 256).  A
// product reads p from LDS, 16 bytes per lane and chunk, and needs no other operand: one
// column on the VALU, two to four columns on v_mfma_f32_4x4x1_16b, whose sixteen blocks take
// the sixteen b's as sixteen different k and whose A operand is the same register (four
// columns cost what two would on the VALU).  The sums over b are two rounds of half swaps,
// which halve the registers as they go, and two rotations within a row of sixteen.  The
// scalars of column c are computed by the lanes = c mod NB of every wave alike and reach the
// others as scalar registers, so that no step of them waits at a barrier.
//
// One workgroup, up to 320 unknowns (256 for two to four columns): wave w holds rows 4Qw on,
// all columns (Q = 2 KC), entry j of x, r, p is thread j's, and a step has four barriers.
// Bound by that serial chain: orders 64 / 150 / 300 and 256 x 4 columns take 1.3 / 1.6 / 1.9
// and 3.8 us a step, over several workgroups 2.4 / 2.4 / 2.5 and 3.9.  At 300 x 2 to 4 columns
// the matrix, 40 accumulators and the columns' vectors no longer fit 256 registers.
//
// Several workgroups, up to 3584 unknowns: a workgroup holds R <= 4Q rows, wave w the chunks
// = w mod 8, and every workgroup the FULL r and p vectors in LDS.  A step:
//   Ap_own = A_own p                   (rows from registers, p from LDS, the waves' sums in LDS)
//   publish Ap_own                     (the step's one grid-wide exchange)
//   read all of Ap; p.Ap, alpha        (every workgroup, same order -> same bits)
//   x_own += alpha p_own;  r -= alpha Ap;  gamma' = r.z, ||r||, beta, p = z + beta p
// with the vector updates done redundantly by every workgroup, so a step needs exactly one
// grid-wide exchange and no separate barrier.  Bound by the exchange and its read-back at one
// column, by the redundant vector work as n nrhs grows.  us a step, against rows in LDS (from
// cache above 1400) with a wave per row and the columns' scalars one after the other, and
// against four chained launches:
//   n = 500 x 1 / 4      2.5 /  4.0    6.1 / 12.5    15 / 14
//   n = 1000 x 1 / 4     2.8 /  4.9    7.0 / 19.9    16 / 14
//   n = 2000 x 1 / 4 / 8 3.3 /  7.0 / 11.3   21.6 / - / -   15 / 15 / 17
//   n = 3500 x 1 / 4     4.4 / 10.4    - / -   20 / 20
//
// The exchange: every Ap entry travels as one 64-bit word (value bits, step tag) written and
// read with agent-scope atomic stores and loads, which the compiler emits as coherent (sc1)
// accesses that do not stop in a per-XCD L2.  Readers load their words and re-read, all
// together, the ones whose tag is still old: the tag is the flag, so a step costs the
// writers' stores landing plus the readers' polling round trips, with no fence, no separate
// flag and no cache maintenance.  The buffers are doubled by step parity: a workgroup can run
// at most one step ahead of the slowest reader (it needs every entry of the current step,
// written after each writer finished reading the previous one), so it never overwrites a word
// still to be read.  Every wait is bounded: after spin_limit polling rounds it gives up,
// records CK_ERR_TIMEOUT in the control block and leaves the loop, so every workgroup ends and
// the launch drains.  All workgroups fit on the device at once (checked by occupancy before
// the launch; a cooperative launch guarantees co-residency, a plain one is the default).
//
// Above 3584 unknowns (one column, up to 7168) the rows of a workgroup no longer fit its
// registers beside the rest and are read again in every step: 32 us a step at 7000, in 4-byte
// loads by a wave per row 253, chained 39.
#include <mutex>

#include "cg_state.hpp"
#include "common.hpp"

using namespace ck;

namespace {

constexpr double kSmall = (double)(float)1e-40;  // cg.py:8, as an fp32 constant
constexpr int kNT = 512, kNW = kNT / 64;
constexpr int kMaxRhs = 8;
constexpr int kMaxBlocks = 256;
// Register-resident rows: chunks of 512 columns and the row quads that fit beside them.  16 rows a
// workgroup (20 above 3072) keep the workgroups at 192, so a quarter of the CUs stays free for what
// other streams run meanwhile.
constexpr int kMaxChunks = 7, kMaxChunks8 = 4;  // for up to four columns; five to eight
__host__ __device__ constexpr int quads_of(int kc) { return kc <= 6 ? 4 : 5; }
constexpr int kMaxResident = 64 * kNW * kMaxChunks;
constexpr int kStreamQuads = 7, kStreamChunks = 14;  // up to 7168 = 256 * 28 = 14 * 512
// One workgroup: chunks of 64 unknowns for one column, for two to four
constexpr int kOneChunks = 5, kOneChunksMulti = 4;
constexpr int64_t kDefaultSpin = int64_t(1) << 22;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct FusedArgs {
  int n, nn, nrhs, G, R;  // order, padded order (multiple of 4), columns, workgroups, rows per workgroup
  const float* A;
  int64_t lda;
  float scale, shift;
  const float* d;  // diagonal preconditioner (nullptr: none): z = dscale * d * r + dshift * r
  float dscale, dshift;
  const float* b;
  int64_t b_rs, b_cs;
  const float* x0;
  int64_t x0_rs, x0_cs;
  float* x;
  int64_t x_rs, x_cs;
  float* r;
  int64_t r_rs, r_cs;
  void* state;
  float tol;
  int max_iters;
  uint64_t* xbuf;  // 2 x nrhs x nn tagged words
  int64_t spin_limit;
  uint32_t wait_offset;
};

__device__ inline double safe_div(double num, double den) {
  if (fabs(den) < kSmall) den = kSmall;
  return num / den;
}

__device__ inline void put(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline uint64_t get(const uint64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void put(int32_t* p, int32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void put(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline uint32_t get(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ inline uint64_t pack(float v, uint32_t tag) { return ((uint64_t)tag << 32) | (uint64_t)__float_as_uint(v); }
__device__ inline uint32_t tag_of(uint64_t w) { return (uint32_t)(w >> 32); }
__device__ inline float value_of(uint64_t w) { return __uint_as_float((uint32_t)w); }


// a + its half swap with b: the sums over lane bit 5 (or 4) of a in the lanes where the bit is
// clear and of b where it is set.
__device__ inline float add_swap32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float add_swap16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// v[m] summed over lane bits 2..5; f(m, sum) is called with the m that this lane's row of
// sixteen holds.
template <int M, typename F>
__device__ inline void sum_over_blocks(float (&v)[M], int lane, F f) {
  constexpr int M1 = (M + 1) / 2, M2 = (M1 + 1) / 2;
  float u[M1];
#pragma unroll
  for (int i = 0; i < M1; ++i) u[i] = add_swap32(v[2 * i], 2 * i + 1 < M ? v[2 * i + 1 < M ? 2 * i + 1 : 0] : 0.f);
#pragma unroll
  for (int i = 0; i < M2; ++i) {
    float w = add_swap16(u[2 * i], 2 * i + 1 < M1 ? u[2 * i + 1 < M1 ? 2 * i + 1 : 0] : 0.f);
    w += dpp_f32<0x124>(w);  // row_ror:4
    w += dpp_f32<0x128>(w);  // row_ror:8
    const int m = 4 * i + 2 * ((lane >> 4) & 1) + (lane >> 5);
    if (m < M) f(m, w);
  }
}


// This thread's entries j = tid + 512 t of every column from the tagged buffer xb (nn words
// per column): the loads of a chunk of CH words are issued together, and the words still
// carrying an old tag are re-read together, one round trip per round, until every tag is
// `want` (bounded by spin rounds; after a timeout nothing more is waited for).  Returns false
// on timeout (and sets *fail).
template <int NB, int KT, int CH>
__device__ inline bool collect(const uint64_t* xb, int n, int nn, int B, uint32_t want, int64_t spin,
                               float (&out)[NB][KT], int* fail) {
  bool ok = true;
  constexpr int E = NB * KT;  // entries e = c * KT + t
#pragma unroll
  for (int e0 = 0; e0 < E; e0 += CH) {
    uint64_t raw[CH];
    uint32_t pending = 0;
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int e = e0 + u, c = e / KT, t = e % KT;
      const int j = threadIdx.x + kNT * t;
      if (e < E && c < B && j < n) pending |= 1u << u;
    }
    if (!ok) pending = 0;
    for (int64_t it = 0; pending; ++it) {
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int e = e0 + u, c = e / KT, t = e % KT;
        if (pending & (1u << u)) raw[u] = get(xb + (int64_t)c * nn + threadIdx.x + kNT * t);
      }
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int e = e0 + u, c = e / KT, t = e % KT;
        if ((pending & (1u << u)) && tag_of(raw[u]) == want) {
          out[c][t] = value_of(raw[u]);
          pending &= ~(1u << u);
        }
      }
      if (!pending) break;
      if (it >= spin) {
        ok = false;
        *fail = 1;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  return ok;
}

// Rows row0 + 4 (wr Q + q) + (lane & 3) < row1 at columns 64 (c WC + wc) + 4 (lane / 4) .. + 3, zero
// outside the matrix.  KC = ceil(n / (64 WC)), so only the last chunk can be short or absent.
template <int Q, int KC, int WC>
__device__ inline void load_rows(const FusedArgs& a, int row0, int row1, int wc, int lane, float (&av)[KC][Q][4]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int row = row0 + 4 * q + (lane & 3);
    const float* rp = a.A + (int64_t)min(row, a.n - 1) * a.lda;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int k = 64 * (c * WC + wc) + 4 * (lane >> 2);
      f32x4 t = {0.f, 0.f, 0.f, 0.f};
      if (c < KC - 1 || k + 3 < a.n) {
        t = *reinterpret_cast<const f32x4u*>(rp + k);
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (k + e < a.n) t[e] = rp[k + e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) av[c][q][e] = row < row1 ? t[e] : 0.f;
    }
  }
}

// acc += the wave's 4Q rows at four columns per b times p there; after all chunks `finish` hands the
// sums over b to f(row, column, sum).  pk: the lane's column of p (lane & 3 of the first four) at its
// four k; the next four columns LD * 4 further.
template <int NB, int Q, int LD>
struct Acc {
  static constexpr int NG = NB == 1 ? 1 : NB / 4;
  float s[NB == 1 ? Q : 1];
  f32x4 m[NB == 1 ? 1 : NG * Q];
  __device__ inline Acc() {
#pragma unroll
    for (float& v : s) v = 0.f;
#pragma unroll
    for (f32x4& v : m) v = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __device__ inline void add(const float (&av)[Q][4], const float* pk) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const f32x4 p4 = *reinterpret_cast<const f32x4*>(pk + 4 * g * LD);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          if constexpr (NB == 1)
            s[q] = fmaf(av[q][e], p4[e], s[q]);
          else
            m[g * Q + q] = __builtin_amdgcn_mfma_f32_4x4x1f32(av[q][e], p4[e], m[g * Q + q], 0, 0, 0);
        }
    }
  }
  template <typename F>
  __device__ inline void finish(int lane, F f) {
    if constexpr (NB == 1) {
      sum_over_blocks<Q>(s, lane, [&](int q, float v) {
        if ((lane & 12) == 0) f(4 * q + (lane & 3), 0, v);
      });
    } else {
      float flat[NG * 4 * Q];
#pragma unroll
      for (int q = 0; q < NG * Q; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) flat[4 * q + i] = m[q][i];
      sum_over_blocks<NG * 4 * Q>(flat, lane, [&](int e, float v) {
        if ((lane & 12) == 0) f(e % (4 * Q), 4 * (e / (4 * Q)) + (lane & 3), v);
      });
    }
  }
};

__device__ inline double add_swap(double a, double b, bool half) {
  const uint64_t ua = __double_as_longlong(a), ub = __double_as_longlong(b);
  const auto lo = half ? __builtin_amdgcn_permlane32_swap((uint32_t)ua, (uint32_t)ub, false, false)
                       : __builtin_amdgcn_permlane16_swap((uint32_t)ua, (uint32_t)ub, false, false);
  const auto hi = half ? __builtin_amdgcn_permlane32_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false)
                       : __builtin_amdgcn_permlane16_swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32), false, false);
  return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}
__device__ inline double row_sum(double v) {  // over sixteen lanes
  v += dpp_f64<0xB1>(v);
  v += dpp_f64<0x4E>(v);
  v += dpp_f64<0x124>(v);
  return v + dpp_f64<0x128>(v);
}

// Sums over the block: each wave's into red, and after a barrier the total of the lane's column.  The
// half swaps of sum_over_blocks take four columns (or the two sums of one) through one chain.
template <int NB>
__device__ inline void put_sums(double* red, const double (&w)[NB]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (NB == 1) {
    const double t = wave_sum(w[0]);
    if (lane == 0) red[wave] = t;
  } else {
#pragma unroll
    for (int g = 0; g < NB; g += 4) {
      const double t = row_sum(add_swap(add_swap(w[g], w[g + 1], true), add_swap(w[g + 2], w[g + 3], true), false));
      if ((lane & 15) == 0) red[wave * NB + g + 2 * ((lane >> 4) & 1) + (lane >> 5)] = t;
    }
  }
}
template <int NB>
__device__ inline void put_sums(double* red, const double (&w0)[NB], const double (&w1)[NB]) {  // w1 from red + kNW * NB
  if constexpr (NB == 1) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double u = add_swap(w0[0], w1[0], true);
    const double t = row_sum(add_swap(u, u, false));
    if ((lane & 31) == 0) red[wave + kNW * (lane >> 5)] = t;
  } else {
    put_sums<NB>(red, w0);
    put_sums<NB>(red + kNW * NB, w1);
  }
}
template <int NB>
__device__ inline double total(const double* red, int col) {
  double t[kNW];
#pragma unroll
  for (int i = 0; i < kNW; ++i) t[i] = red[i * NB + col];
  return ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
}

// The scalars of this lane's column and the loop's state (the same in every wave and workgroup).
template <int NB>
struct Steps {
  float mult, rnorm, gamma, tol, alpha = 0.f, beta = 0.f;
  int k = 0, status = CK_OK;
  bool any, finite, frozen;
  // errors[k] and the loop condition (cg.py:133-138)
  __device__ inline bool check(const FusedArgs& a, CgView& v, bool writer) {
    float mean = 0.f;
    any = false;
    finite = true;
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (c < a.nrhs) {
        const float rn = readlane_f32(rnorm, c);
        mean += rn;
        any = any || rn > readlane_f32(tol, c);
        finite = finite && isfinite(rn);
      }
    if (writer) v.errors[k] = mean / (float)a.nrhs;
    return !(any && k < a.max_iters);
  }
  // cg.py:98-101,122-130: gamma = r.z, threshold tol*||r0|| + tol
  __device__ inline bool start(const FusedArgs& a, CgView& v, bool writer, double rr, double rz) {
    rnorm = (float)sqrt(rr);
    gamma = (float)rz;
    tol = a.tol * rnorm + a.tol;
    const bool done = check(a, v, writer);
    if (!finite) status = CK_ERR_NAN;
    return done;
  }
  // cg.py:143-147
  __device__ inline void set_alpha(double pap) {
    frozen = (double)rnorm < kSmall;
    alpha = frozen ? 0.f : (float)safe_div((double)gamma, pap);
    if (status == CK_OK && __ballot(!frozen && !(pap > 0.0)) != 0) status = CK_ERR_BREAKDOWN;
  }
  // beta = gamma'/gamma (cg.py:150-154), frozen columns keep beta = 0
  __device__ inline void set_beta(double rr, double rz) {
    beta = frozen ? 0.f : (float)safe_div(rz, (double)gamma);
    gamma = (float)rz;
    rnorm = (float)sqrt(rr);
  }
  __device__ inline bool next(const FusedArgs& a, CgView& v, bool writer) {
    ++k;
    const bool done = check(a, v, writer);
    if (done) {
      if (!finite)
        status = CK_ERR_NAN;
      else if (any && status == CK_OK)
        status = CK_ERR_MAXITER;
    }
    return done;
  }
  __device__ inline void store(const FusedArgs& a, CgView& v) {
    const int tid = threadIdx.x;
    if (tid < a.nrhs) {
      v.mult[tid] = mult;
      v.tol[tid] = tol;
      v.gamma[tid] = gamma;
      v.alpha[tid] = alpha;
      v.beta[tid] = beta;
      v.rnorm[tid] = rnorm;
    }
    if (tid == 0) {
      v.ctrl->k = k;
      v.ctrl->done = 1;
      v.ctrl->max_iters = a.max_iters;
      v.ctrl->nrhs = a.nrhs;
      v.ctrl->nparts = a.G;
    }
  }
};

// b / max(||b||, 1e-40) of cg.py:96-97
__device__ inline float norm_of(float mult, int c) {
  const float m = readlane_f32(mult, c);
  return fabsf(m) < 1e-40f ? 1e-40f : m;
}

template <int NB, int KC>
__global__ __launch_bounds__(kNT) void fused_one_kernel(FusedArgs a) {
  constexpr int Q = 2 * KC, NP = 64 * KC, LD = NP + 16;
  __shared__ float pv[NB * LD];  // columns 16 banks apart: the four columns of a 16-byte read don't collide
  __shared__ float yv[NB * NP];
  __shared__ double red1[kNW * NB], red2[2 * kNW * NB];
  const int n = a.n, B = a.nrhs, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = min(lane & (NB - 1), B - 1);  // the column whose scalars this lane computes
  const bool own = tid < n, pre = a.d != nullptr;
  CgView v = cg_view(a.state, B);
  Steps<NB> st;
  float av[KC][Q][4];
  load_rows<Q, KC, 1>(a, 4 * Q * wave, n, 0, lane, av);
  auto product = [&]() {  // yv = A p for p in pv, all columns
    Acc<NB, Q, LD> acc;
    auto at = [&](int c) {
      return *reinterpret_cast<const f32x4*>(pv + (NB > 1 ? lane & 3 : 0) * LD + 64 * c + 4 * (lane >> 2));
    };
    // A lane's sum (20 products at 320 unknowns) as a tree of chunks, those of one column in pairs, as if more
    // lanes had shared the row.  The solutions' errors (means of 60 systems), as multiples of what 64 lanes a
    // row give: 300 x 1 1.25 with one chain and 1.01 as a tree, 256 x 2 1.14 and 0.99, 256 x 4 1.20 and 1.02.
    // A tree costs 0.05 to 0.1 us a step for one column, 0.7 at 256 x 4.
    constexpr int K4 = KC < 4 ? KC : 4;
    auto piece = [&](int c, int q, const f32x4& p) {
      if constexpr (NB == 1) {
        return fmaf(av[c][q][1], p[1], av[c][q][0] * p[0]) + fmaf(av[c][q][3], p[3], av[c][q][2] * p[2]);
      } else {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) t = __builtin_amdgcn_mfma_f32_4x4x1f32(av[c][q][e], p[e], t, 0, 0, 0);
        return t;
      }
    };
    f32x4 p4[K4];
#pragma unroll
    for (int c = 0; c < K4; ++c) p4[c] = at(c);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      auto t = piece(0, q, p4[0]);
      if constexpr (K4 > 1) t += piece(1, q, p4[1]);
      if constexpr (K4 == 3) t += piece(2, q, p4[2]);
      if constexpr (K4 == 4) t += piece(2, q, p4[2]) + piece(3, q, p4[3]);
      if constexpr (NB == 1)
        acc.s[q] = t;
      else
        acc.m[q] = t;
    }
    if constexpr (KC == 5) {  // one column only
      const f32x4 p = at(4);
#pragma unroll
      for (int q = 0; q < Q; ++q) acc.s[q] += piece(4, q, p);
    }
    acc.finish(lane, [&](int row, int c, float s) { yv[c * NP + 4 * Q * wave + row] = s; });
  };
  float x[NB], r[NB], p[NB], z[NB];  // of column c < nrhs at entry tid < n, else zero
  double w0[NB], w1[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    x[c] = 0.f;
    r[c] = own && c < B ? a.b[(int64_t)tid * a.b_rs + (int64_t)c * a.b_cs] : 0.f;
    w0[c] = (double)r[c] * (double)r[c];
  }
  put_sums<NB>(red1, w0);
  const float dj = pre && own ? a.d[tid] : 0.f;
  for (int i = tid; i < NB * LD; i += kNT) pv[i] = 0.f;
  __syncthreads();
  st.mult = (float)sqrt(total<NB>(red1, col));
#pragma unroll
  for (int c = 0; c < NB; ++c) r[c] /= norm_of(st.mult, c);
  if (a.x0) {
    // cg.py:123: r0 = b_norm - A x0 (x0 as given)
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (own && c < B) pv[c * LD + tid] = x[c] = a.x0[(int64_t)tid * a.x0_rs + (int64_t)c * a.x0_cs];
    __syncthreads();
    product();
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (own && c < B) {
        float y = a.scale * yv[c * NP + tid];
        if (a.shift != 0.f) y = fmaf(a.shift, x[c], y);
        r[c] -= y;
      }
  }
  // z = P r, p = z
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    z[c] = pre ? fmaf(a.dscale * dj, r[c], a.dshift * r[c]) : r[c];
    p[c] = z[c];
    if (own) pv[c * LD + tid] = p[c];
    w0[c] = (double)r[c] * (double)r[c];
    w1[c] = (double)r[c] * (double)z[c];
  }
  put_sums<NB>(red2, w0, w1);
  __syncthreads();
  bool done = st.start(a, v, tid == 0, total<NB>(red2, col), total<NB>(red2 + kNW * NB, col));
  while (!done) {
    product();
    __syncthreads();
    float ap[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      ap[c] = own ? a.scale * yv[c * NP + tid] : 0.f;
      if (a.shift != 0.f) ap[c] = fmaf(a.shift, p[c], ap[c]);
      w0[c] = (double)p[c] * (double)ap[c];
    }
    put_sums<NB>(red1, w0);
    __syncthreads();
    st.set_alpha(total<NB>(red1, col));
    // x += alpha p, r -= alpha Ap, gamma' = r.z, ||r||^2
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      const float al = readlane_f32(st.alpha, c);
      x[c] = fmaf(al, p[c], x[c]);
      r[c] = fmaf(-al, ap[c], r[c]);
      z[c] = pre ? fmaf(a.dscale * dj, r[c], a.dshift * r[c]) : r[c];
      w0[c] = (double)r[c] * (double)r[c];
      w1[c] = (double)r[c] * (double)z[c];
    }
    put_sums<NB>(red2, w0, w1);
    __syncthreads();
    st.set_beta(total<NB>(red2, col), total<NB>(red2 + kNW * NB, col));
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      p[c] = fmaf(readlane_f32(st.beta, c), p[c], z[c]);
      if (own) pv[c * LD + tid] = p[c];
    }
    done = st.next(a, v, tid == 0);
    __syncthreads();
  }
  // cg.py:119: x and r back to the scale of b
#pragma unroll
  for (int c = 0; c < NB; ++c)
    if (own && c < B) {
      const float m = readlane_f32(st.mult, c);
      a.x[(int64_t)tid * a.x_rs + (int64_t)c * a.x_cs] = x[c] * m;
      if (a.r) a.r[(int64_t)tid * a.r_rs + (int64_t)c * a.r_cs] = r[c] * m;
    }
  st.store(a, v);
  if (tid == 0) v.ctrl->status = st.status;
}

// RES: the rows in registers (else read again by every product)
template <int NB, int Q, int KC, bool RES>
__global__ __launch_bounds__(kNT, RES ? 2 : 4) void fused_cg_kernel(FusedArgs a) {
  constexpr int RW = 4 * Q;                               // most rows of a workgroup
  constexpr int CH = !RES || Q * KC > 20 ? 8 : 16;        // words a thread reads at once
  constexpr int LD = kNT * KC + 16;                       // 16 banks apart, as above
  extern __shared__ __align__(16) float lds[];
  __shared__ float part[kNW * NB * RW];
  __shared__ double red1[kNW * NB], red2[2 * kNW * NB];
  __shared__ int s_fail;
  const int n = a.n, nn = a.nn, B = a.nrhs, w = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row0 = w * a.R, rows = min(a.R, n - row0);
  const int col = min(lane & (NB - 1), B - 1), pcol = NB > 1 ? min(lane & 3, B - 1) : 0;
  const bool pre = a.d != nullptr;
  // the entry that this thread publishes and whose x it keeps
  const int xc = tid / RW, xi = tid % RW;
  const bool pub = xc < B && xi < rows;
  float* pv = lds;           // B x LD: full p, zero from n on
  float* rv = lds + B * LD;  // B x LD: full r, likewise
  CgView v = cg_view(a.state, B);
  Steps<NB> st;
  if (tid == 0) s_fail = 0;
  float av[RES ? KC : 1][Q][4];
  if constexpr (RES) load_rows<Q, KC, kNW>(a, row0, row0 + rows, wave, lane, av);
  uint32_t sync = 0;
  // A times the vectors in pv for the own rows, published with the next tag into the buffer xb
  auto product = [&](uint64_t* xb) {
    Acc<NB, Q, LD> acc;
    if constexpr (RES) {
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const int k = 64 * (c * kNW + wave);
        if (c < KC - 1 || k < n) acc.add(av[c], pv + pcol * LD + k + 4 * (lane >> 2));
      }
    } else {
#pragma unroll 1
      for (int k0 = 64 * wave; k0 < n; k0 += 64 * kNW) {
        const int k = k0 + 4 * (lane >> 2);
        float t[Q][4];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const float* rp = a.A + (int64_t)min(row0 + 4 * q + (lane & 3), n - 1) * a.lda;
          f32x4 u = {0.f, 0.f, 0.f, 0.f};
          if (k + 3 < n) {
            u = *reinterpret_cast<const f32x4u*>(rp + k);
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (k + e < n) u[e] = rp[k + e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) t[q][e] = u[e];
        }
        acc.add(t, pv + pcol * LD + k);
      }
    }
    acc.finish(lane, [&](int row, int c, float s) { part[(wave * NB + c) * RW + row] = s; });
    __syncthreads();
    ++sync;
    if (pub) {
      float t[kNW];
#pragma unroll
      for (int i = 0; i < kNW; ++i) t[i] = part[(i * NB + xc) * RW + xi];
      float y = a.scale * (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7])));
      if (a.shift != 0.f) y = fmaf(a.shift, pv[xc * LD + row0 + xi], y);
      put(xb + (int64_t)xc * nn + row0 + xi, pack(y, sync));
    }
  };
  auto zof = [&](int j, float rj) { return pre ? fmaf(a.dscale * a.d[min(j, n - 1)], rj, a.dshift * rj) : rj; };

  // cg.py:96-97: column norms of b (every workgroup, same order) and r = b / ||b||
  double w0[NB], w1[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    w0[c] = w1[c] = 0.0;
    if (c < B)
      for (int j = tid; j < kNT * KC; j += kNT) {
        const float bj = j < n ? a.b[(int64_t)j * a.b_rs + (int64_t)c * a.b_cs] : 0.f;
        rv[c * LD + j] = bj;
        w0[c] += (double)bj * (double)bj;
      }
  }
  put_sums<NB>(red1, w0);
  for (int i = tid; i < B * LD; i += kNT) pv[i] = 0.f;
  __syncthreads();
  st.mult = (float)sqrt(total<NB>(red1, col));
#pragma unroll
  for (int c = 0; c < NB; ++c)
    if (c < B) {
      const float m = norm_of(st.mult, c);
      for (int j = tid; j < n; j += kNT) rv[c * LD + j] /= m;
    }
  float ap[NB][KC], xo = 0.f;  // ap: zero from n on
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int t = 0; t < KC; ++t) ap[c][t] = 0.f;
  bool timeout = false;
  if (a.x0) {
    // cg.py:123: r0 = b_norm - A x0 (x0 as given); one exchange of A x0 through the odd buffer
    // (the first step writes the even one, so a fast workgroup never overwrites it)
    uint64_t* xb = a.xbuf + (int64_t)B * nn;
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (c < B)
        for (int j = tid; j < n; j += kNT) pv[c * LD + j] = a.x0[(int64_t)j * a.x0_rs + (int64_t)c * a.x0_cs];
    __syncthreads();
    product(xb);
    if (pub) xo = pv[xc * LD + row0 + xi];
    collect<NB, KC, CH>(xb, n, nn, B, sync + a.wait_offset, a.spin_limit, ap, &s_fail);
    __syncthreads();
    timeout = s_fail != 0;
    if (!timeout) {
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int t = 0; t < KC; ++t)
          if (c < B) rv[c * LD + tid + kNT * t] -= ap[c][t];
    }
  }
  // z = P r, p = z
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    w0[c] = 0.0;
    if (c < B)
      for (int j = tid; j < n; j += kNT) {
        const float rj = rv[c * LD + j], zj = zof(j, rj);
        pv[c * LD + j] = zj;
        w0[c] += (double)rj * (double)rj;
        w1[c] += (double)rj * (double)zj;
      }
  }
  put_sums<NB>(red2, w0, w1);
  __syncthreads();
  const bool writer = w == 0 && tid == 0;
  bool done = st.start(a, v, writer, total<NB>(red2, col), total<NB>(red2 + kNW * NB, col));
  while (!done && !timeout) {
    uint64_t* xb = a.xbuf + (int64_t)(st.k & 1) * B * nn;
    product(xb);
    collect<NB, KC, CH>(xb, n, nn, B, sync + a.wait_offset, a.spin_limit, ap, &s_fail);
    // p.Ap over all n entries (every workgroup, same order)
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      w0[c] = 0.0;
      if (c < B)
#pragma unroll
        for (int t = 0; t < KC; ++t) w0[c] += (double)pv[c * LD + tid + kNT * t] * (double)ap[c][t];
    }
    put_sums<NB>(red1, w0);
    __syncthreads();
    if (s_fail) {
      timeout = true;
      break;
    }
    st.set_alpha(total<NB>(red1, col));
    // r -= alpha Ap (all entries), gamma' = r.z, ||r||^2; x_own += alpha p_own
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      w0[c] = w1[c] = 0.0;
      if (c < B) {
        const float al = readlane_f32(st.alpha, c);
        if (pub && xc == c) xo = fmaf(al, pv[c * LD + row0 + xi], xo);
#pragma unroll
        for (int t = 0; t < KC; ++t) {
          const int j = tid + kNT * t;
          const float rj = fmaf(-al, ap[c][t], rv[c * LD + j]), zj = zof(j, rj);
          rv[c * LD + j] = rj;
          w0[c] += (double)rj * (double)rj;
          w1[c] += (double)rj * (double)zj;
        }
      }
    }
    put_sums<NB>(red2, w0, w1);
    __syncthreads();
    st.set_beta(total<NB>(red2, col), total<NB>(red2 + kNW * NB, col));
#pragma unroll
    for (int c = 0; c < NB; ++c)
      if (c < B) {
        const float be = readlane_f32(st.beta, c);
#pragma unroll
        for (int t = 0; t < KC; ++t) {
          const int j = tid + kNT * t;
          pv[c * LD + j] = fmaf(be, pv[c * LD + j], zof(j, rv[c * LD + j]));
        }
      }
    done = st.next(a, v, writer);
    __syncthreads();
  }
  if (timeout) {
    if (tid == 0) put(&v.ctrl->status, (int32_t)CK_ERR_TIMEOUT);
    if (writer) {
      v.ctrl->k = st.k;
      v.ctrl->done = 1;
    }
    return;
  }
  // cg.py:119: x and r back to the scale of b (own rows)
#pragma unroll
  for (int c = 0; c < NB; ++c)
    if (pub && xc == c) {
      const float m = readlane_f32(st.mult, c);
      a.x[(int64_t)(row0 + xi) * a.x_rs + (int64_t)c * a.x_cs] = xo * m;
      if (a.r) a.r[(int64_t)(row0 + xi) * a.r_rs + (int64_t)c * a.r_cs] = rv[c * LD + row0 + xi] * m;
    }
  if (w == 0) {
    st.store(a, v);
    if (tid == 0) __hip_atomic_fetch_max(&v.ctrl->status, (int32_t)st.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Clears the exchange tags and the status before a solve.
__global__ void fused_reset_kernel(uint64_t* xbuf, int64_t words, void* state) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (int64_t)gridDim.x * blockDim.x)
    xbuf[i] = 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) static_cast<ck_cg_ctrl*>(state)->status = CK_OK;
}

struct Plan {
  bool ok, res;
  int G, R, nn, kc;
  size_t lds;
};

template <int NB, int KC>
const void* resident_kernel(int kc) {
  if (kc == KC) return reinterpret_cast<const void*>(&fused_cg_kernel<NB, quads_of(KC), KC, true>);
  if constexpr (KC > 1) return resident_kernel<NB, KC - 1>(kc);
  return nullptr;
}

const void* kernel_of(const Plan& p, int nrhs) {
  if (!p.res) return reinterpret_cast<const void*>(&fused_cg_kernel<1, kStreamQuads, kStreamChunks, false>);
  return nrhs == 1   ? resident_kernel<1, kMaxChunks>(p.kc)
         : nrhs <= 4 ? resident_kernel<4, kMaxChunks>(p.kc)
                     : resident_kernel<8, kMaxChunks8>(p.kc);
}

// Workgroups that can be resident at once for (kernel, LDS bytes), cached per device.
int max_coresident(const void* kernel, size_t lds) {
  struct Entry {
    int dev;
    const void* kernel;
    size_t lds;
    int val;
  };
  static std::mutex mutex;
  static Entry cache[64];
  static int used = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(mutex);
  for (int i = 0; i < used; ++i)
    if (cache[i].dev == dev && cache[i].kernel == kernel && cache[i].lds == lds) return cache[i].val;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  int per = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kNT, lds) != hipSuccess) return 0;
  const int val = per * cus;
  if (used < 64) cache[used++] = Entry{dev, kernel, lds, val};
  return val;
}

// Workgroups and layout for order n, B columns; nblocks > 0 asks for that many workgroups.
Plan make_plan(int n, int B, int nblocks) {
  Plan p{};
  p.nn = (n + 3) / 4 * 4;
  if (n < 1 || B < 1 || B > kMaxRhs) return p;
  p.res = n <= kMaxResident;
  p.kc = (int)cdiv(n, 64 * kNW);
  if (!p.res && (B > 1 || n > 64 * kNW * kStreamChunks)) return p;
  if (B > 4 && p.kc > kMaxChunks8) return p;
  const int most = 4 * (p.res ? quads_of(p.kc) : kStreamQuads);
  int G = nblocks > 0 ? nblocks : 0;
  if (G < (int)cdiv(n, most)) G = (int)cdiv(n, most);
  if (G > kMaxBlocks) G = kMaxBlocks;
  p.R = (int)cdiv(n, G);
  p.G = (int)cdiv(n, p.R);
  p.lds = sizeof(float) * (size_t)2 * B * (kNT * (p.res ? p.kc : kStreamChunks) + 16);  // at most 129 KiB (2048 x 8)
  p.ok = true;
  return p;
}

// One workgroup takes the solve when nobody asks for more and the matrix fits its registers
// (a wait_offset concerns the waits of the exchange, which one workgroup does not have).
bool one_workgroup(int n, int B, int nblocks, int wait_offset) {
  return nblocks <= 1 && wait_offset == 0 && B <= 4 && n <= 64 * (B == 1 ? kOneChunks : kOneChunksMulti);
}

template <int KC>
void launch_one(const FusedArgs& a, hipStream_t s) {
  if (a.n > 64 * (KC - 1)) {
    if (a.nrhs == 1)
      hipLaunchKernelGGL((fused_one_kernel<1, KC>), dim3(1), dim3(kNT), 0, s, a);
    else if constexpr (KC <= kOneChunksMulti)
      hipLaunchKernelGGL((fused_one_kernel<4, KC>), dim3(1), dim3(kNT), 0, s, a);
  } else if constexpr (KC > 1) {
    launch_one<KC - 1>(a, s);
  }
}

size_t work_bytes_of(int nn, int B) { return sizeof(uint64_t) * (size_t)2 * B * nn; }

bool fused_eligible(const ck_op* A, const ck_op* P, int nrhs) {
  if (!A || A->kind != CK_OP_DENSE_F32 || !A->a || A->lda < A->n) return false;
  if (P && !(P->kind == CK_OP_DIAG_F32 && P->a && P->n == A->n)) return false;
  return nrhs >= 1 && nrhs <= kMaxRhs;
}

// The allocation-free entry point's exchange buffer: a file-scope device array, one copy per
// GPU, held until the process ends.  Host code takes its device address once per GPU with
// hipGetSymbolAddress (with that GPU current) and passes that address to the kernels; the
// array's name itself is only a host-side stand-in.  Every call on one GPU shares the array,
// so calls that overlap on one GPU race; the reset kernel clears its tags before each solve.
constexpr int kScratchWords = 8192;  // 64 KiB: 2 * nrhs * (n rounded up to 4) words, i.e. about n * nrhs <= 4096
__device__ __align__(256) uint64_t scratch[kScratchWords];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
uint64_t* g_scratch_ptr[kMaxDevices] = {};

int scratch_of_current_device(uint64_t** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return CK_ERR_HIP;
  if (dev < 0 || dev >= kMaxDevices) return CK_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return CK_ERR_HIP;
    g_scratch_ptr[dev] = static_cast<uint64_t*>(p);
  }
  *out = g_scratch_ptr[dev];
  return CK_OK;
}

// The solve with its exchange buffer at xbuf (xbuf_bytes available); shared by the entry points.
int fused_launch(const ck_op* A, const ck_op* P, int32_t nrhs, const float* b, int64_t b_rs, int64_t b_cs,
                 const float* x0, int64_t x0_rs, int64_t x0_cs, float* x, int64_t x_rs, int64_t x_cs, float* r,
                 int64_t r_rs, int64_t r_cs, void* state, float tol, int32_t max_iters, uint64_t* xbuf,
                 size_t xbuf_bytes, int32_t nblocks, int64_t spin_limit, int32_t wait_offset, int32_t cooperative,
                 void* stream) {
  if (!A || !b || !x || !state || !xbuf || max_iters < 0 || nblocks < 0 || wait_offset < 0) return CK_ERR_BAD_ARG;
  if (!fused_eligible(A, P, nrhs)) return CK_ERR_UNSUPPORTED;
  const int n = A->n;
  Plan pl = make_plan(n, nrhs, nblocks);
  if (!pl.ok) return CK_ERR_UNSUPPORTED;
  if (xbuf_bytes < work_bytes_of(pl.nn, nrhs)) return CK_ERR_WORKSPACE;
  const bool one = one_workgroup(n, nrhs, nblocks, wait_offset);
  const void* kernel = kernel_of(pl, nrhs);
  if (!one && pl.G > max_coresident(kernel, pl.lds)) return CK_ERR_UNSUPPORTED;
  FusedArgs a{};
  a.n = n;
  a.nn = pl.nn;
  a.nrhs = nrhs;
  a.G = one ? 1 : pl.G;
  a.R = pl.R;
  a.A = static_cast<const float*>(A->a);
  a.lda = A->lda;
  a.scale = A->scale;
  a.shift = A->shift;
  if (P) {
    a.d = static_cast<const float*>(P->a);
    a.dscale = P->scale;
    a.dshift = P->shift;
  }
  a.b = b;
  a.b_rs = b_rs;
  a.b_cs = b_cs;
  a.x0 = x0;
  a.x0_rs = x0_rs;
  a.x0_cs = x0_cs;
  a.x = x;
  a.x_rs = x_rs;
  a.x_cs = x_cs;
  a.r = r;
  a.r_rs = r_rs;
  a.r_cs = r_cs;
  a.state = state;
  a.tol = tol;
  a.max_iters = max_iters;
  a.xbuf = xbuf;
  a.spin_limit = spin_limit > 0 ? spin_limit : kDefaultSpin;
  a.wait_offset = (uint32_t)wait_offset;
  hipStream_t s = (hipStream_t)stream;
  if (one) {
    launch_one<kOneChunks>(a, s);
    CK_CHECK_LAUNCH();
    return CK_OK;
  }
  const int64_t words = (int64_t)2 * nrhs * pl.nn;
  const unsigned rblocks = (unsigned)(cdiv(words, 1024) < 64 ? cdiv(words, 1024) : 64);
  hipLaunchKernelGGL(fused_reset_kernel, dim3(rblocks), dim3(256), 0, s, a.xbuf, words, state);
  CK_CHECK_LAUNCH();
  void* args[] = {&a};
  // every workgroup fits at once (checked above); a cooperative launch also guarantees that
  // they are resident together, a plain one costs about 20 us less per solve -- with the
  // bounded waits, a workgroup that started late makes the others wait, never hang
  const hipError_t e = cooperative
                           ? hipLaunchCooperativeKernel(kernel, dim3(pl.G), dim3(kNT), args, (unsigned)pl.lds, s)
                           : hipLaunchKernel(kernel, dim3(pl.G), dim3(kNT), args, (unsigned)pl.lds, s);
  if (e != hipSuccess) return CK_ERR_HIP;
  return CK_OK;
}

}  // namespace

extern "C" {

size_t ck_cg_fused_workspace_bytes(int64_t n, int32_t nrhs) {
  if (n < 1 || nrhs < 1) return 0;
  return work_bytes_of((int)((n + 3) / 4 * 4), nrhs);
}

int ck_cg_fused_supported(const ck_op* A, const ck_op* P, int32_t nrhs) {
  if (!fused_eligible(A, P, nrhs)) return CK_ERR_UNSUPPORTED;
  Plan p = make_plan(A->n, nrhs, 0);
  return p.ok ? CK_OK : CK_ERR_UNSUPPORTED;
}

int32_t ck_cg_fused_workgroups(const ck_op* A, const ck_op* P, int32_t nrhs, int32_t nblocks, int32_t wait_offset) {
  if (!fused_eligible(A, P, nrhs)) return 0;
  const Plan p = make_plan(A->n, nrhs, nblocks);
  return !p.ok ? 0 : one_workgroup(A->n, nrhs, nblocks, wait_offset) ? 1 : p.G;
}

int32_t ck_device_cus(int32_t device) {
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess) return cus;
  (void)hipGetLastError();  // not the next launch's error
  return 0;
}

int ck_cg_fused(const ck_op* A, const ck_op* P, int32_t nrhs, const float* b, int64_t b_rs, int64_t b_cs,
                const float* x0, int64_t x0_rs, int64_t x0_cs, float* x, int64_t x_rs, int64_t x_cs, float* r,
                int64_t r_rs, int64_t r_cs, void* state, float tol, int32_t max_iters, void* work,
                size_t work_bytes, int32_t nblocks, int64_t spin_limit, int32_t wait_offset, int32_t cooperative,
                void* stream) {
  if (!work || (reinterpret_cast<uintptr_t>(work) & 7) != 0) return !work ? CK_ERR_BAD_ARG : CK_ERR_WORKSPACE;
  return fused_launch(A, P, nrhs, b, b_rs, b_cs, x0, x0_rs, x0_cs, x, x_rs, x_cs, r, r_rs, r_cs, state, tol, max_iters,
                      static_cast<uint64_t*>(work), work_bytes, nblocks, spin_limit, wait_offset, cooperative, stream);
}

int ck_cg_fused_noalloc(const ck_op* A, const ck_op* P, int32_t nrhs, const float* b, int64_t b_rs, int64_t b_cs,
                        const float* x0, int64_t x0_rs, int64_t x0_cs, float* x, int64_t x_rs, int64_t x_cs, float* r,
                        int64_t r_rs, int64_t r_cs, void* state, float tol, int32_t max_iters, int32_t nblocks,
                        int64_t spin_limit, int32_t wait_offset, int32_t cooperative, void* stream) {
  uint64_t* ptr = nullptr;
  const int st = scratch_of_current_device(&ptr);
  if (st != CK_OK) return st;
  return fused_launch(A, P, nrhs, b, b_rs, b_cs, x0, x0_rs, x0_cs, x, x_rs, x_cs, r, r_rs, r_cs, state, tol, max_iters,
                      ptr, sizeof(scratch), nblocks, spin_limit, wait_offset, cooperative, stream);
}

size_t ck_cg_fused_noalloc_max_bytes(void) { return sizeof(scratch); }

}  // extern "C"
