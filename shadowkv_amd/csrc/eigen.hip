// Leading eigenpairs of a symmetric positive semidefinite matrix [n, n] in fp32, n <= 1024: the small
// dense problem inside the prompt factorisation (the keys' Gram matrix; the reference takes an SVD of
// the keys, models/kvcache/shadow.py:426). Four kernels:
//
//   tridiag_kernel   A = Q T Q^T by Householder reflections, one after another (LAPACK's unblocked
//                    scheme, Golub & Van Loan 8.3.1). The matrix stays in registers, 8 columns per
//                    wave, the waves of one problem on the CUs of one XCD.
//   bisect_kernel    the R largest eigenvalues of T: Sturm counts in fp64 (the number of sign changes
//                    of the leading principal minors), one workgroup per eigenvalue.
//   (in it)          their eigenvectors from T by a twisted factorisation in fp64 (Dhillon & Parlett):
//                    forward and backward pivots, joined where the twisted pivot is smallest.
//   backtransform    Q times each vector, one wave per vector.
//
// Bound: n sequential steps. A blocked library reduction pays several launches and several passes over
// the trailing matrix per step (16 to 20 ms at n = 1024). Here a step costs one exchange through the
// XCD's L2: column j's owner publishes {(A v)_j, A[i + 1][j]}, and every wave computes the update
// vector w, the next column and its reflection redundantly from the gathered 2 n numbers. The words
// are their own flags (the exchange area starts as all ones, each step has its own row), so there is
// no counter, no fence and no second trip. The stores are workgroup-scope (they stay in the L2 that the
// problem's workgroups share; agent-scope stores go through to memory and cost 4.4 against 2.65 ms in
// all), the polling loads agent-scope (past the L1). Every wait is bounded: a workgroup that waits too long
// gives up for good, the problem's status says so and the caller takes another way.
//
// MI355X, rank 160, us in all: n = 1024 2190 (the reduction 1640, 1.6 a step; the eigenpairs of T 360; the
// back transformation 180), n = 512 848, n = 256 386 (1.0 a step: the exchange and the chain of
// reductions alone); rocSOLVER's full decomposition 19600, 10400, 4900.
#include <mutex>
#include <type_traits>

#include "wave_reduce.h"

namespace {

constexpr int kCols = 8;        // columns per wave
constexpr int kWgWaves = 4;     // waves per workgroup
constexpr int kXccIds = 8;
constexpr int kHwRegXccId = (3 << 11) | (0 << 6) | 20;  // s_getreg_b32 hwreg(HW_REG_XCC_ID, 0, 4)
// Polls of one wait, 28 ms at 0.22 us: longer than workgroups of other kernels keep this one's off the CUs, and not much
// more than the full decomposition costs that the caller takes then. Three processes whose reductions meet on one
// device (n = 1024; two fit beside one another) paid 114 ms a call at four times as many, 3.4 to 4.9 (one in ten 33) now.
constexpr int kPollLimit = 1 << 17;
constexpr int kMaxN = 1024;

struct EigenArgs {
  const float* a;  // [batch][n][n]
  int n, rank;
  uint64_t* xchg;     // [batch][n][npad]
  float* v;           // [batch][n][npad] reflection vectors
  float* tau;         // [batch][npad]
  float* d;           // [batch][npad] diagonal of T (scaled)
  float* e;           // [batch][npad] off-diagonal
  float* scale;       // [batch] power of two that undoes the scaling of T
  uint32_t* tickets;  // [8]
  int32_t* status;    // [batch] 1 when the problem is reduced; bit 1: a wait ran out
  float* w;           // [batch][rank] eigenvalues, descending
  float* vt;          // [batch][rank][n] eigenvectors
  float* z;           // [batch][rank][npad] eigenvectors of T
  int batch;
};

// Element idx of a vector held as x[r] = element 64 r + lane, idx wave-uniform with idx / 64 in [LO, HI].
template <int LO, int HI, class Col>
__device__ __forceinline__ float pick(const Col& x, int idx) {
  float v = x[LO];
#pragma unroll
  for (int r = LO + 1; r <= HI; ++r) v = (idx >> 6) == r ? x[r] : v;
  return skv::lane_value(v, idx & 63);
}

// f(0), f(1), ... with compile-time arguments (a loop variable that indexes registers before any
// unrolling pass has run).
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

template <int NR>
struct Reduction {
  typedef float Col __attribute__((ext_vector_type(NR)));
  static constexpr int kWavesAll = 8 * NR;  // waves of a problem: 64 NR columns, 8 per wave
  static constexpr int kPad = 64 * NR;
  // (Vector types, not arrays: they stay in registers whatever the order of the unrolling passes.)
  Col A[kCols];  // column s * kWavesAll + wid, row 64 r + lane
  Col a;          // the column being reduced
  float nn;       // squares of the column below its first off-diagonal element
  int wid, lane, wave;
  bool dead = false;   // a wait has run out

  __device__ __forceinline__ static float clean(float x) { return x != x ? __uint_as_float(0x7fc00000u) : x; }

  // Squares of the column below its first off-diagonal element, column i.
  template <int R0>
  __device__ __forceinline__ float tail_norm(int i) const {
    float t = 0.f;
#pragma unroll
    for (int r = R0; r < NR; ++r) t = fmaf(64 * r + lane > i + 1 ? a[r] : 0.f, a[r], t);
    return skv::wave_sum_dpp(t);
  }

  // Steps i in [PH * kWavesAll, (PH + 1) * kWavesAll): columns of slots below PH and the rows above are done.
  template <int PH>
  __device__ __forceinline__ void phase(const EigenArgs& g, int b, float2 (*pc)[kPad]) {
    constexpr int R0 = PH * kWavesAll / 64;                          // first live row block
    constexpr int R1 = ((PH + 1) * kWavesAll) / 64 < NR - 1 ? ((PH + 1) * kWavesAll) / 64 : NR - 1;
    const int i1 = min(g.n - 1, (PH + 1) * kWavesAll);
    for (int i = PH * kWavesAll; i < i1; ++i) {
      // Reflection of column i: v = (0 .., 1, x), H = I - tau v v^T maps the column to (.., beta, 0 ..).
      const float di = pick<R0, R1>(a, i), alpha = pick<R0, R1>(a, i + 1);
      float beta = alpha, tau = 0.f, inv = 0.f;
      if (nn > 1e-36f) {
        // 1 / |beta| and 1 / (alpha - beta) from the hardware estimates and a Newton step each: the
        // divisions and the square root would lie on every step's critical path.
        const float sq = fmaf(alpha, alpha, nn);
        float rs = __builtin_amdgcn_rsqf(sq);
        rs = fmaf(0.5f * rs, fmaf(-sq * rs, rs, 1.f), rs);
        beta = -copysignf(sq * rs, alpha);
        tau = fmaf(fabsf(alpha), rs, 1.f);  // (beta - alpha) / beta
        const float den = alpha - beta;
        inv = __builtin_amdgcn_rcpf(den);
        inv = fmaf(fmaf(-den, inv, 1.f), inv, inv);
      }
      Col v;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const int row = 64 * r + lane;
        v[r] = r < R0 ? 0.f : row > i + 1 ? a[r] * inv : row == i + 1 ? 1.f : 0.f;
      }
      // Own columns: (A v)_j and A[i + 1][j], summed over the wave so that lane t < 8 holds the product
      // of slot t and lane 8 + t its element; then published.
      float f[2 * kCols];
      const bool mine = lane == ((i + 1) & 63);
      static_for<0, kCols>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        float p = 0.f, c = 0.f;
        if constexpr (s >= PH) {
#pragma unroll
          for (int r = R0; r < NR; ++r) p = fmaf(A[s][r], v[r], p);
          c = A[s][R0];
#pragma unroll
          for (int r = R0 + 1; r <= R1; ++r) c = ((i + 1) >> 6) == r ? A[s][r] : c;
        }
        f[s] = p;
        f[kCols + s] = mine ? c : 0.f;
      });
      skv::fold<16, 0x140>(f, lane & 8);
      skv::fold<8, 0x141>(f, lane & 4);
      skv::fold<4, 0x1B>(f, lane & 2);
      skv::fold<2, 0xB1>(f, lane & 1);
      {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[0]), __float_as_uint(f[0]), false, false);
        f[0] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        const auto y = __builtin_amdgcn_permlane16_swap(__float_as_uint(f[0]), __float_as_uint(f[0]), false, false);
        f[0] = __uint_as_float(y[0]) + __uint_as_float(y[1]);
      }
      uint64_t* row = g.xchg + (static_cast<int64_t>(b) * g.n + i) * kPad;
      {
        const int j = (lane & 7) * kWavesAll + wid;
        if (lane < 16 && j > i)
          __hip_atomic_store(reinterpret_cast<uint32_t*>(row + j) + (lane >> 3), __float_as_uint(clean(f[0])),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      // Gather: the workgroup's wave q takes a quarter of the rows.
      float2 (*buf)[kPad] = pc + (i & 1);
      constexpr int kQ = kPad / kWgWaves;             // rows per wave
      constexpr int kPer = kQ >= 64 ? kQ / 64 : 1;    // entries per lane
      uint64_t got[kPer];
      const int r0 = wave * kQ + lane;
      const bool in = kQ >= 64 || lane < kQ;
      for (int tries = 0;; ++tries) {
        bool all = true;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
          const int rr = r0 + 64 * u;
          got[u] = in && rr > i ? __hip_atomic_load(row + rr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
          all = all && static_cast<uint32_t>(got[u]) != 0xffffffffu && static_cast<uint32_t>(got[u] >> 32) != 0xffffffffu;
        }
        if (__all(all) || dead) break;
        if (tries >= kPollLimit) {
          dead = true;
          if (lane == 0) atomicOr(&g.status[b], 2);
        }
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u)
        if (in)
          (*buf)[r0 + 64 * u] = make_float2(__uint_as_float(static_cast<uint32_t>(got[u])),
                                            __uint_as_float(static_cast<uint32_t>(got[u] >> 32)));
      __syncthreads();  // (the other half of pc is written again only after the next one)
      Col p = {}, c = {};
      if (wid == i % kWavesAll) {  // this step's scribe (its stores overlap the rest of the step)
        float* vr = g.v + (static_cast<int64_t>(b) * g.n + i) * kPad;
#pragma unroll
        for (int r = 0; r < NR; ++r) vr[64 * r + lane] = v[r];
        if (lane == 0) {
          g.tau[b * kPad + i] = tau;
          g.d[b * kPad + i] = di;
          g.e[b * kPad + i] = beta;
        }
      }
      float al = 0.f;
#pragma unroll
      for (int r = R0; r < NR; ++r) {
        const float2 t = (*buf)[64 * r + lane];
        p[r] = t.x;
        c[r] = t.y;
        al = fmaf(t.x, v[r], al);
      }
      al = skv::wave_sum_dpp(al);
      const float h = 0.5f * tau * al;
#pragma unroll
      for (int r = R0; r < NR; ++r) p[r] = tau * fmaf(-h, v[r], p[r]);  // w = tau (A v - (tau v.Av / 2) v)
      const float wn = pick<R0, R1>(p, i + 1);
#pragma unroll
      for (int r = R0; r < NR; ++r) a[r] = fmaf(-v[r], wn, c[r] - p[r]);  // v[i + 1] = 1
      // The next reflection's norm, its reduction overlapping the update of the columns below.
      nn = tail_norm<R0>(i + 1);
      static_for<PH, kCols>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        const int j = s * kWavesAll + wid;
        constexpr int kSpan = kWavesAll >= 64 ? kWavesAll / 64 : 1;
        constexpr int lo = s * kWavesAll / 64;
        float vs = v[lo], wsx = p[lo < R0 ? R0 : lo];
#pragma unroll
        for (int r = 1; r < kSpan; ++r) {
          vs = (j >> 6) == lo + r ? v[lo + r] : vs;
          wsx = (j >> 6) == lo + r ? p[lo + r] : wsx;
        }
        const float vj = skv::lane_value(vs, j & 63), wj = skv::lane_value(wsx, j & 63);
#pragma unroll
        for (int r = R0; r < NR; ++r) A[s][r] = fmaf(-v[r], wj, fmaf(-p[r], vj, A[s][r]));
      });
    }
    if constexpr (PH + 1 < kCols) {
      if (i1 < g.n - 1) phase<PH + 1>(g, b, pc);
    }
  }
};

// (Compiled for one wave per SIMD, so that the 8 columns, 128 registers at 1024 rows, stay in registers with all that
// the steps hold; two waves of 4 columns would do the redundant vector work twice. At 232 registers two
// workgroups still fit on a CU, 64 on an XCD.)
// A workgroup takes its part by its order of arrival on its XCD: problem b runs on XCD b, its
// 2 NR workgroups spread over the CUs of an idle device by the dispatcher (a request for LDS that forces one per CU
// changes nothing).
template <int NR>
__global__ void __launch_bounds__(kWgWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 1)))
tridiag_kernel(EigenArgs g) {
  using Red = Reduction<NR>;
  __shared__ float2 pc[2][Red::kPad];
  __shared__ int part;
  const int b = static_cast<int>(__builtin_amdgcn_s_getreg(kHwRegXccId) & 15u);
  if (b >= g.batch) return;
  if (threadIdx.x == 0) part = static_cast<int>(atomicAdd(&g.tickets[b], 1u));
  __syncthreads();
  if (part >= 2 * NR) return;
  Red red;
  red.lane = threadIdx.x & 63;
  red.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  red.wid = __builtin_amdgcn_readfirstlane(part * kWgWaves + red.wave);
  const int n = g.n, lane = red.lane;
  const float* A = g.a + static_cast<int64_t>(b) * n * n;
  // Scale to a largest diagonal entry in [0.5, 1) (the largest entry of a semidefinite matrix): exact.
  float mx = 0.f;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int row = 64 * r + lane;
    mx = fmaxf(mx, row < n ? fabsf(A[static_cast<int64_t>(row) * n + row]) : 0.f);
  }
  mx = skv::wave_max_dpp(mx);
  int ex = 0;
  frexpf(mx, &ex);
  const bool ok = mx > 0.f && mx < INFINITY && ex > -100 && ex < 100;  // uniform over the problem
  if (!ok) return;
  const float sc = ldexpf(1.f, -ex);
  static_for<0, kCols>([&](auto sv) {
    constexpr int s = decltype(sv)::value;
    const int j = s * Red::kWavesAll + red.wid;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int row = 64 * r + lane;
      red.A[s][r] = row < n && j < n ? sc * A[static_cast<int64_t>(j) * n + row] : 0.f;
    }
  });
#pragma unroll
  for (int r = 0; r < NR; ++r) red.a[r] = 64 * r + lane < n ? sc * A[64 * r + lane] : 0.f;
  red.nn = red.template tail_norm<0>(0);
  red.template phase<0>(g, b, pc);
  if (red.wid == 0) {
    float last = 0.f;
#pragma unroll
    for (int r = 0; r < NR; ++r) last = ((n - 1) >> 6) == r ? red.a[r] : last;
    last = skv::lane_value(last, (n - 1) & 63);
    if (lane == 0) {
      g.d[b * Red::kPad + n - 1] = last;
      g.e[b * Red::kPad + n - 1] = 0.f;
      g.scale[b] = ldexpf(1.f, ex);
      atomicOr(&g.status[b], 1);
    }
  }
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One workgroup per eigenpair of T: eigenvalue k of the descending order, then its vector. Bound by the
// chain of n fp64 recurrence steps of every pass, so a pass takes as many points as run beside one
// another without slowing the chain (one wave per SIMD): 256 points in 7 passes, where one wave took 9
// passes of 64. The pivots of the twisted factorisation are quotients of neighbouring minors, taken in
// parallel after the same two-term recurrence: dividing along the chain cost five times as much.
constexpr int kPoints = 256;
constexpr int kPointWaves = kPoints / 64;

__global__ void __launch_bounds__(kPoints) bisect_kernel(EigenArgs g, int npad) {
  const int b = blockIdx.y, k = blockIdx.x, n = g.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (g.status[b] != 1) return;
  __shared__ double red[2][kPointWaves];
  __shared__ int votes[2][kPointWaves];
  __shared__ double2 de[kMaxN];  // diagonal, square of the off-diagonal before it
  __shared__ double es[kMaxN], q0[kMaxN], q1[kMaxN];  // pivots from the front and from the back
  __shared__ double2 pp[2][kMaxN];                     // minors: (p, the one before it), in one scale
  const float* d = g.d + b * npad;
  const float* e = g.e + b * npad;
  double lo = 1e300, hi = -1e300;  // Gershgorin
  for (int i = tid; i < n; i += kPoints) {
    const double di = d[i], ei = i + 1 < n ? e[i] : 0.f, em = i > 0 ? e[i - 1] : 0.f;
    de[i] = make_double2(di, em * em);
    es[i] = ei;
    const double s = fabs(ei) + fabs(em);
    lo = fmin(lo, di - s);
    hi = fmax(hi, di + s);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o, 64));
    hi = fmax(hi, __shfl_xor(hi, o, 64));
  }
  if (lane == 0) {
    red[0][wave] = lo;
    red[1][wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPointWaves; ++i) {
    lo = fmin(lo, red[0][i]);
    hi = fmax(hi, red[1][i]);
  }
  const double norm = fmax(fabs(lo), fabs(hi));
  lo -= 1e-12 * norm;
  hi += 1e-12 * norm;
  // Past n up to a multiple of 8: a factor that changes neither sign nor count.
  const int n8 = (n + 7) / 8 * 8;
  for (int i = n + tid; i < n8; i += kPoints) de[i] = make_double2(hi + norm, 0.0);
  __syncthreads();
  auto rescale = [](double& p0, double& p1) {  // (powers of two would do; only the ratio matters)
    const double m = fmax(fabs(p0), fabs(p1));
    const double f = m > 1e100 ? 1e-100 : m < 1e-100 ? 1e100 : 1.0;
    p0 *= f;
    p1 = m == 0.0 ? 1e-100 : p1 * f;
  };
  // The interior points split [lo, hi] into 257 parts; lambda_k >= x when at least k + 1 eigenvalues are
  // not below x, and the eigenvalues below x are the sign changes of the minors p_i (an exact zero
  // between two nonzero minors counts once with either sign). 7 passes: 257^-7 = 1e-17 of the width
  // (3e-15 is not enough for the vectors of a spectrum that ends in rounding noise).
  for (int pass = 0; pass < 7; ++pass) {
    const double step = (hi - lo) / (kPoints + 1);
    const double x = lo + step * (tid + 1);
    double p0 = 0.0, p1 = 1.0;
    int below = 0;
    // Eight steps at a time, the next eight's coefficients requested ahead (read as they are needed,
    // their LDS latency is half of a step).
    double2 next[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) next[u] = de[u];
    for (int i = 0; i < n8; i += 8) {
      double2 t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = next[u];
      const int ahead = min(i + 8, n8 - 8);
#pragma unroll
      for (int u = 0; u < 8; ++u) next[u] = de[ahead + u];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double p = fma(t[u].x - x, p1, -t[u].y * p0);
        below += static_cast<int>(static_cast<uint32_t>(__double2hiint(p) ^ __double2hiint(p1)) >> 31);
        p0 = p1;
        p1 = p;
      }
      rescale(p0, p1);
    }
    // The threads' points ascend: those at most lambda_k form a prefix.
    const int mine = __popcll(__ballot(n - below >= k + 1));
    if (lane == 0) votes[pass & 1][wave] = mine;
    __syncthreads();
    int c = 0;
#pragma unroll
    for (int i = 0; i < kPointWaves; ++i) c += votes[pass & 1][i];
    const double nlo = c > 0 ? lo + step * c : lo, nhi = c < kPoints ? lo + step * (c + 1) : hi;
    lo = nlo;
    hi = nhi;
  }
  const double lam = 0.5 * (lo + hi);
  // Minors from both ends: thread 0 forward, thread 1 backward. An exact zero becomes a tiny pivot.
  const double tiny = 1e-30 * norm + 1e-300;
  if (tid < 2) {
    double p0 = 0.0, p1 = 1.0;
    double2* out = pp[tid];
    auto coef = [&](int t) {  // of the t-th step: diagonal, square of the off-diagonal before it
      const int i = tid ? n - 1 - t : t;
      const double e2 = tid ? es[i] * es[i] : de[i].y;
      return make_double2(de[i].x - lam, t == 0 ? 0.0 : e2);
    };
    auto advance = [&](int t, const double2& c) {
      double p = fma(c.x, p1, -c.y * p0);
      if (p == 0.0) p = -tiny * p1;
      out[tid ? n - 1 - t : t] = make_double2(p, p1);
      p0 = p1;
      p1 = p;
    };
    int t = 0;
    if (n >= 8) {
      double2 next[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) next[u] = coef(u);
      for (; t + 8 <= n; t += 8) {
        double2 c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = next[u];
        const int ahead = min(t + 8, n - 8);
#pragma unroll
        for (int u = 0; u < 8; ++u) next[u] = coef(ahead + u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) advance(t + u, c[u]);
        rescale(p0, p1);
      }
    }
    for (; t < n; ++t) advance(t, coef(t));
  }
  __syncthreads();
  for (int i = tid; i < n; i += kPoints) {
    double f = pp[0][i].x / pp[0][i].y, r = pp[1][i].x / pp[1][i].y;
    q0[i] = fabs(f) < tiny ? -tiny : f;
    q1[i] = fabs(r) < tiny ? -tiny : r;
  }
  __syncthreads();
  double best = 1e300;
  int at = 0;
  for (int i = tid; i < n; i += kPoints) {
    const double gm = fabs(q0[i] + q1[i] - (de[i].x - lam));
    if (gm < best) {
      best = gm;
      at = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ob = __shfl_xor(best, o, 64);
    const int oa = __shfl_xor(at, o, 64);
    if (ob < best || (ob == best && oa < at)) {
      best = ob;
      at = oa;
    }
  }
  if (lane == 0) {
    red[0][wave] = best;
    votes[0][wave] = at;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPointWaves; ++i) {
    const double ob = red[0][i];
    const int oa = votes[0][i];
    if (ob < best || (ob == best && oa < at)) {
      best = ob;
      at = oa;
    }
  }
  // Ratios of neighbouring entries, then their running products away from the twist.
  for (int i = tid; i < n; i += kPoints) {
    const double up = i + 1 < n ? -es[i] / q0[i] : 0.0;   // z[i] / z[i + 1], i < at
    const double dn = i > 0 ? -es[i - 1] / q1[i] : 0.0;   // z[i] / z[i - 1], i > at
    q0[i] = i < at ? up : i > at ? dn : 1.0;
  }
  __syncthreads();
  double* zz = q1;
  if (tid < 2) {
    double z = 1.0;
    const int steps = tid ? n - 1 - at : at, dir = tid ? 1 : -1;
    const double* src = q0 + at;
    double* dst = zz + at;
    int t = 1;
    for (; t + 8 <= steps + 1; t += 8) {
      double r[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) r[u] = src[dir * (t + u)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        z *= r[u];
        dst[dir * (t + u)] = z;
      }
    }
    for (; t <= steps; ++t) {
      z *= src[dir * t];
      dst[dir * t] = z;
    }
    if (tid == 0) zz[at] = 1.0;
  }
  __syncthreads();
  double ss = 0.0;
  for (int i = tid; i < n; i += kPoints) ss = fma(zz[i], zz[i], ss);
  ss = wave_sum_f64(ss);
  if (lane == 0) red[1][wave] = ss;
  __syncthreads();
  ss = 0.0;
#pragma unroll
  for (int i = 0; i < kPointWaves; ++i) ss += red[1][i];
  const double inv = 1.0 / sqrt(ss);
  float* z = g.z + (static_cast<int64_t>(b) * g.rank + k) * npad;
  for (int i = tid; i < npad; i += kPoints) z[i] = i < n ? static_cast<float>(zz[i] * inv) : 0.f;
  if (tid == 0) g.w[b * g.rank + k] = static_cast<float>(lam * static_cast<double>(g.scale[b]));
}

// vt[k] = H_0 H_1 ... H_{n-2} z_k, one wave per vector, the reflections requested kAhead steps ahead in
// 16-byte loads (the loads bound it: 4-byte ones took 227 against 180 us at n = 1024; two reflections
// per round of reductions were no faster).
template <int NR>
__global__ void __launch_bounds__(64) backtransform_kernel(EigenArgs g) {
  constexpr int kPad = 64 * NR, kAhead = 8;
  const int b = blockIdx.y, k = blockIdx.x, n = g.n, lane = threadIdx.x;
  if (g.status[b] != 1) return;
  const float* vb = g.v + static_cast<int64_t>(b) * n * kPad;
  const float* tau = g.tau + b * kPad;
  // Register r holds row row0(r) = 64 VL (r / VL) + VL lane + r % VL: VL rows, one load, side by side.
  constexpr int VL = NR >= 4 ? 4 : 2;
  typedef float Vec __attribute__((ext_vector_type(VL)));
  Vec z[NR / VL];
  const float* zs = g.z + (static_cast<int64_t>(b) * g.rank + k) * kPad + VL * lane;
#pragma unroll
  for (int r = 0; r < NR / VL; ++r) z[r] = *reinterpret_cast<const Vec*>(zs + 64 * VL * r);
  Vec v[kAhead][NR / VL];
  float t[kAhead];
  auto load = [&](int i, Vec* dst, float& tt) {
    const int ii = max(i, 0);
#pragma unroll
    for (int r = 0; r < NR / VL; ++r)
      dst[r] = *reinterpret_cast<const Vec*>(vb + static_cast<int64_t>(ii) * kPad + VL * lane + 64 * VL * r);
    tt = i < 0 ? 0.f : tau[ii];
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u) load(n - 2 - u, v[u], t[u]);
  for (int i = n - 2; i >= 0; i -= kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      float s = 0.f;
#pragma unroll
      for (int r = 0; r < NR; ++r) s = fmaf(v[u][r / VL][r % VL], z[r / VL][r % VL], s);
      s = skv::wave_sum_dpp(s) * t[u];
#pragma unroll
      for (int r = 0; r < NR; ++r) z[r / VL][r % VL] = fmaf(-s, v[u][r / VL][r % VL], z[r / VL][r % VL]);
      load(i - u - kAhead, v[u], t[u]);
    }
  }
  float* out = g.vt + (static_cast<int64_t>(b) * g.rank + k) * n;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int row = 64 * VL * (r / VL) + VL * lane + r % VL;
    if (row < n) out[row] = z[r / VL][r % VL];
  }
}

__global__ void __launch_bounds__(256) prepare_kernel(ulonglong2* xchg, int64_t count, uint32_t* tickets,
                                                      int32_t* status, int batch) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < count) xchg[i] = ulonglong2{~0ull, ~0ull};
  if (i < kXccIds) tickets[i] = 0;
  if (i < batch) status[i] = 0;
}

// Reductions of one device run one after another, whatever their streams: the 2 NR workgroups of a problem
// wait for one another, an XCD holds 64 of them, and of three calls at n = 1024 each could hold a share and
// wait until it gives up (three threads: 156 ms a round of calls, most without a result; in turn 5.2). Two beside each
// other were no faster than in turn. A captured call is not ordered: its event would belong to the graph.
struct ReductionOrder {
  std::mutex mutex;
  hipEvent_t done = nullptr;  // after the newest reduction
  bool recorded = false;
};
ReductionOrder g_order[64];

int blocks_of(int n) { return n <= 128 ? 2 : n <= 256 ? 4 : n <= 512 ? 8 : 16; }

struct Layout {
  int64_t xchg, v, tau, d, e, scale, tickets, z, total;
};
Layout layout(int batch, int n, int rank) {
  const int64_t pad = 64 * blocks_of(n);
  Layout l;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  l.xchg = take(batch * n * pad * 8);
  l.v = take(batch * n * pad * 4);
  l.tau = take(batch * pad * 4);
  l.d = take(batch * pad * 4);
  l.e = take(batch * pad * 4);
  l.scale = take(batch * 4);
  l.tickets = take(kXccIds * 4);
  l.z = take(static_cast<int64_t>(batch) * rank * pad * 4);
  l.total = at;
  return l;
}

}  // namespace

extern "C" int64_t skv_sym_eig_workspace_bytes(int batch, int n, int rank) {
  if (batch < 1 || batch > kXccIds || n < 2 || n > kMaxN || rank < 1 || rank > n) return 0;
  return layout(batch, n, rank).total;
}

extern "C" int skv_sym_eig_top(const float* a, int batch, int n, int rank, float* w, float* vt, int32_t* status,
                               void* workspace, int64_t workspace_bytes, void* stream) {
  const char* what = "sym_eig_top";
  if (!a || !w || !vt || !status || !workspace) {
    skv_set_error("%s: null pointer", what);
    return SKV_EINVAL;
  }
  if (batch < 1 || batch > kXccIds || n < 2 || n > kMaxN || rank < 1 || rank > n) {
    skv_set_error("%s: batch=%d (1..%d) n=%d (2..%d) rank=%d", what, batch, kXccIds, n, kMaxN, rank);
    return SKV_EUNSUPPORTED;
  }
  const Layout l = layout(batch, n, rank);
  if ((reinterpret_cast<uintptr_t>(workspace) & 15) || workspace_bytes < l.total) {
    skv_set_error("%s: workspace of %lld bytes, 16-byte aligned (%lld needed)", what, (long long)workspace_bytes,
                  (long long)l.total);
    return SKV_EINVAL;
  }
  char* ws = static_cast<char*>(workspace);
  auto f32 = [&](int64_t off) { return reinterpret_cast<float*>(ws + off); };
  EigenArgs g{a, n, rank, reinterpret_cast<uint64_t*>(ws + l.xchg), f32(l.v), f32(l.tau), f32(l.d), f32(l.e),
              f32(l.scale), reinterpret_cast<uint32_t*>(ws + l.tickets), status, w, vt, f32(l.z), batch};
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int nr = blocks_of(n);
  const int64_t words = static_cast<int64_t>(batch) * n * 64 * nr / 2;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  int device = 0;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess || hipGetDevice(&device) != hipSuccess || device < 0 ||
      device >= 64) {
    skv_set_error("%s: no stream state or device", what);
    return SKV_ELAUNCH;
  }
  hipLaunchKernelGGL(prepare_kernel, dim3(static_cast<unsigned>((words + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<ulonglong2*>(ws + l.xchg), words, g.tickets, status, batch);
  const bool ordered = capture == hipStreamCaptureStatusNone;
  ReductionOrder& order = g_order[device];
  auto run = [&](auto nrv) {
    constexpr int NR = decltype(nrv)::value;
    std::unique_lock<std::mutex> lock(order.mutex, std::defer_lock);
    if (ordered) {
      lock.lock();
      if (!order.done && hipEventCreateWithFlags(&order.done, hipEventDisableTiming) != hipSuccess) return false;
      if (order.recorded && hipStreamWaitEvent(s, order.done, 0) != hipSuccess) return false;
    }
    // 64 workgroups per XCD where the dispatcher deals them round robin, at most 32 of them with a part.
    hipLaunchKernelGGL(tridiag_kernel<NR>, dim3(512), dim3(kWgWaves * 64), 0, s, g);
    if (ordered) {
      if (hipEventRecord(order.done, s) != hipSuccess) return false;
      order.recorded = true;
      lock.unlock();
    }
    hipLaunchKernelGGL(bisect_kernel, dim3(rank, batch), dim3(kPoints), 0, s, g, 64 * NR);
    hipLaunchKernelGGL(backtransform_kernel<NR>, dim3(rank, batch), dim3(64), 0, s, g);
    return true;
  };
  const bool launched = nr == 2   ? run(std::integral_constant<int, 2>{})
                        : nr == 4 ? run(std::integral_constant<int, 4>{})
                        : nr == 8 ? run(std::integral_constant<int, 8>{})
                                  : run(std::integral_constant<int, 16>{});
  if (!launched) {
    skv_set_error("%s: no event to order the reductions by", what);
    return SKV_ELAUNCH;
  }
  return skv_check_launch(what);
}
