// Depth-1 EWS scan of a block-diagonal generator made of uniform chains, any number of chains: Jordan chains
// (AParamJordanRepeated: real chains of 2-4 coordinates, complex chains of 2-4 complex coordinates), and, as chains of
// one coordinate, rotation planes and real diagonals. Forward and adjoint, float64 state per chain in registers,
// chunked in time with float64 carries between chunks.
//
// At depth 1 the EWS prefix row is the state S_t = M_t S_{t-1} + s_t (ews/core/chen_scan.py:125-152 at N = 1),
// and a block-diagonal A makes every chain an independent linear recurrence. A chain is J = c I + eps Nil with
// (Nil P)_i = P_{i+1}: a real chain of n coordinates (c = lambda), or a complex chain of k coordinates
// P_i = v_{2i} + i v_{2i+1} (c = a + ib, the 2x2 blocks [[a, -b], [b, a]] with the 2x2 identity above them). An
// analytic g gives g(J) = sum_p g^(p)(c) / p! (eps Nil)^p, so with x = -h c (jordan_engine.py:1-12, combine.py:143-190):
//   flow   exp(-h J) = e^x sum_p (-h eps)^p / p! Nil^p                         (exact at any step)
//   leaf   s_t = phi(-h J) v = sum_p (-h)^p u_p(x) (eps Nil)^p v,  u_p = phi^(p) / p!
// with phi(y) = (e^y - 1) / y (the exact integral: jordan_closed, plane_closed, block_series and van_loan's level 1),
// or, for the series leaf of order q (series_leaf.py:72-113 at level 1: sum_{p<=q} (-h)^p A^p v / (p+1)!),
// u_r = sum_{n=r..q} C(n, r) x^(n-r) / (n+1)!, the r-th derivative over r! of the degree-q Taylor polynomial of phi.
// u_r for the exact leaf: the entire series sum_j x^j / ((j + r + 1) j!) / r! below |x| = 2, else the recurrence
// phi^(r) = (e^x - r phi^(r-1)) / x from (e^x - 1) / x, in float64.
//
// Passes: chunk summaries from a zero state; a float64 carry scan over chunks per (sample, chain) (a workgroup each:
// runs of chunks composed in parallel, then chained), the chunk's flow taken in closed form over its clock span (the
// chain's flows commute); the rows from the carries. Adjoint: each chunk's own rows from a zero cotangent (its
// cotangent on the carry-in state), a float64 reverse scan over chunks (the same parallel scan), then each chunk
// from the cotangent at its end with the states by inverting its steps (or recomputed from its carry): the knot
// gradients and the chain-parameter partials (c, eps), summed in a fixed order (deterministic). Gradients of A land on the entries the chain is read
// from (A[f, f], A[f+1, f] and the coupling A[f, f+1] or A[f, f+2], f the chain's first row), as the reference's
// closed-form leaf and jordan_flows read them; a parametrisation of uniform chains gets its exact parameter gradient
// from them.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ews_hip.h"

namespace ews {
namespace chain {

struct zd {
  double re, im;
};
__device__ __forceinline__ zd Z(double r, double i = 0.0) { return zd{r, i}; }
__device__ __forceinline__ zd operator+(zd a, zd b) { return zd{a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ zd operator-(zd a, zd b) { return zd{a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ zd operator*(zd a, zd b) {
  return zd{fma(a.re, b.re, -a.im * b.im), fma(a.re, b.im, a.im * b.re)};
}
__device__ __forceinline__ zd operator*(double s, zd a) { return zd{s * a.re, s * a.im}; }
__device__ __forceinline__ zd& operator+=(zd& a, zd b) {
  a.re += b.re;
  a.im += b.im;
  return a;
}
__device__ __forceinline__ zd cj(zd a) { return zd{a.re, -a.im}; }
__device__ __forceinline__ zd cjm(zd a, zd b) {  // conj(a) b
  return zd{fma(a.re, b.re, a.im * b.im), fma(a.re, b.im, -a.im * b.re)};
}
__device__ __forceinline__ double redot(zd a, zd b) { return fma(a.re, b.re, a.im * b.im); }  // Re(conj(a) b)
__device__ __forceinline__ zd zdiv(zd a, zd b) {  // Smith's algorithm
  if (fabs(b.re) >= fabs(b.im)) {
    const double r = b.im / b.re, den = b.re + b.im * r;
    return zd{(a.re + a.im * r) / den, (a.im - a.re * r) / den};
  }
  const double r = b.re / b.im, den = b.im + b.re * r;
  return zd{(a.re * r + a.im) / den, (a.im * r - a.re) / den};
}
__device__ __forceinline__ zd zexp(zd a) {
  double s, c;
  sincos(a.im, &s, &c);
  const double m = exp(a.re);
  return zd{m * c, m * s};
}

// terms of the phi^(r) series by |x|: the tails are below 1e-20 (2^-9: x^7 / 7! = 2e-23; 1/8: 3e-22; 2: 1e-21)
constexpr int kTaylor0 = 7, kTaylor1 = 13, kTaylor = 28;
constexpr double kReach0 = 1.0 / 512, kReach1 = 0.125;
constexpr double kSwitch = 2.0;   // |x| above which the recurrence from e^x takes over
constexpr int kMaxT = 64;         // longest chunk
constexpr double kInvert = 8.0;   // largest log contraction of a chunk whose steps the adjoint inverts

struct CArgs {
  int B, L, n, d, K, size, cplx, M;  // M: coordinates per chain (complex for complex chains)
  int T, C, KP, CPW;                 // chunk length and count; lanes per chunk (power of 2 >= K); chunks per wave
  int flow_mode, leaf_mode, readout, lvl0, W, q;
  const float* path;
  const float* clock;
  const float* A;
  float* out;
  const float* gout;
  double* carries;  // (B, C+1, K, M) complex: the state before each chunk, and after the last
  double* summ;     // (B, C, K, M) complex: each chunk from a zero state
  double* mu;       // (B, C, K, M) complex: the chunk's own rows' cotangent on its carry-in state
  double* mt;       // (B, C, K, M) complex: the cotangent at the chunk's end from the later chunks
  float* dvb;       // (B, C, 2, d) increment cotangents of each chunk's first and last interval
  float* dhb;       // (B, C, 2) step cotangents of those (every chain's)
  float* st;        // (B, n, d) states before each step, of the chunks whose steps are not inverted
  double* pp;       // (B, C, K, 5): partials of Re c, Im c, eps, and of the reference steps theta1-theta0, theta2-theta1
  float* gpath;
  float* gclock;
  float* gA;
};

// the chain's eigenvalue and coupling, read from its first rows (jordan_engine.py:338-353)
__device__ __forceinline__ void chain_params(const CArgs& a, int j, zd& c, double& eps) {
  const int f = j * a.size;
  eps = 0.0;  // a chain of one coordinate (a diagonal entry, a rotation plane) has no coupling
  if (a.cplx) {
    c = Z((double)a.A[(size_t)f * a.d + f], (double)a.A[(size_t)(f + 1) * a.d + f]);
    if (a.M > 1) eps = (double)a.A[(size_t)f * a.d + f + 2];
  } else {
    c = Z((double)a.A[(size_t)f * a.d + f]);
    if (a.M > 1) eps = (double)a.A[(size_t)f * a.d + f + 1];
  }
}

// the clock step of interval t under a flow mode (chen_scan.py:155-168): its own, or the shared reference step
// theta1 - theta0 (cached) / theta2 - theta1 with interval 0 taking none (cached with basepoint)
__device__ __forceinline__ double mode_step(const float* th, int L, int t, double h_own, int mode) {
  if (mode == EWS_FLOW_PER_INTERVAL) return h_own;
  if (mode == EWS_FLOW_CACHED) return (double)th[1] - (double)th[0];
  if (t == 0 || L < 3) return 0.0;
  return (double)th[2] - (double)th[1];
}

// sum_{j < NT} x^j / ((j + r + 1) j! r!), r = 0..R, the constants at compile time
template <int R, int NT>
__device__ __forceinline__ void u_series(zd x, zd* u) {
  zd t = Z(1.0);  // x^j
  double jf = 1.0, rf[R + 1];
  rf[0] = 1.0;
#pragma unroll
  for (int r = 1; r <= R; ++r) rf[r] = rf[r - 1] * (double)r;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
#pragma unroll
    for (int r = 0; r <= R; ++r) {
      const double k = 1.0 / ((double)(j + r + 1) * jf * rf[r]);
      u[r].re = fma(k, t.re, u[r].re);
      u[r].im = fma(k, t.im, u[r].im);
    }
    t = t * x;
    jf *= (double)(j + 1);
  }
}

// u[r] = phi^(r)(x) / r!, r = 0..R: exact (q = 0) or of the degree-q Taylor polynomial of phi; ex = e^x for q = 0.
// The exact series takes as many terms as the wavefront's largest |x| needs: a gated clock's steps of 1/L lie far
// inside 2^-9, where 7 terms serve for 28.
template <int R>
__device__ __forceinline__ void u_table(zd x, int q, zd* u, zd& ex) {
  ex = Z(1.0);
#pragma unroll
  for (int r = 0; r <= R; ++r) u[r] = Z(0.0);
  if (q > 0) {
#pragma unroll
    for (int r = 0; r <= R; ++r) {
      if (r > q) continue;
      // sum_{m=0..q-r} a_m x^m, a_m = C(m+r, r) / (m+r+1)!, by Horner from the top coefficient
      double top = 1.0;  // C(q, r) / (q+1)!
      for (int i = 1; i <= q + 1; ++i) top /= (double)i;
      for (int i = 0; i < r; ++i) top = top * (double)(q - i) / (double)(i + 1);
      zd acc = Z(top);
      double am = top;
      for (int m = q - r - 1; m >= 0; --m) {
        am = am * (double)(m + 1) * (double)(m + r + 2) / (double)(m + r + 1);
        acc = acc * x + Z(am);
      }
      u[r] = acc;
    }
    return;
  }
  if (x.re * x.re + x.im * x.im <= kSwitch * kSwitch) {
    const double ax2 = x.re * x.re + x.im * x.im;
    if (!__any(ax2 > kReach0 * kReach0)) u_series<R, kTaylor0>(x, u);
    else if (!__any(ax2 > kReach1 * kReach1)) u_series<R, kTaylor1>(x, u);
    else u_series<R, kTaylor>(x, u);
    ex = Z(1.0) + x * u[0];
  } else {
    const zd e = zexp(x);
    ex = e;
    zd ph = zdiv(e - Z(1.0), x);
    u[0] = ph;
    double f = 1.0;
#pragma unroll
    for (int r = 1; r <= R; ++r) {
      ph = zdiv(e - (double)r * ph, x);
      f *= (double)r;
      u[r] = (1.0 / f) * ph;
    }
  }
}

// one interval's coefficients: leaf g[p] = (-hl)^p u_p(-hl c), flow e[p] = e^{-hf c} (-hf eps)^p / p!
template <int M>
struct Coef {
  zd g[M], e[M];
};
template <int M>
__device__ __forceinline__ void coefs(zd c, double eps, double hl, double hf, int q, Coef<M>& k) {
  zd u[M], ex;
  u_table<M - 1>(-hl * c, q, u, ex);
  double hp = 1.0;
#pragma unroll
  for (int p = 0; p < M; ++p) {
    k.g[p] = hp * u[p];
    hp *= -hl;
  }
  k.e[0] = q == 0 && hl == hf ? ex : zexp(-hf * c);  // one step for the leaf and the flow: e^x = 1 + x phi(x)
#pragma unroll
  for (int p = 1; p < M; ++p) k.e[p] = (-hf * eps / (double)p) * k.e[p - 1];
}
// the step S <- E S + s with s = sum_p g[p] (eps Nil)^p v
template <int M>
__device__ __forceinline__ void step(const Coef<M>& k, double eps, const zd* v, zd* S) {
  zd ew[M];  // eps^p
  ew[0] = Z(1.0);
#pragma unroll
  for (int p = 1; p < M; ++p) ew[p] = eps * ew[p - 1];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    zd acc = Z(0.0);
#pragma unroll
    for (int p = 0; p + i < M; ++p) acc += k.e[p] * S[i + p] + k.g[p] * (ew[p].re * v[i + p]);
    S[i] = acc;
  }
}
// the chunk's flow over a clock span tau: e^{-tau c} sum_p (-tau eps)^p / p! Nil^p
template <int M>
__device__ __forceinline__ void span_flow(zd c, double eps, double tau, zd* F) {
  F[0] = zexp(-tau * c);
#pragma unroll
  for (int p = 1; p < M; ++p) F[p] = (-tau * eps / (double)p) * F[p - 1];
}
// the flow over one interval's step: e^x from the series of phi while |x| is small (a sine, a cosine and an
// exponential in float64 otherwise)
template <int M>
__device__ __forceinline__ void flow_of(zd c, double eps, double h, zd* F) {
  const zd x = -h * c;
  if (x.re * x.re + x.im * x.im <= kReach1 * kReach1) {
    zd u[1], ex;
    u_table<0>(x, 0, u, ex);
    F[0] = ex;
  } else {
    F[0] = zexp(x);
  }
#pragma unroll
  for (int p = 1; p < M; ++p) F[p] = (-h * eps / (double)p) * F[p - 1];
}
// the flow span of chunk cc under the flow mode
__device__ __forceinline__ double chunk_span(const CArgs& a, const float* th, int cc) {
  const int t0 = cc * a.T, t1 = min(t0 + a.T, a.n);
  if (a.flow_mode == EWS_FLOW_PER_INTERVAL) return (double)th[t1] - (double)th[t0];
  const double hr = mode_step(th, a.L, 1, 0.0, a.flow_mode);
  const int nstep = (a.flow_mode == EWS_FLOW_CACHED_BASEPOINT && t0 == 0) ? t1 - 1 : t1 - t0;
  return hr * (double)nstep;
}

// knot row t of the chain's coordinates (complex coordinates of a complex chain)
template <int M, bool CPLX>
__device__ __forceinline__ void load_knot(const CArgs& a, int b, int t, int j, zd* x) {
  const float* r = a.path + ((size_t)b * a.L + t) * a.d + (size_t)j * a.size;
#pragma unroll
  for (int i = 0; i < M; ++i) x[i] = CPLX ? Z((double)r[2 * i], (double)r[2 * i + 1]) : Z((double)r[i]);
}

// A chain's coordinates of one row as loaded (floats, converted at their use), and stored.
template <int M, bool CPLX> struct Knot {
  float x[CPLX ? 2 * M : M];
  __device__ __forceinline__ void row(const float* r) {
#pragma unroll
    for (int i = 0; i < (CPLX ? 2 * M : M); ++i) x[i] = r[i];
  }
  __device__ __forceinline__ void load(const CArgs& a, int b, int t, int j) {
    row(a.path + ((size_t)b * a.L + t) * a.d + (size_t)j * a.size);
  }
  __device__ __forceinline__ void get(zd* z) const {
#pragma unroll
    for (int i = 0; i < M; ++i) z[i] = CPLX ? Z((double)x[2 * i], (double)x[2 * i + 1]) : Z((double)x[i]);
  }
};
template <int M, bool CPLX> __device__ __forceinline__ void st_row(float* r, const zd* z) {
#pragma unroll
  for (int i = 0; i < M; ++i) {
    if (CPLX) {
      r[2 * i] = (float)z[i].re;
      r[2 * i + 1] = (float)z[i].im;
    } else {
      r[i] = (float)z[i].re;
    }
  }
}

struct Lane {
  int b, j, c, t0, Tc;
  bool live, group;  // live: a real chain of an existing chunk; group: the lane's chunk exists
};
__device__ __forceinline__ Lane lane_of(const CArgs& a) {
  Lane l;
  const int lane = threadIdx.x;
  l.b = blockIdx.y;
  l.j = lane % a.KP;
  l.c = blockIdx.x * a.CPW + lane / a.KP;
  l.group = l.c < a.C;
  l.live = l.group && l.j < a.K;
  l.t0 = l.c * a.T;
  l.Tc = l.group ? min(a.T, a.n - l.t0) : 0;
  return l;
}
__device__ __forceinline__ size_t st_off(const CArgs& a, int b, int c, int j) {  // (B, C(+1), K, M) complex rows
  return (((size_t)b * (a.C + 1) + c) * a.K + j) * a.M * 2;
}
__device__ __forceinline__ size_t ch_off(const CArgs& a, int b, int c, int j) {  // (B, C, K, M)
  return (((size_t)b * a.C + c) * a.K + j) * a.M * 2;
}
template <int M>
__device__ __forceinline__ void ld_state(const double* p, zd* S) {
#pragma unroll
  for (int i = 0; i < M; ++i) S[i] = Z(p[2 * i], p[2 * i + 1]);
}
template <int M>
__device__ __forceinline__ void st_state(double* p, const zd* S) {
#pragma unroll
  for (int i = 0; i < M; ++i) {
    p[2 * i] = S[i].re;
    p[2 * i + 1] = S[i].im;
  }
}

// ------------------------------------------------------------------------------------------------ forward
// ROWS false: the chunk's summary from a zero state; true: the prefix rows from the chunk's carry
template <int M, bool CPLX, bool ROWS>
__device__ __forceinline__ void fwd_body(const CArgs& a) {
  const Lane l = lane_of(a);
  if (!l.live) return;
  zd c;
  double eps;
  chain_params(a, l.j, c, eps);
  zd S[M];
  if (ROWS) {
    ld_state<M>(a.carries + st_off(a, l.b, l.c, l.j), S);
  } else {
#pragma unroll
    for (int i = 0; i < M; ++i) S[i] = Z(0.0);
  }
  const float* th = a.clock + (size_t)l.b * a.L;
  // the knots and clock values run two intervals ahead of their use (the recursion waits on no load)
  zd x0[M], v[M];
  Knot<M, CPLX> x1, x2;
  load_knot<M, CPLX>(a, l.b, l.t0, l.j, x0);
  x1.load(a, l.b, l.t0 + 1, l.j);
  double th0 = (double)th[l.t0];
  float th1 = th[l.t0 + 1];
  Coef<M> k;
  const bool fixed = a.flow_mode != EWS_FLOW_PER_INTERVAL && a.leaf_mode != EWS_FLOW_PER_INTERVAL;
  if (fixed) coefs<M>(c, eps, mode_step(th, a.L, 1, 0.0, a.leaf_mode), mode_step(th, a.L, 1, 0.0, a.flow_mode), a.q, k);
  for (int s = 0; s < l.Tc; ++s) {
    const int t = l.t0 + s, tn = l.t0 + min(s + 2, l.Tc);
    x2.load(a, l.b, tn, l.j);
    const float th2 = th[tn];
    const double h = (double)th1 - th0;
    zd xc[M];
    x1.get(xc);
#pragma unroll
    for (int i = 0; i < M; ++i) v[i] = xc[i] - x0[i];
    if (!fixed || (t <= 1 && (a.flow_mode == EWS_FLOW_CACHED_BASEPOINT || a.leaf_mode == EWS_FLOW_CACHED_BASEPOINT)))
      coefs<M>(c, eps, mode_step(th, a.L, t, h, a.leaf_mode), mode_step(th, a.L, t, h, a.flow_mode), a.q, k);
    step<M>(k, eps, v, S);
    if (ROWS) {
      st_row<M, CPLX>(a.out + ((size_t)l.b * a.n + t) * a.W + a.lvl0 + (size_t)l.j * a.size, S);
      if (a.lvl0 && l.j == 0) a.out[((size_t)l.b * a.n + t) * a.W] = 1.0f;
    }
#pragma unroll
    for (int i = 0; i < M; ++i) x0[i] = xc[i];
    x1 = x2;
    th0 = (double)th1;
    th1 = th2;
  }
  if (!ROWS) st_state<M>(a.summ + ch_off(a, l.b, l.c, l.j), S);
}
template <int M, bool CPLX>
__global__ __launch_bounds__(64) void k_summary(CArgs a) {
  fwd_body<M, CPLX, false>(a);
}
template <int M, bool CPLX>
__global__ __launch_bounds__(64) void k_rows(CArgs a) {
  fwd_body<M, CPLX, true>(a);
}

// ---- carry scans over the chunks: a workgroup per (sample, chain), its 256 threads each owning a run of
// consecutive chunks. A chunk acts on the chain's state as S -> F S + z (F its flow over the chunk's clock span, a
// polynomial in Nil; z its summary) and, in the adjoint, on the cotangent as X -> F^H X + m with the chunks taken
// from the last. Each thread composes its run into one such map, thread 0 chains the 256 maps from the initial
// state in order (float64, fixed order), and each thread re-walks its run from its start state writing the carries
// (cotangents). The maps compose as (F2, z2) o (F1, z1) = (F2 F1, F2 z1 + z2) (adjoint: F2^H z1 + z2), the flows
// being polynomials in Nil that commute.
constexpr int kCarryThreads = 256;
constexpr int kGroup = 16;  // runs per group of the chaining

template <int M>
__device__ __forceinline__ void nil_apply(const zd* F, const zd* S, zd* o) {  // (F S)_i = sum_p F[p] S_{i+p}
#pragma unroll
  for (int i = 0; i < M; ++i) {
    zd acc = Z(0.0);
#pragma unroll
    for (int p = 0; p + i < M; ++p) acc += F[p] * S[i + p];
    o[i] = acc;
  }
}
template <int M>
__device__ __forceinline__ void nil_apply_h(const zd* F, const zd* X, zd* o) {  // (F^H X)_k = sum_p conj(F[p]) X_{k-p}
#pragma unroll
  for (int k = 0; k < M; ++k) {
    zd acc = Z(0.0);
#pragma unroll
    for (int p = 0; p <= k; ++p) acc += cjm(F[p], X[k - p]);
    o[k] = acc;
  }
}
template <int M>
__device__ __forceinline__ void nil_mul(const zd* F2, const zd* F1, zd* o) {  // product of polynomials in Nil
#pragma unroll
  for (int r = 0; r < M; ++r) {
    zd acc = Z(0.0);
#pragma unroll
    for (int p = 0; p <= r; ++p) acc += F2[p] * F1[r - p];
    o[r] = acc;
  }
}
// the map of chunk cc (application order: ascending chunks forward, descending in the adjoint)
template <int M, bool BWD>
__device__ __forceinline__ void chunk_map(const CArgs& a, int b, int j, zd c, double eps, const float* th, int cc,
                                          zd* F, zd* z) {
  span_flow<M>(c, eps, chunk_span(a, th, cc), F);
  if (!BWD) {
    ld_state<M>(a.summ + ch_off(a, b, cc, j), z);
  } else if (a.readout != EWS_READOUT_TERMINAL) {
    ld_state<M>(a.mu + ch_off(a, b, cc, j), z);
  } else {
#pragma unroll
    for (int i = 0; i < M; ++i) z[i] = Z(0.0);
  }
}
template <int M, bool BWD>
__device__ __forceinline__ void map_apply(const zd* F, const zd* z, zd* S) {
  zd o[M];
  if (BWD) nil_apply_h<M>(F, S, o);
  else nil_apply<M>(F, S, o);
#pragma unroll
  for (int i = 0; i < M; ++i) S[i] = o[i] + z[i];
}
template <int M, bool CPLX, bool BWD>
__device__ __forceinline__ void carry_scan(const CArgs& a) {
  __shared__ double s_map[kCarryThreads][4 * M];  // each thread's composed map: F, then z (complex)
  __shared__ double s_in[kCarryThreads][2 * M];   // each thread's start state
  __shared__ double s_grp[kCarryThreads / kGroup][4 * M];
  const int b = blockIdx.x / a.K, j = blockIdx.x % a.K, tid = threadIdx.x;
  zd c;
  double eps;
  chain_params(a, j, c, eps);
  const float* th = a.clock + (size_t)b * a.L;
  const int nth = blockDim.x, per = (a.C + nth - 1) / nth, nrun = (a.C + per - 1) / per;
  const int q0 = tid * per, q1 = min(a.C, q0 + per);  // the thread's run, in application order
  zd AF[M], Az[M], F[M], z[M], t[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    AF[i] = Z(i == 0 ? 1.0 : 0.0);
    Az[i] = Z(0.0);
  }
  for (int q = q0; q < q1; ++q) {
    const int cc = BWD ? a.C - 1 - q : q;
    chunk_map<M, BWD>(a, b, j, c, eps, th, cc, F, z);
    nil_mul<M>(F, AF, t);  // the chunk after the run so far
#pragma unroll
    for (int i = 0; i < M; ++i) AF[i] = t[i];
    map_apply<M, BWD>(F, z, Az);
  }
  st_state<M>(&s_map[tid][0], AF);
  st_state<M>(&s_map[tid][2 * M], Az);
  __syncthreads();
  // the threads' maps chained from the initial state in two levels (a single chain over up to 256 maps was a quarter
  // of the scan's time): kGroup runs composed per group, the groups' maps chained, the runs of a group from its state
  const int ng = (nrun + kGroup - 1) / kGroup;
  if (tid < ng) {
#pragma unroll
    for (int i = 0; i < M; ++i) {
      AF[i] = Z(i == 0 ? 1.0 : 0.0);
      Az[i] = Z(0.0);
    }
    for (int u = tid * kGroup; u < min(nrun, (tid + 1) * kGroup); ++u) {
      ld_state<M>(&s_map[u][0], F);
      ld_state<M>(&s_map[u][2 * M], z);
      nil_mul<M>(F, AF, t);
#pragma unroll
      for (int i = 0; i < M; ++i) AF[i] = t[i];
      map_apply<M, BWD>(F, z, Az);
    }
    st_state<M>(&s_grp[tid][0], AF);
    st_state<M>(&s_grp[tid][2 * M], Az);
  }
  __syncthreads();
  if (tid == 0) {
    zd S[M];
    if (BWD && a.readout == EWS_READOUT_TERMINAL) {
      const float* r = a.gout + (size_t)b * a.W + a.lvl0 + (size_t)j * a.size;
#pragma unroll
      for (int i = 0; i < M; ++i) S[i] = CPLX ? Z((double)r[2 * i], (double)r[2 * i + 1]) : Z((double)r[i]);
    } else {
#pragma unroll
      for (int i = 0; i < M; ++i) S[i] = Z(0.0);
    }
    for (int u = 0; u < ng; ++u) {
      st_state<M>(&s_in[u * kGroup][0], S);  // the state before the group's first run
      ld_state<M>(&s_grp[u][0], F);
      ld_state<M>(&s_grp[u][2 * M], z);
      map_apply<M, BWD>(F, z, S);
    }
  }
  __syncthreads();
  if (tid < ng) {
    zd S[M];
    ld_state<M>(&s_in[tid * kGroup][0], S);
    for (int u = tid * kGroup; u < min(nrun, (tid + 1) * kGroup); ++u) {  // the threads past nrun own no chunk
      st_state<M>(&s_in[u][0], S);
      ld_state<M>(&s_map[u][0], F);
      ld_state<M>(&s_map[u][2 * M], z);
      map_apply<M, BWD>(F, z, S);
    }
  }
  __syncthreads();
  if (tid >= nrun) return;
  zd S[M];
  ld_state<M>(&s_in[tid][0], S);
  for (int q = q0; q < q1; ++q) {
    const int cc = BWD ? a.C - 1 - q : q;
    if (BWD) st_state<M>(a.mt + ch_off(a, b, cc, j), S);  // the cotangent at the chunk's end
    else st_state<M>(a.carries + st_off(a, b, cc, j), S);  // the state before the chunk
    chunk_map<M, BWD>(a, b, j, c, eps, th, cc, F, z);
    map_apply<M, BWD>(F, z, S);
    if (!BWD && cc == a.C - 1) st_state<M>(a.carries + st_off(a, b, a.C, j), S);
  }
}
template <int M, bool CPLX>
__global__ __launch_bounds__(kCarryThreads) void k_carry(CArgs a) {
  carry_scan<M, CPLX, false>(a);
}

// the terminal row: the state after the last chunk
template <int M, bool CPLX>
__global__ void k_terminal(CArgs a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.B * a.W) return;
  const int b = e / a.W, col = e % a.W;
  if (a.lvl0 && col == 0) {
    a.out[e] = 1.0f;
    return;
  }
  const int r = col - a.lvl0, j = r / a.size, w = r % a.size;
  const double* s = a.carries + st_off(a, b, a.C, j);
  a.out[e] = (float)(CPLX ? s[w] : s[2 * w]);  // complex coordinate i at (2i, 2i+1) = (re, im); real: re
}

// ------------------------------------------------------------------------------------------------ adjoint
// Lam <- E^H Lam
template <int M>
__device__ __forceinline__ void adj_flow(const zd* e, zd* Lam) {
  zd o[M];
#pragma unroll
  for (int i = 0; i < M; ++i) o[i] = Z(0.0);
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int p = 0; p + i < M; ++p) o[i + p] += cjm(e[p], Lam[i]);
#pragma unroll
  for (int i = 0; i < M; ++i) Lam[i] = o[i];
}

// the chunk's own rows from a zero cotangent at its end: the cotangent on its carry-in state
template <int M, bool CPLX>
__global__ __launch_bounds__(64) void k_local(CArgs a) {
  const Lane l = lane_of(a);
  if (!l.live) return;
  zd c;
  double eps;
  chain_params(a, l.j, c, eps);
  const float* th = a.clock + (size_t)l.b * a.L;
  zd Lam[M], g[M], e[M];
#pragma unroll
  for (int i = 0; i < M; ++i) Lam[i] = Z(0.0);
  // row cotangents and clock values two intervals ahead of their use
  Knot<M, CPLX> g0, g1, g2;
  const float* gr = a.gout + (size_t)l.b * a.n * a.W + a.lvl0 + (size_t)l.j * a.size;
  const int tl = l.t0 + l.Tc - 1;
  g0.row(gr + (size_t)tl * a.W);
  g1.row(gr + (size_t)max(tl - 1, l.t0) * a.W);
  float thu = th[tl + 1], th0 = th[tl], th1 = th[max(tl - 1, l.t0)];
  for (int s = l.Tc - 1; s >= 0; --s) {
    const int t = l.t0 + s, tp = max(t - 2, l.t0);
    g2.row(gr + (size_t)tp * a.W);
    const float th2 = th[tp];
    g0.get(g);
#pragma unroll
    for (int i = 0; i < M; ++i) Lam[i] += g[i];
    const double hf = mode_step(th, a.L, t, (double)thu - (double)th0, a.flow_mode);
    flow_of<M>(c, eps, hf, e);
    adj_flow<M>(e, Lam);
    g0 = g1;
    g1 = g2;
    thu = th0;
    th0 = th1;
    th1 = th2;
  }
  st_state<M>(a.mu + ch_off(a, l.b, l.c, l.j), Lam);
}

// the reverse carry scan: mt[c] = the cotangent at chunk c's end from the later chunks (the terminal row's at the
// last chunk); mt[c-1] = F_c^H mt[c] + mu[c]
template <int M, bool CPLX>
__global__ __launch_bounds__(kCarryThreads) void k_carry_bwd(CArgs a) {
  carry_scan<M, CPLX, true>(a);
}

// Each chunk from the cotangent at its end: the steps in reverse with the increment and step cotangents and the
// chain-parameter partials. The states S_{t-1} come from inverting each step from the chunk's end state in float64
// while the whole chunk contracts by less than e^kInvert (errors then stay below 1e-12, where states kept in float32
// had 6e-8); a wavefront with a stronger contraction, or an end state that is not finite, first recomputes its states from
// the carry into st. The sweep keeps the interval after in registers, so a chunk's interior knot gradients
// dX_{t+1} = dv_t - dv_{t+1} (and the clock's) are written here; the cotangents of its first and last interval go to dvb /
// dhb for the boundary knots (k_bounds). Bound by float64 issue: at B = 8, L = 49,920, 16 complex chains of two
// coordinates, 543 us with the 28-term series at every step, the states recomputed into LDS (one wavefront per SIMD) and
// dv, dh through memory; 171 us now (the step 1.12 -> 0.60 ms).
template <int M, bool CPLX>
__global__ __launch_bounds__(64) void k_full(CArgs a) {
  constexpr int NX = CPLX ? 2 * M : M;
  const Lane l = lane_of(a);
  if (!l.group) return;  // the lanes of one chunk stay together: the dh sums exchange across them
  const bool live = l.live;
  zd c = Z(0.0);
  double eps = 0.0;
  if (live) chain_params(a, l.j, c, eps);
  const float* th = a.clock + (size_t)l.b * a.L;
  const int tl = l.t0 + l.Tc - 1;
  // the chunk's total flow step, a lane per step
  double tot = 0.0;
  for (int s = l.j; s < l.Tc; s += a.KP) {
    const int t = l.t0 + s;
    tot += fabs(mode_step(th, a.L, t, (double)th[t + 1] - (double)th[t], a.flow_mode));
  }
  for (int o = 1; o < a.KP; o <<= 1) tot += __shfl_xor(tot, o, 64);
  zd S[M], v[M], xc[M], xn[M];
  double end = 0.0;  // finite if the chunk's end state is: padding with NaN must not reach the rows before it
  if (live) {
    ld_state<M>(a.carries + st_off(a, l.b, l.c + 1, l.j), S);
#pragma unroll
    for (int i = 0; i < M; ++i) end += fabs(S[i].re) + fabs(S[i].im);
  }
  const bool invert = !__any(live && !((fabs(c.re) + fabs(eps)) * tot <= kInvert && isfinite(end)));
  Knot<M, CPLX> x1, x2;
  float* my = a.st + ((size_t)l.b * a.n + l.t0) * a.d + (size_t)l.j * NX;  // the states of the lane's steps
  if (!invert && live) {
    Coef<M> k;
    zd x0[M];
    ld_state<M>(a.carries + st_off(a, l.b, l.c, l.j), S);
    load_knot<M, CPLX>(a, l.b, l.t0, l.j, x0);
    x1.load(a, l.b, l.t0 + 1, l.j);
    double th0 = (double)th[l.t0];
    float th1 = th[l.t0 + 1];
    for (int s = 0; s < l.Tc; ++s) {
      const int t = l.t0 + s, tn = l.t0 + min(s + 2, l.Tc);
      st_row<M, CPLX>(my + (size_t)s * a.d, S);
      if (s == l.Tc - 1) break;
      x2.load(a, l.b, tn, l.j);
      const float th2 = th[tn];
      x1.get(xc);
      const double h = (double)th1 - th0;
#pragma unroll
      for (int i = 0; i < M; ++i) v[i] = xc[i] - x0[i];
      coefs<M>(c, eps, mode_step(th, a.L, t, h, a.leaf_mode), mode_step(th, a.L, t, h, a.flow_mode), a.q, k);
      step<M>(k, eps, v, S);
#pragma unroll
      for (int i = 0; i < M; ++i) x0[i] = xc[i];
      x1 = x2;
      th0 = (double)th1;
      th1 = th2;
    }
  }
  // 2. the steps in reverse from the cotangent at the chunk's end; knots, row cotangents and clock values two intervals
  // ahead of their use
  const bool rows = a.readout != EWS_READOUT_TERMINAL, own_step = a.leaf_mode == a.flow_mode && a.q == 0;
  zd Lam[M], g[M], Gc = Z(0.0);
  double deps = 0.0, dref0 = 0.0, dref1 = 0.0;
  float dvn[NX], dhn = 0.0f;  // of the interval after
  Knot<M, CPLX> g0{}, g1{}, g2{};
  const float* gr = a.gout + (size_t)l.b * a.n * a.W + a.lvl0 + (size_t)l.j * a.size;
  float thu = th[tl + 1], th0 = th[tl], th1 = th[max(tl - 1, l.t0)];
  if (live) {
    ld_state<M>(a.mt + ch_off(a, l.b, l.c, l.j), Lam);
    load_knot<M, CPLX>(a, l.b, tl + 1, l.j, xn);
    x1.load(a, l.b, tl, l.j);
    x2.load(a, l.b, max(tl - 1, l.t0), l.j);
    if (rows) {
      g0.row(gr + (size_t)tl * a.W);
      g1.row(gr + (size_t)max(tl - 1, l.t0) * a.W);
    }
  }
  for (int s = l.Tc - 1; s >= 0; --s) {
    const int t = l.t0 + s, tp = max(t - 2, l.t0);
    double dh_own = 0.0;
    const float th2 = th[tp];
    if (live) {
      Knot<M, CPLX> x3;
      x3.load(a, l.b, tp, l.j);
      if (rows) {
        g2.row(gr + (size_t)tp * a.W);
        g0.get(g);
#pragma unroll
        for (int i = 0; i < M; ++i) Lam[i] += g[i];
        g0 = g1;
        g1 = g2;
      }
      x1.get(xc);
#pragma unroll
      for (int i = 0; i < M; ++i) {
        v[i] = xn[i] - xc[i];
        xn[i] = xc[i];
      }
      x1 = x2;
      x2 = x3;
      const double h = (double)thu - (double)th0;
      const double hl = mode_step(th, a.L, t, h, a.leaf_mode), hf = mode_step(th, a.L, t, h, a.flow_mode);
      zd u[M + 1], ex;
      u_table<M>(-hl * c, a.q, u, ex);
      zd ew[M];  // eps^p, as reals
      ew[0] = Z(1.0);
#pragma unroll
      for (int p = 1; p < M; ++p) ew[p] = eps * ew[p - 1];
      // leaf: s_i = sum_p z_p eps^p v_{i+p}, z_p = (-hl)^p u_p(-hl c)
      zd dv[M], Es[M];  // Es: E S_{t-1} = S_t - s_t
#pragma unroll
      for (int i = 0; i < M; ++i) {
        dv[i] = Z(0.0);
        Es[i] = S[i];
      }
      double hp = 1.0, hq = 0.0, dhl = 0.0;  // (-hl)^p, (-hl)^(p-1)
#pragma unroll
      for (int p = 0; p < M; ++p) {
        const zd zp = hp * u[p];
        zd Gz = Z(0.0);  // cotangent of z_p
#pragma unroll
        for (int i = 0; i + p < M; ++i) {
          Gz += cjm(ew[p].re * v[i + p], Lam[i]);
          dv[i + p] += (ew[p].re) * cjm(zp, Lam[i]);
          Es[i] = Es[i] - zp * (ew[p].re * v[i + p]);
          if (p > 0) deps += (double)p * ew[p - 1].re * redot(Lam[i], zp * v[i + p]);
        }
        // dz_p / dc = -hl (p+1) (-hl)^p u_{p+1}; dz_p / dhl = -p (-hl)^(p-1) u_p - c (p+1) (-hl)^p u_{p+1}
        const zd dzc = (-hl * (double)(p + 1) * hp) * u[p + 1];
        Gc += cjm(dzc, Gz);
        const zd dzh = (-(double)p * hq) * u[p] - ((double)(p + 1) * hp) * (c * u[p + 1]);
        dhl += redot(Gz, dzh);
        hq = hp;
        hp *= -hl;
      }
      // flow: (E S)_i = sum_p e_p S_{i+p}, e_p = e^{-hf c} (-hf eps)^p / p!
      zd Sp[M], e[M];
      e[0] = own_step ? ex : zexp(-hf * c);
#pragma unroll
      for (int p = 1; p < M; ++p) e[p] = (-hf * eps / (double)p) * e[p - 1];
      const zd ef = e[0];
      if (invert) {  // back substitution from the last coordinate
        const double nrm = 1.0 / fma(ef.re, ef.re, ef.im * ef.im);
        const zd ei = Z(nrm * ef.re, -nrm * ef.im);
#pragma unroll
        for (int i = M - 1; i >= 0; --i) {
          zd r = Es[i];
#pragma unroll
          for (int p = 1; p + i < M; ++p) r = r - e[p] * Sp[i + p];
          Sp[i] = ei * r;
        }
      } else {
        Knot<M, CPLX> w;
        w.row(my + (size_t)s * a.d);
        w.get(Sp);
      }
#pragma unroll
      for (int i = 0; i < M; ++i) S[i] = Sp[i];
      double dhf = 0.0;
      double xp = 1.0, fp = 1.0;  // (-hf eps)^(p-1), (p-1)!
#pragma unroll
      for (int p = 0; p < M; ++p) {
        zd Ge = Z(0.0);
#pragma unroll
        for (int i = 0; i + p < M; ++i) Ge += cjm(Sp[i + p], Lam[i]);
        Gc += cjm((-hf) * e[p], Ge);
        zd deh = Z(0.0) - c * e[p];
        if (p > 0) {
          deh += (-eps * xp / fp) * ef;
          deps += redot(Ge, (-hf * xp / fp) * ef);
          xp *= -hf * eps;
          fp *= (double)p;
        }
        dhf += redot(Ge, deh);
      }
      adj_flow<M>(e, Lam);
      // increment cotangent of the interval: the knot after it, or the chunk's boundary rows
      float dvf[NX];
      st_row<M, CPLX>(dvf, dv);
      const size_t col = (size_t)l.j * a.size;
      float* bnd = a.dvb + ((size_t)l.b * a.C + l.c) * 2 * a.d + col;
      if (s < l.Tc - 1) {
        float* o = a.gpath + ((size_t)l.b * a.L + t + 1) * a.d + col;
#pragma unroll
        for (int i = 0; i < NX; ++i) o[i] = dvf[i] - dvn[i];
      } else {
#pragma unroll
        for (int i = 0; i < NX; ++i) bnd[a.d + i] = dvf[i];
      }
      if (s == 0) {
#pragma unroll
        for (int i = 0; i < NX; ++i) bnd[i] = dvf[i];
      }
#pragma unroll
      for (int i = 0; i < NX; ++i) dvn[i] = dvf[i];
      // steps: the interval's own, or the shared reference steps (theta1 - theta0: cached; theta2 - theta1:
      // cached with basepoint, interval 0 none)
      if (a.leaf_mode == EWS_FLOW_PER_INTERVAL) dh_own += dhl;
      else if (a.leaf_mode == EWS_FLOW_CACHED) dref0 += dhl;
      else if (t > 0) dref1 += dhl;
      if (a.flow_mode == EWS_FLOW_PER_INTERVAL) dh_own += dhf;
      else if (a.flow_mode == EWS_FLOW_CACHED) dref0 += dhf;
      else if (t > 0) dref1 += dhf;
    }
    thu = th0;
    th0 = th1;
    th1 = th2;
    if (!a.gclock) continue;
    // dh of the interval: every chain of the sample, summed across the chunk's lane group
    double acc = dh_own;
    for (int o = 1; o < a.KP; o <<= 1) acc += __shfl_xor(acc, o, 64);
    if (l.j == 0) {
      const float dhf = (float)acc;
      float* bnd = a.dhb + ((size_t)l.b * a.C + l.c) * 2;
      if (s < l.Tc - 1) a.gclock[(size_t)l.b * a.L + t + 1] = dhf - dhn;
      else bnd[1] = dhf;
      if (s == 0) bnd[0] = dhf;
      dhn = dhf;
    }
  }
  if (live) {
    double* pp = a.pp + (((size_t)l.b * a.C + l.c) * a.K + l.j) * 5;
    pp[0] = Gc.re;
    pp[1] = Gc.im;
    pp[2] = deps;
    pp[3] = dref0;
    pp[4] = dref1;
  }
}

// The knots between chunks, and the first and last: dX = dv of the chunk before's last interval - dv of this chunk's
// first; the clock's likewise, plus the reference steps' shares (summed over the sample's chunks and chains in order)
// on knots 0 to 2. A thread per (sample, chunk or the last knot, column; column d the clock).
__global__ void k_bounds(CArgs a) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t per = (size_t)(a.C + 1) * (a.d + 1);
  if (e >= (size_t)a.B * per) return;
  const size_t b = e / per, r = e % per, c = r / (a.d + 1), ch = r % (a.d + 1);
  const size_t t = c < (size_t)a.C ? c * a.T : (size_t)a.n;
  const size_t row = b * a.C + c;  // this chunk's boundary rows
  if (ch < (size_t)a.d) {
    const float lo = c > 0 ? a.dvb[((row - 1) * 2 + 1) * a.d + ch] : 0.0f;
    const float hi = c < (size_t)a.C ? a.dvb[row * 2 * a.d + ch] : 0.0f;
    a.gpath[(b * a.L + t) * a.d + ch] = lo - hi;
    return;
  }
  if (!a.gclock) return;
  double g = (c > 0 ? (double)a.dhb[(row - 1) * 2 + 1] : 0.0) - (c < (size_t)a.C ? (double)a.dhb[row * 2] : 0.0);
  const bool shared = a.flow_mode != EWS_FLOW_PER_INTERVAL || a.leaf_mode != EWS_FLOW_PER_INTERVAL;
  if (shared && t <= 2) {
    double r0 = 0.0, r1 = 0.0;
    for (size_t i = 0; i < (size_t)a.C * a.K; ++i) {
      r0 += a.pp[(b * a.C * a.K + i) * 5 + 3];
      r1 += a.pp[(b * a.C * a.K + i) * 5 + 4];
    }
    g += t == 0 ? -r0 : t == 1 ? r0 - r1 : r1;
    if (t == 0)  // knots 1 and 2 where they lie inside chunk 0 (its adjoint wrote them)
      for (int k = 1; k <= 2; ++k)
        if (k < a.n && k % a.T != 0) a.gclock[b * a.L + k] += (float)(k == 1 ? r0 - r1 : r1);
  }
  a.gclock[b * a.L + t] = (float)g;
}

// grad_A: zero, then each chain's entries from the partials (one workgroup per chain and component, float64 sums in
// a fixed order)
__global__ void k_zero_a(CArgs a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < a.d * a.d) a.gA[e] = 0.0f;
}
constexpr int kParamThreads = 1024;
__global__ __launch_bounds__(kParamThreads) void k_params(CArgs a) {
  __shared__ double red[kParamThreads];
  const int j = blockIdx.x / 3, comp = blockIdx.x % 3, tid = threadIdx.x;
  if ((!a.cplx && comp == 1) || (comp == 2 && a.M == 1)) return;  // uniform across the workgroup
  const size_t tot = (size_t)a.B * a.C;
  double acc = 0.0;
  for (size_t it = tid; it < tot; it += 4 * kParamThreads) {  // four loads in flight
    double x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const size_t i = it + (size_t)u * kParamThreads;
      x[u] = i < tot ? a.pp[(i * a.K + j) * 5 + comp] : 0.0;
    }
    acc += (x[0] + x[1]) + (x[2] + x[3]);
  }
  red[tid] = acc;
  __syncthreads();
  for (int o = kParamThreads / 2; o > 0; o >>= 1) {
    if (tid < o) red[tid] += red[tid + o];
    __syncthreads();
  }
  if (tid == 0) {
    const int f = j * a.size;
    size_t idx;
    if (comp == 0) idx = (size_t)f * a.d + f;
    else if (comp == 1) idx = (size_t)(f + 1) * a.d + f;
    else idx = a.cplx ? (size_t)f * a.d + f + 2 : (size_t)f * a.d + f + 1;
    a.gA[idx] = (float)red[0];
  }
}

// ------------------------------------------------------------------------------------------------ token cache
// The cached scan's per-token terms at depth 1 (ews/core/token_scan.py:44-88): P (V, d) the level 1 of a token's segment
// (increment dx_g, step dtheta_g), D (V, d, d) its flow exp(-dtheta_g A), zero outside the chains' blocks. Both are the
// coefficients of one interval, so one thread per (token, chain) forms them, and their adjoint, directly: on the scan
// kernels the cache was V one-interval samples and V d basis injections through every pass of both directions, and some
// forty torch operations around them (V = 8, d = 64: 0.17 ms of kernels, 0.4 ms of a training step's host time).
struct KArgs {
  int V, d, K, size, q;
  const float *dx, *dth, *gP, *gD;
  float *P, *D, *gdx, *gdth, *gA;
  double* pp;  // (V, K, 4): partials of Re c, Im c, eps and the token's step
};
__device__ __forceinline__ CArgs chain_view(const KArgs& a, const float* A, int M, bool cplx) {
  CArgs c{};
  c.d = a.d;
  c.size = a.size;
  c.M = M;
  c.cplx = cplx;
  c.A = A;
  return c;
}
template <int M, bool CPLX>
__global__ __launch_bounds__(256) void k_cache(KArgs a, const float* A) {
  const int g = blockIdx.x, tid = threadIdx.x;
  float* D = a.D + (size_t)g * a.d * a.d;
  for (int e = tid; e < a.d * a.d; e += 256)
    if (e / a.d / a.size != e % a.d / a.size) D[e] = 0.0f;
  if (tid >= a.K) return;
  const int f = tid * a.size;
  zd c;
  double eps;
  chain_params(chain_view(a, A, M, CPLX), tid, c, eps);
  const double h = (double)a.dth[g];
  Coef<M> k;
  coefs<M>(c, eps, h, h, a.q, k);
  zd v[M], S[M];
  Knot<M, CPLX> x;
  x.row(a.dx + (size_t)g * a.d + f);
  x.get(v);
#pragma unroll
  for (int i = 0; i < M; ++i) S[i] = Z(0.0);
  step<M>(k, eps, v, S);
  st_row<M, CPLX>(a.P + (size_t)g * a.d + f, S);
  // (E S)_i = sum_p e_p S_{i+p}: a complex coordinate is the 2 x 2 block [[re, -im], [im, re]]
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const zd e = m >= i ? k.e[m >= i ? m - i : 0] : Z(0.0);
      if (CPLX) {
        float* r = D + (size_t)(f + 2 * i) * a.d + f + 2 * m;
        r[0] = (float)e.re;
        r[1] = -(float)e.im;
        r[a.d] = (float)e.im;
        r[a.d + 1] = (float)e.re;
      } else {
        D[(size_t)(f + i) * a.d + f + m] = (float)e.re;
      }
    }
}
// a thread per (token, chain): dx's cotangent and the partials of the chain's parameters and the token's step
template <int M, bool CPLX>
__global__ __launch_bounds__(64) void k_cache_bwd(KArgs a, const float* A) {
  const int e0 = blockIdx.x * 64 + threadIdx.x;
  if (e0 >= a.V * a.K) return;
  const int g = e0 / a.K, j = e0 % a.K, f = j * a.size;
  zd c;
  double eps;
  chain_params(chain_view(a, A, M, CPLX), j, c, eps);
  const double h = (double)a.dth[g];
  zd v[M], Lam[M], u[M + 1], ex;
  Knot<M, CPLX> x;
  x.row(a.dx + (size_t)g * a.d + f);
  x.get(v);
  x.row(a.gP + (size_t)g * a.d + f);
  x.get(Lam);
  u_table<M>(-h * c, a.q, u, ex);
  double ew[M];
  ew[0] = 1.0;
#pragma unroll
  for (int p = 1; p < M; ++p) ew[p] = eps * ew[p - 1];
  zd dv[M], Gc = Z(0.0);
  double deps = 0.0, dh = 0.0, hp = 1.0, hq = 0.0;
#pragma unroll
  for (int i = 0; i < M; ++i) dv[i] = Z(0.0);
#pragma unroll
  for (int p = 0; p < M; ++p) {  // the leaf, as in the scan's adjoint
    const zd zp = hp * u[p];
    zd Gz = Z(0.0);
#pragma unroll
    for (int i = 0; i + p < M; ++i) {
      Gz += cjm(ew[p] * v[i + p], Lam[i]);
      dv[i + p] += ew[p] * cjm(zp, Lam[i]);
      if (p > 0) deps += (double)p * ew[p - 1] * redot(Lam[i], zp * v[i + p]);
    }
    Gc += cjm((-h * (double)(p + 1) * hp) * u[p + 1], Gz);
    dh += redot(Gz, (-(double)p * hq) * u[p] - ((double)(p + 1) * hp) * (c * u[p + 1]));
    hq = hp;
    hp *= -h;
  }
  st_row<M, CPLX>(a.gdx + (size_t)g * a.d + f, dv);
  // the flow: its coefficients' cotangents are sums over the block's diagonals
  const float* D = a.gD + (size_t)g * a.d * a.d;
  zd e[M];
  e[0] = a.q == 0 ? ex : zexp(-h * c);
#pragma unroll
  for (int p = 1; p < M; ++p) e[p] = (-h * eps / (double)p) * e[p - 1];
  double xp = 1.0, fp = 1.0;
#pragma unroll
  for (int p = 0; p < M; ++p) {
    zd Ge = Z(0.0);
#pragma unroll
    for (int i = 0; i + p < M; ++i) {
      if (CPLX) {
        const float* r = D + (size_t)(f + 2 * i) * a.d + f + 2 * (i + p);
        Ge += Z((double)r[0] + (double)r[a.d + 1], (double)r[a.d] - (double)r[1]);
      } else {
        Ge += Z((double)D[(size_t)(f + i) * a.d + f + i + p]);
      }
    }
    Gc += cjm(-h * e[p], Ge);
    zd deh = Z(0.0) - c * e[p];
    if (p > 0) {
      deh += (-eps * xp / fp) * e[0];
      deps += redot(Ge, (-h * xp / fp) * e[0]);
      xp *= -h * eps;
      fp *= (double)p;
    }
    dh += redot(Ge, deh);
  }
  double* pp = a.pp + (size_t)e0 * 4;
  pp[0] = Gc.re;
  pp[1] = Gc.im;
  pp[2] = deps;
  pp[3] = dh;
}
// the sums in order: a chain's parameters over the tokens, a token's step over the chains; grad_A's other entries zero
__global__ __launch_bounds__(1024) void k_cache_sums(KArgs a, int M, int cplx) {
  const int tid = threadIdx.x;
  if (blockIdx.x > 0) {  // the tokens' steps
    const int g = (blockIdx.x - 1) * 1024 + tid;
    if (g >= a.V) return;
    double s = 0.0;
    for (int j = 0; j < a.K; ++j) s += a.pp[((size_t)g * a.K + j) * 4 + 3];
    a.gdth[g] = (float)s;
    return;
  }
  for (int e = tid; e < a.d * a.d; e += 1024) a.gA[e] = 0.0f;
  __syncthreads();
  const int j = tid / 3, comp = tid % 3;
  if (j >= a.K || (comp == 1 && !cplx) || (comp == 2 && M == 1)) return;
  double s = 0.0;
  for (int g = 0; g < a.V; ++g) s += a.pp[((size_t)g * a.K + j) * 4 + comp];
  const int f = j * a.size;
  const int r = comp == 1 ? f + 1 : f, col = comp < 2 ? f : (cplx ? f + 2 : f + 1);
  a.gA[(size_t)r * a.d + col] = (float)s;
}

}  // namespace chain

namespace {

using chain::CArgs;

int chain_check(const ews_chain_desc* s) {
  if (!s) return EWS_ERR_NULL;
  if (s->batch < 1 || s->length < 2 || s->dim < 1) return EWS_ERR_SHAPE;
  if (s->kind == EWS_JORDAN_REAL) {
    if (s->size < 1 || s->size > 4) return EWS_ERR_OPTION;
  } else if (s->kind == EWS_JORDAN_COMPLEX) {
    if (s->size != 2 && s->size != 4 && s->size != 6 && s->size != 8) return EWS_ERR_OPTION;
  } else {
    return EWS_ERR_OPTION;
  }
  if (s->dim % s->size || s->dim / s->size > 64) return EWS_ERR_SHAPE;
  for (int m : {s->flow_mode, s->leaf_mode})
    if (m != EWS_FLOW_PER_INTERVAL && m != EWS_FLOW_CACHED && m != EWS_FLOW_CACHED_BASEPOINT) return EWS_ERR_OPTION;
  if (s->readout != EWS_READOUT_PREFIX && s->readout != EWS_READOUT_TERMINAL) return EWS_ERR_OPTION;
  if (s->series_q < 0 || s->series_q > 48) return EWS_ERR_OPTION;
  if (s->chunk < 0 || s->chunk > chain::kMaxT) return EWS_ERR_SHAPE;
  return EWS_OK;
}

CArgs chain_args(const ews_chain_desc* s) {
  CArgs a{};
  a.B = s->batch;
  a.L = s->length;
  a.n = s->length - 1;
  a.d = s->dim;
  a.size = s->size;
  a.cplx = s->kind == EWS_JORDAN_COMPLEX;
  a.M = a.cplx ? s->size / 2 : s->size;
  a.K = s->dim / s->size;
  a.KP = 1;
  while (a.KP < a.K) a.KP <<= 1;
  a.CPW = 64 / a.KP;
  // 32 intervals a chunk, or down to 8 while that leaves under 512 wavefronts (a chunk is a sequential chain; kernels of
  // a training step at K = 16, T = 32 / 16 / 8: 24 wavefronts at T = 32 158 / 100 / 77 us, 312: 163 / 127 / 135, 3120:
  // 394 / 436 / 553)
  a.T = s->chunk ? s->chunk : 32;
  if (!s->chunk)
    while (a.T > 8 && (long)a.B * ((a.n + a.T - 1) / a.T) < 512L * a.CPW) a.T /= 2;
  a.C = (a.n + a.T - 1) / a.T;
  a.flow_mode = s->flow_mode;
  a.leaf_mode = s->leaf_mode;
  a.readout = s->readout;
  a.lvl0 = s->level0 ? 1 : 0;
  a.W = a.lvl0 + a.d;
  a.q = s->series_q;
  return a;
}

size_t al256c(size_t x) { return (x + 255) & ~(size_t)255; }
size_t carries_bytes(const CArgs& a) { return al256c((size_t)a.B * (a.C + 1) * a.K * a.M * 16); }
size_t chunk_state_bytes(const CArgs& a) { return al256c((size_t)a.B * a.C * a.K * a.M * 16); }

// the workspace: summaries (forward); mu, mt, the boundary cotangents and the partials (backward)
struct WsOff {
  size_t summ, mu, mt, dvb, dhb, pp, st, total;
};
WsOff ws_off(const CArgs& a) {
  WsOff w{};
  size_t o = 0;
  w.summ = o; o += chunk_state_bytes(a);
  w.mu = o; o += chunk_state_bytes(a);
  w.mt = o; o += chunk_state_bytes(a);
  w.dvb = o; o += al256c((size_t)a.B * a.C * 2 * a.d * 4);
  w.dhb = o; o += al256c((size_t)a.B * a.C * 2 * 4);
  w.pp = o; o += al256c((size_t)a.B * a.C * a.K * 5 * 8);
  w.st = o; o += al256c((size_t)a.B * a.n * a.d * 4);
  w.total = o;
  return w;
}

// threads of a carry-scan workgroup: one per chunk up to 256, in whole wavefronts
int carry_threads(int C) { return std::min(chain::kCarryThreads, std::max(64, (C + 63) / 64 * 64)); }

#define EWS_CHAIN_LAUNCH(KERNEL, GRID, BLK, LDS, ST, A)                                                       \
  do {                                                                                                        \
    const bool cp = (A).cplx != 0;                                                                            \
    switch ((A).M) {                                                                                          \
      case 1:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<1, true>), GRID, BLK, LDS, ST, A);                                  \
        else hipLaunchKernelGGL((KERNEL<1, false>), GRID, BLK, LDS, ST, A);                                    \
        break;                                                                                                \
      case 2:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<2, true>), GRID, BLK, LDS, ST, A);                                  \
        else hipLaunchKernelGGL((KERNEL<2, false>), GRID, BLK, LDS, ST, A);                                    \
        break;                                                                                                \
      case 3:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<3, true>), GRID, BLK, LDS, ST, A);                                  \
        else hipLaunchKernelGGL((KERNEL<3, false>), GRID, BLK, LDS, ST, A);                                    \
        break;                                                                                                \
      default:                                                                                                \
        if (cp) hipLaunchKernelGGL((KERNEL<4, true>), GRID, BLK, LDS, ST, A);                                  \
        else hipLaunchKernelGGL((KERNEL<4, false>), GRID, BLK, LDS, ST, A);                                    \
        break;                                                                                                \
    }                                                                                                         \
    if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;                                               \
  } while (0)

#define EWS_CHAIN_LAUNCH2(KERNEL, GRID, BLK, ST, A, ARG, PTR)                                                  \
  do {                                                                                                        \
    const bool cp = (A).cplx != 0;                                                                            \
    switch ((A).M) {                                                                                          \
      case 1:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<1, true>), GRID, BLK, 0, ST, ARG, PTR);                             \
        else hipLaunchKernelGGL((KERNEL<1, false>), GRID, BLK, 0, ST, ARG, PTR);                               \
        break;                                                                                                \
      case 2:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<2, true>), GRID, BLK, 0, ST, ARG, PTR);                             \
        else hipLaunchKernelGGL((KERNEL<2, false>), GRID, BLK, 0, ST, ARG, PTR);                               \
        break;                                                                                                \
      case 3:                                                                                                 \
        if (cp) hipLaunchKernelGGL((KERNEL<3, true>), GRID, BLK, 0, ST, ARG, PTR);                             \
        else hipLaunchKernelGGL((KERNEL<3, false>), GRID, BLK, 0, ST, ARG, PTR);                               \
        break;                                                                                                \
      default:                                                                                                \
        if (cp) hipLaunchKernelGGL((KERNEL<4, true>), GRID, BLK, 0, ST, ARG, PTR);                             \
        else hipLaunchKernelGGL((KERNEL<4, false>), GRID, BLK, 0, ST, ARG, PTR);                               \
        break;                                                                                                \
    }                                                                                                         \
    if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;                                               \
  } while (0)

}  // namespace
}  // namespace ews

extern "C" {

size_t ews_chain_residual_bytes(const ews_chain_desc* desc) {
  if (ews::chain_check(desc) != EWS_OK) return 0;
  return ews::carries_bytes(ews::chain_args(desc));
}

size_t ews_chain_workspace_bytes(const ews_chain_desc* desc) {
  if (ews::chain_check(desc) != EWS_OK) return 0;
  return ews::ws_off(ews::chain_args(desc)).total;
}

int ews_chain_forward(const ews_chain_desc* desc, const void* path, const float* clock, const float* A, float* out,
                      void* residual, void* workspace, ews_stream_t stream) {
  const int rc = ews::chain_check(desc);
  if (rc != EWS_OK) return rc;
  if (!path || !clock || !A || !out || !residual || !workspace) return EWS_ERR_NULL;
  ews::chain::CArgs a = ews::chain_args(desc);
  a.path = (const float*)path;
  a.clock = clock;
  a.A = A;
  a.out = out;
  a.carries = (double*)residual;
  a.summ = (double*)((char*)workspace + ews::ws_off(a).summ);
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((a.C + a.CPW - 1) / a.CPW, a.B), blk(64);
  EWS_CHAIN_LAUNCH(ews::chain::k_summary, grid, blk, 0, st, a);
  const dim3 ct(ews::carry_threads(a.C));
  EWS_CHAIN_LAUNCH(ews::chain::k_carry, dim3(a.B * a.K), ct, 0, st, a);
  if (a.readout == EWS_READOUT_PREFIX) {
    EWS_CHAIN_LAUNCH(ews::chain::k_rows, grid, blk, 0, st, a);
  } else {
    const dim3 gt((a.B * a.W + 255) / 256);
    EWS_CHAIN_LAUNCH(ews::chain::k_terminal, gt, dim3(256), 0, st, a);
  }
  return EWS_OK;
}

int ews_chain_backward(const ews_chain_desc* desc, const void* path, const float* clock, const float* A,
                       const void* residual, const float* grad_out, float* grad_path, float* grad_clock,
                       float* grad_A, void* workspace, ews_stream_t stream) {
  const int rc = ews::chain_check(desc);
  if (rc != EWS_OK) return rc;
  if (!path || !clock || !A || !residual || !grad_out || !grad_path || !grad_A || !workspace) return EWS_ERR_NULL;
  ews::chain::CArgs a = ews::chain_args(desc);
  a.path = (const float*)path;
  a.clock = clock;
  a.A = A;
  a.gout = grad_out;
  a.carries = (double*)residual;
  const ews::WsOff w = ews::ws_off(a);
  char* ws = (char*)workspace;
  a.summ = (double*)(ws + w.summ);
  a.mu = (double*)(ws + w.mu);
  a.mt = (double*)(ws + w.mt);
  a.dvb = (float*)(ws + w.dvb);
  a.dhb = (float*)(ws + w.dhb);
  a.pp = (double*)(ws + w.pp);
  a.st = (float*)(ws + w.st);
  a.gpath = grad_path;
  a.gclock = grad_clock;
  a.gA = grad_A;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((a.C + a.CPW - 1) / a.CPW, a.B), blk(64);
  if (a.readout == EWS_READOUT_PREFIX) EWS_CHAIN_LAUNCH(ews::chain::k_local, grid, blk, 0, st, a);
  EWS_CHAIN_LAUNCH(ews::chain::k_carry_bwd, dim3(a.B * a.K), dim3(ews::carry_threads(a.C)), 0, st, a);
  EWS_CHAIN_LAUNCH(ews::chain::k_full, grid, blk, 0, st, a);
  const size_t kt = (size_t)a.B * (a.C + 1) * (a.d + 1);
  hipLaunchKernelGGL(ews::chain::k_bounds, dim3((unsigned)((kt + 255) / 256)), dim3(256), 0, st, a);
  if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;
  hipLaunchKernelGGL(ews::chain::k_zero_a, dim3((a.d * a.d + 255) / 256), dim3(256), 0, st, a);
  if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;
  hipLaunchKernelGGL(ews::chain::k_params, dim3(a.K * 3), dim3(ews::chain::kParamThreads), 0, st, a);
  return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
}

size_t ews_chain_cache_workspace_bytes(const ews_chain_desc* desc) {
  if (ews::chain_check(desc) != EWS_OK) return 0;
  return ews::al256c((size_t)desc->batch * (desc->dim / desc->size) * 4 * 8);
}

int ews_chain_cache(const ews_chain_desc* desc, const float* dx, const float* dtheta, const float* A, float* P_cache,
                    float* D_cache, ews_stream_t stream) {
  const int rc = ews::chain_check(desc);
  if (rc != EWS_OK) return rc;
  if (!dx || !dtheta || !A || !P_cache || !D_cache) return EWS_ERR_NULL;
  const ews::chain::CArgs a = ews::chain_args(desc);
  ews::chain::KArgs k{};
  k.V = a.B; k.d = a.d; k.K = a.K; k.size = a.size; k.q = a.q;
  k.dx = dx; k.dth = dtheta; k.P = P_cache; k.D = D_cache;
  hipStream_t st = (hipStream_t)stream;
  EWS_CHAIN_LAUNCH2(ews::chain::k_cache, dim3(a.B), dim3(256), st, a, k, A);
  return EWS_OK;
}

int ews_chain_cache_backward(const ews_chain_desc* desc, const float* dx, const float* dtheta, const float* A,
                             const float* grad_P, const float* grad_D, float* grad_dx, float* grad_dtheta,
                             float* grad_A, void* workspace, ews_stream_t stream) {
  const int rc = ews::chain_check(desc);
  if (rc != EWS_OK) return rc;
  if (!dx || !dtheta || !A || !grad_P || !grad_D || !grad_dx || !grad_dtheta || !grad_A || !workspace)
    return EWS_ERR_NULL;
  const ews::chain::CArgs a = ews::chain_args(desc);
  ews::chain::KArgs k{};
  k.V = a.B; k.d = a.d; k.K = a.K; k.size = a.size; k.q = a.q;
  k.dx = dx; k.dth = dtheta; k.gP = grad_P; k.gD = grad_D;
  k.gdx = grad_dx; k.gdth = grad_dtheta; k.gA = grad_A;
  k.pp = (double*)workspace;
  hipStream_t st = (hipStream_t)stream;
  EWS_CHAIN_LAUNCH2(ews::chain::k_cache_bwd, dim3((unsigned)(((size_t)a.B * a.K + 63) / 64)), dim3(64), st, a, k, A);
  hipLaunchKernelGGL(ews::chain::k_cache_sums, dim3(1 + (a.B + 1023) / 1024), dim3(1024), 0, st, k, a.M, a.cplx);
  return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
}

}  // extern "C"
