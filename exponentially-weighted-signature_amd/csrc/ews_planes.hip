// Wave-per-chunk kernels for rotation planes at depth 2 and any width (d = 6 to 32; d = 16 has its own pair-group
// kernels in ews_pairs.hip): chunk classification and summaries, prefix rows, chunk-local adjoints, and the full adjoint of chunks
// whose clock steps are uniform to float32 precision (flag kStrict). The recursion is the one of ews_diag.hip.
//
// The generic kernels take a lane per pair (j, k): at d = 24 three wavefronts per chunk, the row and column sums of
// every adjoint step through LDS behind two workgroup barriers, and the level-1 work of plane j repeated by all K of its
// lanes. Here one wavefront owns a chunk (two chunks at up to 8 planes): lane (j, kg), kg = 0..3, holds plane j's level 1
// and the KP = ceil(K / 4) pairs (j, KP kg ..), so a row sum is KP additions and a quad exchange, the plane's own work is
// shared by KP pairs, column terms wait in LDS for a block of NB steps, and nothing waits on another wavefront. The
// cotangent rows come straight into registers NB steps ahead. B = 8, L = 49,920, d = 24, bfloat16 path (399k intervals):
// full adjoint 964 -> 403 us, chunk-local adjoints 377 -> 298, rows 305 -> 225, summaries 160 -> 121. The full adjoint is
// bound by instruction issue, the local one by its 0.96 GB of cotangents.
//
// States, coefficients and cotangents are kept halved or doubled (half SA, SB, phi_k, IB, IA; twice the pair cotangents),
// which takes the factors 1/2 of the row layout out of every step, as in ews_pairs.hip.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ews_args.h"
#include "ews_hip.h"
#include "ews_lanes.h"
#include "ews_numerics.h"
#include "ews_planes.h"

namespace ews {
namespace planes {

constexpr int kMaxT = 64;  // longest chunk (a lane per step in the classification)
constexpr int kUniform = 1, kInvert = 2, kSmall = 8, kStrict = 16;  // chunk class bits (ews_diag.hip)

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ cf cjm(cf a, cf b) { return cf{fmaf(a.re, b.re, a.im * b.im), fmaf(a.re, b.im, -a.im * b.re)}; }
__device__ __forceinline__ cf fma_c(cf a, cf b, cf c) {
  return cf{fmaf(a.re, b.re, fmaf(-a.im, b.im, c.re)), fmaf(a.re, b.im, fmaf(a.im, b.re, c.im))};
}
template <int I, int N, class F> __device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}
template <int I, class F> __device__ __forceinline__ void static_down(F&& f) {
  if constexpr (I >= 0) {
    f(std::integral_constant<int, I>{});
    static_down<I - 1>(f);
  }
}
__device__ __forceinline__ void wave_order() { __builtin_amdgcn_wave_barrier(); }

// R plane rows per chunk group (8 or 16): G = 4 R lanes per chunk, GPW chunks per wavefront
template <int R> struct Geo {
  static constexpr int G = 4 * R, GPW = 64 / G;
};
template <int G> __device__ __forceinline__ float group_max(float v) {
  v = fmaxf(v, lanes::dpp<lanes::kXor1>(v));
  v = fmaxf(v, lanes::dpp<lanes::kXor2>(v));
  v = fmaxf(v, lanes::dpp<lanes::kHalfMirror>(v));
  v = fmaxf(v, lanes::dpp<lanes::kMirror>(v));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  if constexpr (G == 64) {
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
  }
  return v;
}
__device__ __forceinline__ cf sum4(cf v) { return cf{lanes::sum4(v.re), lanes::sum4(v.im)}; }

__device__ __forceinline__ cf load_u(const float* params, int j) { return cf{-params[2 * j], params[2 * j + 1]}; }
__device__ __forceinline__ float load_path(const DiagArgs& a, size_t idx) {
  if (a.path_bf16) return __uint_as_float(((unsigned)reinterpret_cast<const unsigned short*>(a.path)[idx]) << 16);
  return reinterpret_cast<const float*>(a.path)[idx];
}

// The lane's place: its group's chunk, its plane, its pairs. Lanes past K take the last plane, pairs past K the row's
// last pair (their values are finite copies that no result reads).
template <int R, int KP> struct Lane {
  int gi, gl, j, kg, c, t0, Tc, ci;
  bool row, owns;  // row: a real plane; owns: the chunk exists and is this kernel's
  bool full;  // K = 4 KP: no pair of a row is padding (a lane past K repeats the last plane, writing its values again)
  int k[KP];
  bool live[KP];
  __device__ __forceinline__ bool counts(int q) const { return full || live[q]; }
  __device__ __forceinline__ Lane(const DiagArgs& a, int b, int need) {
    constexpr int G = Geo<R>::G;
    gl = threadIdx.x % G;
    gi = threadIdx.x / G;
    const int jr = gl >> 2;
    kg = gl & 3;
    row = jr < a.K;
    full = a.K == 4 * KP;
    j = min(jr, a.K - 1);
    c = blockIdx.x * Geo<R>::GPW + gi;
    ci = b * a.C + min(c, a.C - 1);
    owns = c < a.C && (need == 0 || (a.cflag[ci] & need) == need);
    t0 = min(c, a.C - 1) * a.T;
    Tc = min(a.T, a.n_int - t0);
    static_for<0, KP>([&](auto qc) {
      constexpr int q = qc;
      const int kk = kg * KP + q;
      live[q] = row && kk < a.K;
      k[q] = min(kk, a.K - 1);
    });
  }
};

// Increments of the group's chunk into LDS (row t at t d), eight steps' loads in flight per lane.
template <int R> __device__ __forceinline__ void stage(const DiagArgs& a, int b, int gl, int t0, int Tc, float* s_v) {
  constexpr int G = Geo<R>::G;
  const size_t base = ((size_t)b * a.L + t0) * a.d;
  const int n = Tc * a.d;
  for (int i = gl; i < n; i += 8 * G) {
    float x0[8], x1[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const size_t e = base + min(i + u * G, n - 1);
      x0[u] = load_path(a, e);
      x1[u] = load_path(a, e + a.d);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i + u * G < n) s_v[i + u * G] = x1[u] - x0[u];
  }
}
template <int R, int KP>
__device__ __forceinline__ void load_p(const float* v, const Lane<R, KP>& l, cf& pj, cf* pk) {
  const float2 x = *reinterpret_cast<const float2*>(v + 2 * l.j);
  pj = cf{x.x, x.y};
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    const float2 y = *reinterpret_cast<const float2*>(v + 2 * l.k[q]);
    pk[q] = cf{y.x, y.y};
  });
}

// e^{h u} in float64 for |h u| <= kPolyR (degree-14 Taylor: remainder below 1e-18), rounded once by the caller
struct cd {
  double re, im;
};
__device__ __forceinline__ cd mul(cd a, cd b) { return cd{fma(a.re, b.re, -a.im * b.im), fma(a.re, b.im, a.im * b.re)}; }
__device__ __forceinline__ cd exp_small(double h, cf u) {
  const cd x{h * (double)u.re, h * (double)u.im};
  cd r{1.0, 0.0};
#pragma unroll
  for (int m = 14; m >= 1; --m) {
    r = mul(r, x);
    r.re = fma(r.re, 1.0 / m, 1.0);
    r.im *= 1.0 / m;
  }
  return r;
}
__device__ __forceinline__ cd fma_d(cd a, cd b, cd c) {
  return cd{fma(a.re, b.re, fma(-a.im, b.im, c.re)), fma(a.re, b.im, fma(a.im, b.re, c.im))};
}
__device__ __forceinline__ cd flow_d(double h, cf u, bool small) {
  if (small) return exp_small(h, u);
  const double m = exp(h * (double)u.re);
  double sn, cs;
  sincos(h * (double)u.im, &sn, &cs);
  return cd{m * cs, m * sn};
}
__device__ __forceinline__ cf to_f(cd a) { return cf{(float)a.re, (float)a.im}; }

// Coefficients at the chunk's mean step. small: the polynomial model (ews_numerics.h kPolyR) with the flows from float64
// exponentials; else the closed forms. INV: the inverse flows too.
template <int KP, bool INV> struct Coefs {
  cf rho, rhoi, phi;
  cf phk[KP], IB[KP], IA[KP];           // halved
  cf LB[KP], LA[KP], LBi[KP], LAi[KP];
};
template <int KP, bool INV>
__device__ __forceinline__ void eval(const DiagArgs& a, int j, const int* k, float h, bool small, Coefs<KP, INV>& f) {
  const cf uj = load_u(a.params, j);
  if (small) {
    cf p[kPolyD + 1];
    poly_phi(uj, p);
    f.phi = poly_val<kPolyPhi>(p, h);
    const cd rj = exp_small(h, uj);
    f.rho = to_f(rj);
    cd ij{1.0, 0.0};
    if (INV) {
      ij = exp_small(-(double)h, uj);
      f.rhoi = to_f(ij);
    }
    static_for<0, KP>([&](auto qc) {
      constexpr int q = qc;
      const cf uk = load_u(a.params, k[q]);
      poly_phi(uk, p);
      f.phk[q] = 0.5f * poly_val<kPolyPhi>(p, h);
      poly_dd3(uj, uj + uk, p);
      f.IB[q] = 0.5f * poly_val<kPolyD>(p, h);
      poly_dd3(uj, uj + conj(uk), p);
      f.IA[q] = 0.5f * poly_val<kPolyD>(p, h);
      const cd rk = exp_small(h, uk);
      f.LB[q] = to_f(mul(rj, rk));
      f.LA[q] = to_f(mul(rj, cd{rk.re, -rk.im}));
      if (INV) {
        const cd ik = exp_small(-(double)h, uk);
        f.LBi[q] = to_f(mul(ij, ik));
        f.LAi[q] = to_f(mul(ij, cd{ik.re, -ik.im}));
      }
    });
    return;
  }
  const cf xj = h * uj;
  const Node1<cf> nj = node1q(xj, a.sq1);
  f.rho = nj.e;
  f.phi = nj.p;
  if (INV) f.rhoi = expv(-xj);
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    const cf uk = load_u(a.params, k[q]);
    const cf ub = uj + uk, ua = uj + conj(uk);
    f.phk[q] = 0.5f * node1q(h * uk, a.sq1).p;
    f.IB[q] = 0.5f * dd3q<cf, false>(xj, h * ub, a.sq2).d;
    f.IA[q] = 0.5f * dd3q<cf, false>(xj, h * ua, a.sq2).d;
    f.LB[q] = expv(h * ub);
    f.LA[q] = expv(h * ua);
    if (INV) {
      f.LBi[q] = expv(-(h * ub));
      f.LAi[q] = expv(-(h * ua));
    }
  });
}

// ------------------------------------------------------------------------------------------------ summaries
// The chunk's class, a lane per step: uniform (within 2^-16 / 2R of the mean, as the generic kernels take first-order
// models), strict (steps and their running sum within 2^-21 / R: constant coefficients), invertible, small.
template <int G>
__device__ __forceinline__ int classify(const DiagArgs& a, int b, int t0, int Tc, int gl, float& hb) {
  const float* th = a.clock + (size_t)b * a.L + t0;
  const float th0 = th[0], tau = th[Tc] - th0;
  hb = tau / (float)Tc;
  float dev = 0.0f, drift = 0.0f, hmax = 0.0f, bad = 0.0f, back = 0.0f, R = 0.0f, Dm = 0.0f, Gm = 0.0f;
  for (int t = gl; t < Tc; t += G) {
    const float x0 = th[t], x1 = th[t + 1], h = x1 - x0;
    if (!isfinite(h)) bad = 1.0f;
    dev = fmaxf(dev, fabsf(h - hb));
    drift = fmaxf(drift, fabsf((x1 - th0) - (float)(t + 1) * hb));
    hmax = fmaxf(hmax, fabsf(h));
    back += fmaxf(-h, 0.0f);
  }
  if (gl < a.K) {
    const cf u = load_u(a.params, gl);
    R = absv(u);
    Dm = fmaxf(0.0f, -u.re);
    Gm = fmaxf(0.0f, u.re);
    if (!isfinite(R)) bad = 1.0f;
  }
  dev = group_max<G>(dev);
  drift = group_max<G>(drift);
  hmax = group_max<G>(hmax);
  bad = group_max<G>(bad);
  R = group_max<G>(R);
  Dm = group_max<G>(Dm);
  Gm = group_max<G>(Gm);
  back = lanes::sum_n(back, G);
  const bool fin = bad == 0.0f && isfinite(tau);
  const float lim = 4.76837158e-7f;  // 2^-21
  const bool uni = fin && dev * 2.0f * R < 1.52587890625e-5f;
  const bool strict = uni && R * dev <= lim && R * drift <= lim;
  const bool inv = fin && invert_growth(tau, back, Dm, Gm) <= 0.69314718f;
  const bool small = fin && poly_order_ok(a.sq1, a.sq2) && poly_small(R, hmax);
  return (uni ? kUniform : 0) | (inv ? kInvert : 0) | (small ? kSmall : 0) | (strict ? kStrict : 0);
}

// A clock whose rounding passes the strict bound part way (float32 values double their spacing at every power of two) splits
// a sample between these kernels and the generic ones, and with few chunks each side only takes the length of its own
// chains: B = 16, L = 8192, clock from 0 to 8, one training pass 459 us split and 334 us by the generic kernels alone (d = 10;
// d = 18 714 and 613). Below kFewWaves wavefronts a sample is strict as a whole or not at all: not where its last full chunk
// is uniform without being strict. With more of them the split gains (B = 8, L = 49,920, 3120 wavefronts, d = 6: 545 us and
// 622 alone; d = 14 849 and 888), and at 16 planes, where the generic kernels take 256 lanes a chunk, at any number.
constexpr int kFewWaves = 3072;
template <int G, int GPW>
__device__ __forceinline__ int classify_chunk(const DiagArgs& a, int b, int t0, int Tc, int gl, float& hb) {
  int f = classify<G>(a, b, t0, Tc, gl, hb);
  const int last = (a.n_int / a.T - 1) * a.T;  // the last full chunk's first step
  if (a.K < 16 && (long)a.B * ((a.C + GPW - 1) / GPW) < kFewWaves && last >= 0) {
    float hl;
    const int fl = classify<G>(a, b, last, a.T, gl, hl);
    if ((fl & (kUniform | kStrict)) == kUniform) f &= ~kStrict;
  }
  return f;
}

// Level 1 runs in float64: its roundings over a chunk, and that of its flow, are what the states' error at L = 50k came
// from (level 2 takes them over: rows 5.8e-6 off with float32 here, 2.9e-6 with float64; 114 -> 121 us).
template <int R, int KP>
__global__ __launch_bounds__(64) void k_summary(DiagArgs a) {
  constexpr int G = Geo<R>::G, GPW = Geo<R>::GPW;
  __shared__ __align__(16) float s_v[GPW][kMaxT * 8 * KP];
  const int b = blockIdx.y;
  const Lane<R, KP> l(a, b, 0);
  float hb;
  const int flag = classify_chunk<G, GPW>(a, b, l.t0, l.Tc, l.gl, hb);
  if (l.owns && l.gl == 0) {
    a.cflag[l.ci] = flag;
    a.chbar[l.ci] = hb;
  }
  const bool mine = l.owns && (flag & kStrict);
  if (!__any(mine)) return;
  float* vg = s_v[l.gi];
  stage<R>(a, b, l.gl, l.t0, l.Tc, vg);
  Coefs<KP, false> f;
  eval<KP, false>(a, l.j, l.k, hb, (flag & kSmall) != 0, f);
  wave_order();
  const bool small = (flag & kSmall) != 0;
  const cf uj = load_u(a.params, l.j);
  const cd rho = flow_d(hb, uj, small), phi{(double)f.phi.re, (double)f.phi.im};
  cd S1{0.0, 0.0};
  cf SA[KP], SB[KP];
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    SA[q] = SB[q] = cf{0.0f, 0.0f};
  });
  for (int t = 0; t < l.Tc; ++t) {
    cf pj, pk[KP];
    load_p<R, KP>(vg + t * a.d, l, pj, pk);
    const cd cd1 = mul(rho, S1);
    const cf cj = to_f(cd1);
    S1 = fma_d(phi, cd{(double)pj.re, (double)pj.im}, cd1);
    static_for<0, KP>([&](auto qc) {
      constexpr int q = qc;
      const cf sg = f.phk[q] * pk[q];
      const float aa = pj.re * pk[q].re, bb = pj.im * pk[q].im, cc = pj.re * pk[q].im, dd = pj.im * pk[q].re;
      SB[q] = fma_c(f.LB[q], SB[q], fma_c(cj, sg, f.IB[q] * cf{aa - bb, cc + dd}));
      SA[q] = fma_c(f.LA[q], SA[q], fma_c(cj, conj(sg), f.IA[q] * cf{aa + bb, dd - cc}));
    });
  }
  if (!mine || !l.row) return;
  float* sp = a.summ + (size_t)l.ci * a.D;
  if (l.kg == 0) *reinterpret_cast<f2u*>(sp + 2 * l.j) = f2u{(float)S1.re, (float)S1.im};
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    if (l.live[q])
      *reinterpret_cast<f4u*>(sp + a.d + 4 * (l.j * a.K + l.k[q])) =
          f4u{2.0f * SA[q].re, 2.0f * SA[q].im, 2.0f * SB[q].re, 2.0f * SB[q].im};
  });
}

// ------------------------------------------------------------------------------------------------ prefix rows
// A strictly uniform chunk's prefix rows from its float64 carry. Each step's level-2 block goes through LDS, so that the
// row leaves as contiguous 16-byte stores (1 KB per instruction); the write stream bounds it.
template <int R, int KP>
__global__ __launch_bounds__(64) void k_rows(DiagArgs a) {
  constexpr int G = Geo<R>::G, GPW = Geo<R>::GPW;
  __shared__ __align__(16) float s_v[GPW][kMaxT * 8 * KP];
  __shared__ __align__(16) float s_row[GPW][64 * KP * KP];
  const int b = blockIdx.y;
  const Lane<R, KP> l(a, b, kUniform | kStrict);
  if (!__any(l.owns)) return;
  float* vg = s_v[l.gi];
  float* buf = s_row[l.gi];
  stage<R>(a, b, l.gl, l.t0, l.Tc, vg);
  Coefs<KP, false> f;
  eval<KP, false>(a, l.j, l.k, a.chbar[l.ci], (a.cflag[l.ci] & kSmall) != 0, f);
  cf S1, SA[KP], SB[KP];
  const double* cr = a.carries + ((size_t)b * (a.C + 1) + min(l.c, a.C - 1)) * a.D;
  S1 = cf{(float)cr[2 * l.j], (float)cr[2 * l.j + 1]};
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    const int e = a.d + 4 * (l.j * a.K + l.k[q]);
    SA[q] = cf{(float)(0.5 * cr[e]), (float)(0.5 * cr[e + 1])};
    SB[q] = cf{(float)(0.5 * cr[e + 2]), (float)(0.5 * cr[e + 3])};
  });
  wave_order();
  float* row = a.out + ((size_t)b * a.n_int + l.t0) * a.W;
  const int n4 = a.d * a.d / 4;  // d is even: whole quads
  for (int t = 0; t < l.Tc; ++t, row += a.W) {
    cf pj, pk[KP];
    load_p<R, KP>(vg + t * a.d, l, pj, pk);
    const cf cj = f.rho * S1;
    S1 = fma_c(f.phi, pj, cj);
    static_for<0, KP>([&](auto qc) {
      constexpr int q = qc;
      const cf sg = f.phk[q] * pk[q];
      const float aa = pj.re * pk[q].re, bb = pj.im * pk[q].im, cc = pj.re * pk[q].im, dd = pj.im * pk[q].re;
      SB[q] = fma_c(f.LB[q], SB[q], fma_c(cj, sg, f.IB[q] * cf{aa - bb, cc + dd}));
      SA[q] = fma_c(f.LA[q], SA[q], fma_c(cj, conj(sg), f.IA[q] * cf{aa + bb, dd - cc}));
      if (l.live[q]) {  // the real 2 x 2 block of the halved states
        float* r0 = buf + 2 * l.j * a.d + 2 * l.k[q];
        *reinterpret_cast<float2*>(r0) = float2{SA[q].re + SB[q].re, SB[q].im - SA[q].im};
        *reinterpret_cast<float2*>(r0 + a.d) = float2{SA[q].im + SB[q].im, SA[q].re - SB[q].re};
      }
    });
    wave_order();
    if (l.owns) {
      if (a.lvl0 && l.gl == 0) row[0] = 1.0f;
      if (l.kg == 0 && l.row) *reinterpret_cast<f2u*>(row + a.off1 + 2 * l.j) = f2u{S1.re, S1.im};
      for (int i = l.gl; i < n4; i += G) {
        const float4 v = *reinterpret_cast<const float4*>(buf + 4 * i);
        *reinterpret_cast<f4u*>(row + a.off2 + 4 * i) = f4u{v.x, v.y, v.z, v.w};
      }
    }
    wave_order();
  }
}

// ------------------------------------------------------------------------------------------------ cotangent rows
// The lane's part of one cotangent row: level 1 of plane j and the 2 x 2 blocks of its pairs.
template <int KP> struct GRow {
  f2u g1, r0[KP], r1[KP];
};
template <int R, int KP>
__device__ __forceinline__ GRow<KP> load_g(const float* row, int o1, int o2, int d, const Lane<R, KP>& l) {
  GRow<KP> g;
  g.g1 = *reinterpret_cast<const f2u*>(row + o1);
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    g.r0[q] = *reinterpret_cast<const f2u*>(row + o2 + 2 * l.k[q]);
    g.r1[q] = *reinterpret_cast<const f2u*>(row + o2 + d + 2 * l.k[q]);
  });
  return g;
}

// The row cotangent added to the doubled pair cotangents (block entries g00, g01 / g10, g11) and to level 1 (w1 of it).
// Every use of a ring slot lies here, before the slot is loaded again: a copy of a row kept across its slot's reload made
// the compiler drain all loads in every step (full adjoint 1.9 ms).
template <int KP>
__device__ __forceinline__ void add_g(const GRow<KP>& g, float w1, cf& l1, cf* lA, cf* lB) {
  l1.re = fmaf(w1, g.g1.x, l1.re);
  l1.im = fmaf(w1, g.g1.y, l1.im);
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    lA[q] += cf{g.r0[q].x + g.r1[q].y, g.r1[q].x - g.r0[q].y};
    lB[q] += cf{g.r0[q].x - g.r1[q].y, g.r0[q].y + g.r1[q].x};
  });
}

// ------------------------------------------------------------------------------------------------ local adjoint
// mu: the cotangent on the chunk's carry-in state of its own rows. By linearity each lane carries its pairs' share of
// plane j's level-1 cotangent, summed over the quad at the end.
template <int R, int KP>
__global__ __launch_bounds__(64) void k_local(DiagArgs a) {
  constexpr int GPW = Geo<R>::GPW, RING = 4;
  __shared__ __align__(16) float s_v[GPW][kMaxT * 8 * KP];
  const int b = blockIdx.y;
  const Lane<R, KP> l(a, b, kUniform | kStrict);
  if (!__any(l.owns)) return;
  float* vg = s_v[l.gi];
  const int o1 = a.off1 + 2 * l.j, o2 = a.off2 + 2 * l.j * a.d;
  const float* grow = a.gout + ((size_t)b * a.n_int + l.t0) * a.W;
  const int nblk = (a.T + RING - 1) / RING;
  GRow<KP> ring[RING];
  static_for<0, RING>([&](auto ic) {
    constexpr int i = ic;
    ring[i] = load_g<R, KP>(grow + (size_t)max(min(nblk * RING - 1 - i, l.Tc - 1), 0) * a.W, o1, o2, a.d, l);
  });
  stage<R>(a, b, l.gl, l.t0, l.Tc, vg);
  Coefs<KP, false> f;
  eval<KP, false>(a, l.j, l.k, a.chbar[l.ci], (a.cflag[l.ci] & kSmall) != 0, f);
  wave_order();
  const float w1 = l.kg == 0 ? 1.0f : 0.0f;
  cf l1{0.0f, 0.0f}, lA[KP], lB[KP];
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    lA[q] = lB[q] = cf{0.0f, 0.0f};
  });
  for (int blk = nblk - 1; blk >= 0; --blk) {
    static_for<0, RING>([&](auto ic) {
      constexpr int i = ic;
      const int t = blk * RING + RING - 1 - i;
      if (t < l.Tc) add_g<KP>(ring[i], w1, l1, lA, lB);
      ring[i] = load_g<R, KP>(grow + (size_t)max(min(t - RING, l.Tc - 1), 0) * a.W, o1, o2, a.d, l);
      if (t >= l.Tc) return;
      cf pj, pk[KP];
      load_p<R, KP>(vg + t * a.d, l, pj, pk);
      cf toC{0.0f, 0.0f};
      static_for<0, KP>([&](auto qc) {
        constexpr int q = qc;
        if (l.counts(q)) {
          const cf sg = f.phk[q] * pk[q];
          toC += cjm(sg, lB[q]) + sg * lA[q];
        }
        lB[q] = cjm(f.LB[q], lB[q]);
        lA[q] = cjm(f.LA[q], lA[q]);
      });
      l1 = cjm(f.rho, l1 + toC);
    });
  }
  l1 = sum4(l1);
  if (!l.owns || !l.row) return;
  float* mp = a.mu + (size_t)l.ci * a.D;
  if (l.kg == 0) *reinterpret_cast<f2u*>(mp + 2 * l.j) = f2u{l1.re, l1.im};
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    if (l.live[q])
      *reinterpret_cast<f4u*>(mp + a.d + 4 * (l.j * a.K + l.k[q])) =
          f4u{0.5f * lA[q].re, 0.5f * lA[q].im, 0.5f * lB[q].re, 0.5f * lB[q].im};
  });
}

// ------------------------------------------------------------------------------------------------ full adjoint
// A chunk from the cotangent at its end (mt) and its rows, the states S(t-1) by inverting each step from the float64
// state at the chunk's end: dv of every step and the chunk's parameter partials.
template <int R, int KP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_full(DiagArgs a) {
  constexpr int G = Geo<R>::G, GPW = Geo<R>::GPW, NB = KP <= 3 ? 4 : 2, RP = R + 1;
  constexpr int NW = NB * 4 * KP * RP * 2, NP = 4 * KP * (RP + 1) * 2 + R * 4;  // column terms; parameter terms
  __shared__ __align__(16) float s_v[GPW][kMaxT * 8 * KP];
  __shared__ __align__(16) float s_w[GPW][NW > NP ? NW : NP];  // w[s][k][j] (complex); at the end the parameter terms
  __shared__ __align__(16) float s_dvp[GPW][NB * R * 2];       // plane part of dv[s][j] (complex)
  __shared__ float s_h[GPW][kMaxT];                            // clock steps
  const int b = blockIdx.y;
  const Lane<R, KP> l(a, b, kUniform | kInvert | kStrict);
  if (!__any(l.owns)) return;
  float* vg = s_v[l.gi];
  const int o1 = a.off1 + 2 * l.j, o2 = a.off2 + 2 * l.j * a.d;
  const float* grow = a.gout + ((size_t)b * a.n_int + l.t0) * a.W;
  const int nblk = (a.T + NB - 1) / NB;
  GRow<KP> ring[NB];
  static_down<NB - 1>([&](auto sc) {
    constexpr int s = sc;
    ring[s] = load_g<R, KP>(grow + (size_t)max(min((nblk - 1) * NB + s, l.Tc - 1), 0) * a.W, o1, o2, a.d, l);
  });
  stage<R>(a, b, l.gl, l.t0, l.Tc, vg);
  float* hg = s_h[l.gi];
  {
    const float* th = a.clock + (size_t)b * a.L + l.t0;
    for (int t = l.gl; t < l.Tc; t += G) hg[t] = th[t + 1] - th[t];
  }
  const float hb = a.chbar[l.ci];
  const bool small = (a.cflag[l.ci] & kSmall) != 0;
  Coefs<KP, true> f;
  eval<KP, true>(a, l.j, l.k, hb, small, f);
  cf S1, SA[KP], SB[KP], l1, lA[KP], lB[KP];
  {
    const double* cr = a.carries + ((size_t)b * (a.C + 1) + min(l.c, a.C - 1) + 1) * a.D;
    const float* mp = a.mt + (size_t)l.ci * a.D;
    S1 = cf{(float)cr[2 * l.j], (float)cr[2 * l.j + 1]};
    l1 = cf{mp[2 * l.j], mp[2 * l.j + 1]};
    static_for<0, KP>([&](auto qc) {
      constexpr int q = qc;
      const int e = a.d + 4 * (l.j * a.K + l.k[q]);
      SA[q] = cf{(float)(0.5 * cr[e]), (float)(0.5 * cr[e + 1])};
      SB[q] = cf{(float)(0.5 * cr[e + 2]), (float)(0.5 * cr[e + 3])};
      lA[q] = cf{2.0f * mp[e], 2.0f * mp[e + 1]};
      lB[q] = cf{2.0f * mp[e + 2], 2.0f * mp[e + 3]};
    });
  }
  // The coefficient cotangents, summed with each step's own h: the coefficients are constant where |u| times the steps'
  // deviation is below 2^-21, but for a small |u| or a fine clock the deviation may be as large as the step (float32
  // values near 1 leave steps of 2e-5 off by 3e-3 of themselves), and a sum times the mean step is then off as much.
  cf kIB[KP], kIA[KP], kLB[KP], kLA[KP], kph[KP], krho{0.0f, 0.0f}, kphj{0.0f, 0.0f};
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    kIB[q] = kIA[q] = kLB[q] = kLA[q] = kph[q] = cf{0.0f, 0.0f};
  });
  float* w_g = s_w[l.gi];
  float* dvp_g = s_dvp[l.gi];
  wave_order();
  for (int blk = nblk - 1; blk >= 0; --blk) {
    const int tb = blk * NB;
    static_down<NB - 1>([&](auto sc) {
      constexpr int s = sc;
      const int t = tb + s;
      if (t < l.Tc) add_g<KP>(ring[s], 1.0f, l1, lA, lB);
      ring[s] = load_g<R, KP>(grow + (size_t)max(min(t - NB, l.Tc - 1), 0) * a.W, o1, o2, a.d, l);
      if (t >= l.Tc) return;
      cf pj, pk[KP];
      load_p<R, KP>(vg + t * a.d, l, pj, pk);
      const float h = hg[t];
      const cf cj = S1 - f.phi * pj;  // c_j = rho S1(t-1)
      const cf H1 = f.rhoi * cj;
      cf toC{0.0f, 0.0f}, toP{0.0f, 0.0f};
      static_for<0, KP>([&](auto qc) {
        constexpr int q = qc;
        // doubled cotangents A, B of SA(t), SB(t); shared sums P = B + A, Q = B - A, F = gf + ge, E = gf - ge
        const float Ar = lA[q].re, Ai = lA[q].im, Br = lB[q].re, Bi = lB[q].im;
        const float Pr = Br + Ar, Pi = Bi + Ai, Qr = Br - Ar, Qi = Bi - Ai;
        const cf pkq = pk[q], ph = f.phk[q];
        const float sgr = fmaf(ph.re, pkq.re, -ph.im * pkq.im), sgi = fmaf(ph.re, pkq.im, ph.im * pkq.re);
        const float aa = pj.re * pkq.re, bb = pj.im * pkq.im, cc = pj.re * pkq.im, dd = pj.im * pkq.re;
        const float pir = aa - bb, pii = cc + dd, pcr = aa + bb, pci = dd - cc;  // p_j p_k, p_j conj(p_k)
        const float rr = cj.re * sgr, ii = cj.im * sgi, ri = cj.re * sgi, ir = cj.im * sgr;
        const cf IB = f.IB[q], IA = f.IA[q];
        // previous states: X = S(t) - local terms, H = flow^-1 X
        const float XBr = fmaf(IB.im, pii, fmaf(-IB.re, pir, SB[q].re - rr + ii));
        const float XBi = fmaf(-IB.im, pir, fmaf(-IB.re, pii, SB[q].im - ri - ir));
        const float XAr = fmaf(IA.im, pci, fmaf(-IA.re, pcr, SA[q].re - rr - ii));
        const float XAi = fmaf(-IA.im, pcr, fmaf(-IA.re, pci, SA[q].im - ir + ri));
        const cf LBi = f.LBi[q], LAi = f.LAi[q];
        const float HBr = fmaf(LBi.re, XBr, -LBi.im * XBi), HBi = fmaf(LBi.re, XBi, LBi.im * XBr);
        const float HAr = fmaf(LAi.re, XAr, -LAi.im * XAi), HAi = fmaf(LAi.re, XAi, LAi.im * XAr);
        const float gfr = fmaf(IB.re, Br, IB.im * Bi), gfi = fmaf(IB.re, Bi, -IB.im * Br);  // conj(IB) B
        const float ger = fmaf(IA.re, Ar, IA.im * Ai), gei = fmaf(IA.re, Ai, -IA.im * Ar);  // conj(IA) A
        const float Fr = gfr + ger, Fi = gfi + gei, Er = gfr - ger, Ei = gfi - gei;
        if (l.counts(q)) {  // row terms (plane j): conj(sg) B + sg A, conj(p_k) gf + p_k ge
          toC.re = fmaf(sgr, Pr, fmaf(sgi, Qi, toC.re));
          toC.im = fmaf(sgr, Pi, fmaf(-sgi, Qr, toC.im));
          toP.re = fmaf(pkq.re, Fr, fmaf(pkq.im, Ei, toP.re));
          toP.im = fmaf(pkq.re, Fi, fmaf(-pkq.im, Er, toP.im));
        }
        // column terms (plane k): tS = conj(c_j) B + conj(A) c_j; w = conj(phi_k / 2) tS + conj(p_j) gf + conj(ge) p_j
        const float tSr = fmaf(cj.re, Pr, cj.im * Pi), tSi = fmaf(cj.re, Qi, -cj.im * Qr);
        const float wr = fmaf(ph.re, tSr, fmaf(ph.im, tSi, fmaf(pj.re, Fr, pj.im * Fi)));
        const float wi = fmaf(ph.re, tSi, fmaf(-ph.im, tSr, fmaf(pj.re, Ei, -pj.im * Er)));
        if (l.counts(q)) *reinterpret_cast<float2*>(w_g + ((s * 4 * KP + l.k[q]) * RP + l.j) * 2) = float2{wr, wi};
        // coefficient cotangents times h: conj(p_k) tS, conj(pi) B, conj(pic) A, conj(HB) B, conj(HA) A
        const float tSrh = h * tSr, tSih = h * tSi, Arh = h * Ar, Aih = h * Ai, Brh = h * Br, Bih = h * Bi;
        kph[q].re = fmaf(pkq.re, tSrh, fmaf(pkq.im, tSih, kph[q].re));
        kph[q].im = fmaf(pkq.re, tSih, fmaf(-pkq.im, tSrh, kph[q].im));
        kIB[q].re = fmaf(pir, Brh, fmaf(pii, Bih, kIB[q].re));
        kIB[q].im = fmaf(pir, Bih, fmaf(-pii, Brh, kIB[q].im));
        kIA[q].re = fmaf(pcr, Arh, fmaf(pci, Aih, kIA[q].re));
        kIA[q].im = fmaf(pcr, Aih, fmaf(-pci, Arh, kIA[q].im));
        kLB[q].re = fmaf(HBr, Brh, fmaf(HBi, Bih, kLB[q].re));
        kLB[q].im = fmaf(HBr, Bih, fmaf(-HBi, Brh, kLB[q].im));
        kLA[q].re = fmaf(HAr, Arh, fmaf(HAi, Aih, kLA[q].re));
        kLA[q].im = fmaf(HAr, Aih, fmaf(-HAi, Arh, kLA[q].im));
        const cf LB = f.LB[q], LA = f.LA[q];
        lB[q] = cf{fmaf(LB.re, Br, LB.im * Bi), fmaf(LB.re, Bi, -LB.im * Br)};
        lA[q] = cf{fmaf(LA.re, Ar, LA.im * Ai), fmaf(LA.re, Ai, -LA.im * Ar)};
        SB[q] = cf{HBr, HBi};
        SA[q] = cf{HAr, HAi};
      });
      toC = sum4(toC);
      toP = sum4(toP);
      const cf gc = l1 + toC;
      if (l.kg == 0 && l.row) {
        const cf dvp = cjm(f.phi, l1) + toP;
        *reinterpret_cast<float2*>(dvp_g + (s * R + l.j) * 2) = float2{dvp.re, dvp.im};
      }
      kphj += cjm(pj, h * l1);
      krho += cjm(H1, h * gc);
      l1 = cjm(f.rho, gc);
      S1 = H1;
    });
    wave_order();
    // column sums of the block: dv[t][k] = plane part + sum_j w[t][k][j]
    for (int it = l.gl; it < NB * a.K; it += G) {
      const int s = it / a.K, k = it - s * a.K, t = tb + s;
      if (t < l.Tc && l.owns) {
        const float2* wp = reinterpret_cast<const float2*>(w_g + (s * 4 * KP + k) * RP * 2);
        float2 dv = *reinterpret_cast<const float2*>(dvp_g + (s * R + k) * 2), e{0.0f, 0.0f};
        int j = 0;
        for (; j + 1 < a.K; j += 2) {
          dv.x += wp[j].x;
          dv.y += wp[j].y;
          e.x += wp[j + 1].x;
          e.y += wp[j + 1].y;
        }
        if (j < a.K) {
          dv.x += wp[j].x;
          dv.y += wp[j].y;
        }
        *reinterpret_cast<f2u*>(a.dv + ((size_t)b * a.n_int + l.t0 + t) * a.d + 2 * k) = f2u{dv.x + e.x, dv.y + e.y};
      }
    }
    wave_order();
  }
  // parameter partials (a moment's further powers of h at the mean step): node cotangents -> (d_j, w_j) per plane. A node h u contributes (-Re G, Im G) to its plane for
  // u = -conj(z) and (-Re G, -Im G) for u = -z (the conj(u_k) of the A pairs).
  const cf uj = load_u(a.params, l.j);
  const cf xj = hb * uj;
  float rd = 0.0f, rw = 0.0f;
  cf Gx{0.0f, 0.0f};
  float* colp = w_g;                         // [k][j] (d, w) column parts, pitch RP + 1 pairs
  float* rowp = w_g + 4 * KP * (RP + 1) * 2;  // [j] (d, w)
  static_for<0, KP>([&](auto qc) {
    constexpr int q = qc;
    const cf uk = load_u(a.params, l.k[q]);
    const cf ub = uj + uk, ua = uj + conj(uk);
    cf gxB, gyB, gxA, gyA, gk;  // sum_t h g_t conj(d coefficient / d node) of the halved coefficients' cotangents
    if (small) {
      cf m[kPolyD];
      auto moments = [&](cf k0) {
        m[0] = k0;
#pragma unroll
        for (int i = 1; i < kPolyD; ++i) m[i] = hb * m[i - 1];
      };
      moments(kIB[q]);
      poly_dd3_node(uj, ub, m, gxB, gyB);
      moments(kIA[q]);
      poly_dd3_node(uj, ua, m, gxA, gyA);
      moments(kph[q]);
      gk = poly_phi_node(uk, m);
    } else {
      const DD3<cf> db = dd3q<cf, true>(xj, hb * ub, a.sq2), da = dd3q<cf, true>(xj, hb * ua, a.sq2);
      gxB = kIB[q] * conj(db.dx);
      gyB = kIB[q] * conj(db.dy);
      gxA = kIA[q] * conj(da.dx);
      gyA = kIA[q] * conj(da.dy);
      gk = kph[q] * conj(node1q(hb * uk, a.sq1).dp);
    }
    const cf GyB = 0.5f * gyB + kLB[q] * conj(f.LB[q]);
    const cf GyA = 0.5f * gyA + kLA[q] * conj(f.LA[q]);
    const cf Gk = 0.5f * gk;
    if (l.live[q]) {
      Gx += 0.5f * (gxB + gxA);
      rd -= GyB.re + GyA.re;
      rw += GyB.im + GyA.im;
      *reinterpret_cast<float2*>(colp + (l.k[q] * (RP + 1) + l.j) * 2) =
          float2{-GyB.re - GyA.re - Gk.re, GyB.im - GyA.im + Gk.im};
    }
  });
  rd = lanes::sum4(rd - Gx.re);
  rw = lanes::sum4(rw + Gx.im);
  if (l.kg == 0 && l.row) {
    cf gp;
    if (small) {
      cf m[kPolyPhi];
      m[0] = kphj;
#pragma unroll
      for (int i = 1; i < kPolyPhi; ++i) m[i] = hb * m[i - 1];
      gp = poly_phi_node(uj, m);
    } else {
      gp = kphj * conj(node1q(xj, a.sq1).dp);
    }
    gp += krho * conj(f.rho);
    *reinterpret_cast<float2*>(rowp + 2 * l.j) = float2{rd - gp.re, rw + gp.im};
  }
  wave_order();
  if (l.owns && l.gl < a.K) {
    const int p = l.gl;
    float sd = rowp[2 * p], sw = rowp[2 * p + 1];
    for (int jj = 0; jj < a.K; ++jj) {
      sd += colp[(p * (RP + 1) + jj) * 2];
      sw += colp[(p * (RP + 1) + jj) * 2 + 1];
    }
    float* gpo = a.gp + (size_t)l.ci * a.npar;
    gpo[2 * p] = sd;
    gpo[2 * p + 1] = sw;
  }
}

}  // namespace planes

bool planes_eligible(const DiagArgs& a) {
  return a.N == 2 && a.K >= 3 && a.K <= 16 && !a.fast_ok && a.readout == EWS_READOUT_PREFIX &&
         a.flow_mode == EWS_FLOW_PER_INTERVAL && a.T <= planes::kMaxT && a.T >= 4 && poly_order_ok(a.sq1, a.sq2);
}

#define EWS_PLANES_LAUNCH(KERNEL)                                                                                      \
  do {                                                                                                                 \
    const dim3 g2((a.C + 1) / 2, a.B), g1(a.C, a.B), blk(64);                                                          \
    if (a.K <= 4) hipLaunchKernelGGL((planes::KERNEL<8, 1>), g2, blk, 0, st, a);                                       \
    else if (a.K <= 8) hipLaunchKernelGGL((planes::KERNEL<8, 2>), g2, blk, 0, st, a);                                  \
    else if (a.K <= 12) hipLaunchKernelGGL((planes::KERNEL<16, 3>), g1, blk, 0, st, a);                                \
    else hipLaunchKernelGGL((planes::KERNEL<16, 4>), g1, blk, 0, st, a);                                               \
    return hipGetLastError() == hipSuccess ? 0 : -1;                                                                   \
  } while (0)

int planes_summary(const DiagArgs& a, hipStream_t st) { EWS_PLANES_LAUNCH(k_summary); }
int planes_rows(const DiagArgs& a, hipStream_t st) {
  if (a.log) return 0;
  EWS_PLANES_LAUNCH(k_rows);
}
int planes_local(const DiagArgs& a, hipStream_t st) { EWS_PLANES_LAUNCH(k_local); }
int planes_full(const DiagArgs& a, hipStream_t st) { EWS_PLANES_LAUNCH(k_full); }

}  // namespace ews
