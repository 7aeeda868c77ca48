// Token-cached scan at depth 1 for cached flows of any width up to 64 (ews/core/token_scan.py:91-118 with trunc 1):
// S_t = D_{g_t} S_{t-1} + P_{g_t} from S = 0, a padded step keeping the state (D = I, P = 0). D_cache (V, d, d) is a
// dense flow per token, P_cache (V, d) the token's level 1.
//
// Forward: one wavefront per sample, lane i the state coordinate i; a step reads the token's transposed flow (a
// transposed copy made first, so that lane i reads D[g][i][j] for fixed j from consecutive addresses) against the
// previous state broadcast through LDS. Backward: one wavefront per sample walks the steps in reverse,
// lam_t = g_t + D_{t+1}^T lam_{t+1} (lane j reads row i of D[g] contiguously), and stores every step's cotangent;
// then per token dP_g = sum lam_t and dD_g = sum lam_t S_{t-1}^T over the steps carrying it, from the forward's rows
// (the states), in per-chunk partials reduced in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ews_hip.h"
#include "ews_lanes.h"

namespace ews {
namespace tok1 {

constexpr int kMaxD = 64;
constexpr int kChunk = 2048;  // steps per partial of the token gradients
constexpr int kStage = 16;    // steps staged in LDS at once

struct TArgs {
  int B, n, d, V;
  const int32_t* tokens;  // (B, n)
  const uint8_t* mask;    // (B, n) or null
  const float* P;         // (V, d)
  const float* D;         // (V, d, d)
  float* Dt;              // (V, d, d) transposed copy (workspace)
  float* out;             // (B, n, d)
  const float* rows;      // the forward's rows (backward)
  const float* gout;      // (B, n, d)
  float* lam;             // (B, n, d) cotangent of every step's state (workspace)
  float* part;            // (V, nch, d*d + d) per-chunk partials (workspace)
  int nch;
  float* gP;
  float* gD;
};

__device__ __forceinline__ int tok_at(const TArgs& a, size_t e, bool& live) {
  live = a.mask == nullptr || a.mask[e] != 0;
  const int g = a.tokens[e];
  return g < 0 ? 0 : (g >= a.V ? a.V - 1 : g);
}

__global__ void k_transpose(TArgs a) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t dd = (size_t)a.d * a.d;
  if (e >= (size_t)a.V * dd) return;
  const size_t g = e / dd, r = e % dd, i = r / a.d, j = r % a.d;
  a.Dt[g * dd + j * a.d + i] = a.D[e];
}

__global__ __launch_bounds__(64) void k_fwd(TArgs a) {
  __shared__ float s_x[kMaxD];
  const int b = blockIdx.x, i = threadIdx.x;
  const bool on = i < a.d;
  float S = 0.0f;
  for (int t = 0; t < a.n; ++t) {
    const size_t e = (size_t)b * a.n + t;
    bool live;
    const int g = tok_at(a, e, live);
    if (on) s_x[i] = S;
    __syncthreads();
    if (live && on) {
      const float* dt = a.Dt + (size_t)g * a.d * a.d + i;  // Dt[g][j][i] = D[g][i][j]
      float acc = a.P[(size_t)g * a.d + i];
      for (int j = 0; j < a.d; ++j) acc = fmaf(dt[(size_t)j * a.d], s_x[j], acc);
      S = acc;
    }
    if (on) a.out[e * a.d + i] = S;
    __syncthreads();  // s_x is rewritten by the next step
  }
}

__global__ __launch_bounds__(64) void k_bwd_lam(TArgs a) {
  __shared__ float s_l[kMaxD];
  const int b = blockIdx.x, j = threadIdx.x;
  const bool on = j < a.d;
  float lam = 0.0f;
  for (int t = a.n - 1; t >= 0; --t) {
    const size_t e = (size_t)b * a.n + t;
    if (on) {
      lam += a.gout[e * a.d + j];
      a.lam[e * a.d + j] = lam;
      s_l[j] = lam;
    }
    __syncthreads();
    bool live;
    const int g = tok_at(a, e, live);
    if (live && on) {  // lam_{t-1} carried = D_g^T lam_t: lane j takes column j (row i contiguous over lanes)
      const float* dg = a.D + (size_t)g * a.d * a.d + j;
      float acc = 0.0f;
      for (int i = 0; i < a.d; ++i) acc = fmaf(dg[(size_t)i * a.d], s_l[i], acc);
      lam = acc;
    }
    __syncthreads();
  }
}

// partials of token g over steps [c * kChunk, (c + 1) * kChunk) of the flattened (sample, step) order: each thread
// owns 16 entries of dD_g (d <= 64), threads < d also an entry of dP_g
__global__ __launch_bounds__(256) void k_grads(TArgs a) {
  __shared__ float s_l[kStage][kMaxD], s_s[kStage][kMaxD];
  __shared__ int s_use[kStage];
  const int g = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  const size_t tot = (size_t)a.B * a.n, e0 = (size_t)c * kChunk, e1 = min(tot, e0 + kChunk);
  const int dd = a.d * a.d;
  float acc[16], accp = 0.0f;
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.0f;
  for (size_t s0 = e0; s0 < e1; s0 += kStage) {
    // stage the block's steps that carry token g: their cotangents and the states before them
    for (int q = tid; q < kStage * kMaxD; q += 256) {
      const int r = q / kMaxD, col = q % kMaxD;
      const size_t e = s0 + r;
      bool use = false;
      if (e < e1) {
        bool live;
        use = tok_at(a, e, live) == g && live;
      }
      if (col == 0) s_use[r] = use;
      float lv = 0.0f, sv = 0.0f;
      if (use && col < a.d) {
        lv = a.lam[e * a.d + col];
        const size_t t = e % a.n;
        sv = t > 0 ? a.rows[(e - 1) * a.d + col] : 0.0f;  // S_{t-1} (zero before the first step)
      }
      s_l[r][col] = lv;
      s_s[r][col] = sv;
    }
    __syncthreads();
    for (int r = 0; r < kStage; ++r) {
      if (!s_use[r]) continue;  // uniform across the workgroup
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int q = tid + 256 * k;
        if (q < dd) acc[k] = fmaf(s_l[r][q / a.d], s_s[r][q % a.d], acc[k]);
      }
      if (tid < a.d) accp += s_l[r][tid];
    }
    __syncthreads();
  }
  float* out = a.part + ((size_t)g * a.nch + c) * (dd + a.d);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int q = tid + 256 * k;
    if (q < dd) out[q] = acc[k];
  }
  if (tid < a.d) out[dd + tid] = accp;
}

// the chunks' partials summed in order, float64
__global__ void k_reduce(TArgs a) {
  const int dd = a.d * a.d, W = dd + a.d;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)a.V * W) return;
  const size_t g = e / W, q = e % W;
  double s = 0.0;
  for (int c = 0; c < a.nch; ++c) s += (double)a.part[((size_t)g * a.nch + c) * W + q];
  if ((int)q < dd) a.gD[g * dd + q] = (float)s;
  else a.gP[g * a.d + (q - dd)] = (float)s;
}

// ---- block-diagonal caches (desc->block = BS): the flow of every token is block-diagonal with blocks of BS
// consecutive coordinates (the chain-structured caches: rotation planes BS = 2, Jordan chains BS = their size, a
// real diagonal BS = 1). Lane i then needs only row i of its block: S_i = P_g[i] + sum_r D_g[i][base + r] S_{base+r}
// (base = BS floor(i / BS)), with the block partners' states by lane shuffles: no LDS broadcast, no barrier. The
// caches' block entries are staged in LDS when they fit (row i of token g's block at (g d + i) BS), the step's token
// and mask bit come from a register holding the next 64 steps. The backward walks the steps in reverse with the
// cotangent lam_{t-1} = D_g^T lam_t (+ the row cotangent), and accumulates the token gradients per lane in LDS
// (lane i owns dP_g[i] and row i of dD_g's block): per-sample partials, then a fixed-order sum over the samples.
// Entries of D outside the blocks are taken as zero and their gradients are written as zero.
//
// A sample's steps are one dependent chain, and one wavefront per sample leaves most of the chip idle, so the NW
// wavefronts of a sample's workgroup take one span of steps each: first the span's affine map of the state (its effect
// from zero, and on the BS unit states of a block, all BS + 1 chains side by side in registers, in float64: the spans'
// start states are then more exact than the float32 chain's), then, the maps of the spans before it applied in order,
// the span again from its own start state with the rows written. The adjoint does the
// same from the last span, with the transposed flows, before the sweep that accumulates the gradients. (BS + 2) / NW of
// the steps are on the chain for 1. B = 256 x 512 tokens, d = 64, BS = 2: forward 50 -> 28 us, backward 110 -> 39 us at
// NW = 8. Blocks of 6 and 8, whose lane exchanges go through LDS, keep NW = 1, a constant for them: with the span and the
// LDS offsets from the launch's size their kernels took a quarter longer than without spans at all (1 x 1000 tokens, blocks
// of 6: 163 and 371 us; 130 and 263 as constants). The new state is a select: as a branch around each step it held back the
// loads of the steps after it.
constexpr int kStageFloats = 12288;  // caches staged in LDS up to 48 KB
template <int BS> constexpr bool kSpans = BS <= 4;  // block sizes whose samples are split into spans

template <bool STAGED>
__device__ __forceinline__ float blk_d(const TArgs& a, const float* sD, int BS, int g, int row, int r) {
  if constexpr (STAGED) return sD[((size_t)g * a.d + row) * BS + r];
  return a.D[((size_t)g * a.d + row) * a.d + (row / BS) * BS + r];
}

// v of lane base + r, the r-th lane of this lane's block (base = BS floor(lane / BS)); every lane of the wavefront
// takes part. Blocks of 2 and 4 lie inside a quad of lanes: one DPP quad permutation (a VALU operand, no memory
// round trip); blocks of 3, 6 and 8 go through an LDS permute.
template <int BS, class T>
__device__ __forceinline__ T blk_lane(T v, int base, int r) {
  if constexpr (BS == 1) {
    return v;
  } else if constexpr (BS == 2) {
    return r == 0 ? lanes::dpp<0xA0>(v) : lanes::dpp<0xF5>(v);  // quad_perm [0, 0, 2, 2], [1, 1, 3, 3]
  } else if constexpr (BS == 4) {
    switch (r) {  // quad_perm [r, r, r, r]
      case 0: return lanes::dpp<0x00>(v);
      case 1: return lanes::dpp<0x55>(v);
      case 2: return lanes::dpp<0xAA>(v);
      default: return lanes::dpp<0xFF>(v);
    }
  } else {
    return __shfl(v, base + r);
  }
}

// the block caches into LDS (row i of token g's block at (g d + i) BS, then P), eight loads in flight per lane
template <int BS>
__device__ __forceinline__ void stage_blk(const TArgs& a, float* sP, float* sD, bool with_p) {
  const int nd = a.V * a.d * BS, i = threadIdx.x, nt = blockDim.x;
  for (int q0 = i; q0 < nd; q0 += 8 * nt) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = min(q0 + nt * u, nd - 1);  // clamped: every load unconditional
      const int gr = q / BS, r = q - gr * BS, g = gr / a.d, row = gr - g * a.d;
      v[u] = a.D[((size_t)g * a.d + row) * a.d + (row / BS) * BS + r];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (q0 + nt * u < nd) sD[q0 + nt * u] = v[u];
    }
  }
  if (with_p) {
    const int np = a.V * a.d;
    for (int q0 = i; q0 < np; q0 += 8 * nt) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = a.P[min(q0 + nt * u, np - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (q0 + nt * u < np) sP[q0 + nt * u] = v[u];
      }
    }
  }
}

// The spans: wavefront w of NW takes steps [w span, (w + 1) span), whole groups of eight.
__device__ __forceinline__ int span_len(const TArgs& a, int nw) { return ((a.n + nw - 1) / nw + 7) / 8 * 8; }
// x + sum_c U[c] y_{base + c}: a span's map applied to the state (cotangent) y of the lane's block. A zero of y adds
// nothing (the map of a span of growing flows may have overflowed).
template <int BS>
__device__ __forceinline__ double span_apply(double x, const double* U, int stride, double y, int base) {
#pragma unroll
  for (int c = 0; c < BS; ++c) {
    const double yc = blk_lane<BS>(y, base, c);
    x = yc != 0.0 ? fma(U[c * stride], yc, x) : x;
  }
  return x;
}
template <bool MAP> using span_t = std::conditional_t<MAP, double, float>;

// The step loops take the caches from LDS (STAGED) or from global memory, a compile-time choice: one load kind each.
// MAP: the span's map instead of its rows: S from zero and U[c], the states from the units of the lane's block.
template <int BS, bool STAGED, bool MAP>
__device__ __forceinline__ void fwd_blk_steps(const TArgs& a, const float* sP, const float* sD, int b, int i, int tb,
                                              int te, span_t<MAP>& S, span_t<MAP>* U) {
  using T = span_t<MAP>;
  const bool on = i < a.d;
  const int base = (i / BS) * BS;
  const int row = on ? i : 0;  // lanes past d read row 0 and keep S = 0
  for (int t0 = tb; t0 < te; t0 += 64) {
    int tokv = 0, livev = 0;
    if (t0 + i < te) {
      bool live;
      tokv = tok_at(a, (size_t)b * a.n + t0 + i, live);
      livev = live ? 1 : 0;
    }
    const int cnt = min(64, te - t0);
    // groups of eight steps without a branch (the lane reads are convergent, so only a constant trip count is
    // unrolled; the states are stored after the group), so that the group's cache reads are issued ahead of the
    // state chain; steps past the span carry token 0 and no mask bit
    for (int s0 = 0; s0 < (kSpans<BS> ? cnt : 64); s0 += 8) {
      float Sv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int g = __builtin_amdgcn_readlane(tokv, s0 + u), live = __builtin_amdgcn_readlane(livev, s0 + u);
        T acc = STAGED ? sP[g * a.d + row] : a.P[(size_t)g * a.d + row];
        T dr[BS];
#pragma unroll
        for (int r = 0; r < BS; ++r) dr[r] = blk_d<STAGED>(a, sD, BS, g, row, r);
#pragma unroll
        for (int r = 0; r < BS; ++r) acc = fma(dr[r], blk_lane<BS>(S, base, r), acc);
        if constexpr (MAP) {
#pragma unroll
          for (int c = 0; c < BS; ++c) {
            T ua = 0;
#pragma unroll
            for (int r = 0; r < BS; ++r) ua = fma(dr[r], blk_lane<BS>(U[c], base, r), ua);
            if (live) U[c] = ua;
          }
        }
        S = live && on ? acc : S;
        Sv[u] = (float)S;
      }
      if (!MAP && on) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (s0 + u < cnt) a.out[((size_t)b * a.n + t0 + s0 + u) * a.d + i] = Sv[u];
        }
      }
    }
  }
}

template <int BS, bool STAGED>
__device__ __forceinline__ void fwd_blk_body(const TArgs& a, const float* sP, const float* sD, double* sX) {
  const int b = blockIdx.x, i = threadIdx.x & 63;
  const int w = kSpans<BS> ? threadIdx.x >> 6 : 0, nw = kSpans<BS> ? (int)(blockDim.x >> 6) : 1;
  const int span = kSpans<BS> ? span_len(a, nw) : a.n, tb = kSpans<BS> ? min(a.n, w * span) : 0;
  const int te = min(a.n, tb + span), base = (i / BS) * BS;
  double S = 0.0;
  if constexpr (kSpans<BS>) {
    if (nw > 1) {
      double U[BS];
      if (w + 1 < nw) {
#pragma unroll
        for (int c = 0; c < BS; ++c) U[c] = i - base == c ? 1.0 : 0.0;
        fwd_blk_steps<BS, STAGED, true>(a, sP, sD, b, i, tb, te, S, U);
        double* x = sX + (size_t)w * (BS + 1) * 64 + i;
#pragma unroll
        for (int c = 0; c < BS; ++c) x[c * 64] = U[c];
        x[BS * 64] = S;
      }
      __syncthreads();
      S = 0.0;
      for (int u = 0; u < w; ++u) {
        const double* x = sX + (size_t)u * (BS + 1) * 64 + i;
        S = span_apply<BS>(x[BS * 64], x, 64, S, base);
      }
    }
  }
  float S0 = (float)S;
  fwd_blk_steps<BS, STAGED, false>(a, sP, sD, b, i, tb, te, S0, nullptr);
}

template <int BS>
__global__ __launch_bounds__(512) void k_fwd_blk(TArgs a) {
  extern __shared__ double s_c[];
  double* sX = s_c;  // (NW, BS + 1, 64): the spans' maps
  float* sP = reinterpret_cast<float*>(sX + (size_t)(kSpans<BS> ? blockDim.x >> 6 : 1) * (BS + 1) * 64);
  float* sD = sP + (size_t)a.V * a.d;
  if ((size_t)a.V * a.d * (BS + 1) <= (size_t)kStageFloats) {
    stage_blk<BS>(a, sP, sD, true);
    __syncthreads();
    fwd_blk_body<BS, true>(a, sP, sD, sX);
  } else {
    fwd_blk_body<BS, false>(a, sP, sD, sX);
  }
}

// kStage steps' row cotangents (and, ROWS, the states before them) from step u1 - 1 down: lane i's column, loads
// unconditional from clamped addresses and zeroed afterwards
template <bool ROWS>
__device__ __forceinline__ void load_stage(const TArgs& a, int b, int ic, int tb, int u1, float* gv, float* rv) {
#pragma unroll
  for (int k = 0; k < kStage; ++k) {
    const int t = max(u1 - 1 - k, tb);
    gv[k] = a.gout[((size_t)b * a.n + t) * a.d + ic];
    if (ROWS) rv[k] = a.rows[((size_t)b * a.n + max(t - 1, 0)) * a.d + ic];  // S_{t-1}
  }
}

// MAP: the span's adjoint map: lam from zero at its end and U[c] from the unit cotangents; else the sweep from lam at
// the span's end, the token gradients added to sAcc.
template <int BS, bool STAGED, bool MAP>
__device__ __forceinline__ void bwd_blk_steps(const TArgs& a, const float* sD, float* sAcc, int b, int i, int tb, int te,
                                              span_t<MAP>& lam, span_t<MAP>* U) {
  using T = span_t<MAP>;
  const bool on = i < a.d;
  const int base = (i / BS) * BS;
  // lanes past d read block row 0 (their products are dropped); their lam, state and accumulators stay zero
  const int rowb = on ? base : 0, col = on ? i - base : 0, ic = on ? i : 0;
  if (tb >= te) return;
  float gv[kStage], rv[kStage], gn[kStage], rn[kStage];
  load_stage<!MAP>(a, b, ic, tb, te, gn, rn);
  for (int t1 = te; t1 > tb; t1 -= 64) {
    const int t0 = max(tb, t1 - 64);
    int tokv = 0, livev = 0;  // lane l: step t1 - 1 - l
    if (t1 - 1 - i >= t0) {
      bool live;
      tokv = tok_at(a, (size_t)b * a.n + t1 - 1 - i, live);
      livev = live ? 1 : 0;
    }
    for (int q0 = 0; q0 < t1 - t0; q0 += kStage) {
      const int u1 = t1 - q0;
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        gv[k] = gn[k];
        if (!MAP) rv[k] = rn[k];
      }
      load_stage<!MAP>(a, b, ic, tb, max(u1 - kStage, tb + 1), gn, rn);  // the next stage's, in flight meanwhile
      // unrolled and without a branch (see the forward): a step before the span or without its mask bit adds zero to
      // the accumulators (exact: they start at +0 and never become -0) and keeps lam
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        const int t = u1 - 1 - k;
        const bool in = t >= t0;
        // uniform over the wavefront: the step's token and mask bit from lane t1 - 1 - t
        const int g = __builtin_amdgcn_readlane(tokv, q0 + k);
        const bool live = __builtin_amdgcn_readlane(livev, q0 + k) && in;
        lam += on && in ? gv[k] : 0.0f;
        T dc[BS], ln = 0;
#pragma unroll
        for (int r = 0; r < BS; ++r) dc[r] = blk_d<STAGED>(a, sD, BS, g, rowb + r, col);
        if constexpr (MAP) {
#pragma unroll
          for (int c = 0; c < BS; ++c) {
            T ua = 0;
#pragma unroll
            for (int r = 0; r < BS; ++r) ua = fma(dc[r], blk_lane<BS>(U[c], base, r), ua);
            if (live) U[c] = ua;
          }
#pragma unroll
          for (int r = 0; r < BS; ++r) ln = fma(dc[r], blk_lane<BS>(lam, base, r), ln);
        } else {
          const float sp = on && in && t > 0 ? rv[k] : 0.0f;
          const float lw = live ? lam : 0.0f;
          float* acc = sAcc + (size_t)g * (BS + 1) * 64 + i;
#pragma unroll
          for (int r = 0; r < BS; ++r) {
            const float s_r = blk_lane<BS>(sp, base, r), l_r = blk_lane<BS>(lam, base, r);
            acc[r * 64] += lw * s_r;        // dD_g[i][base + r]
            ln = fmaf(dc[r], l_r, ln);      // (D_g^T lam)_i
          }
          acc[BS * 64] += lw;  // dP_g[i]
        }
        lam = live ? (on ? ln : (T)0) : lam;
      }
    }
  }
}

template <int BS, bool STAGED>
__device__ __forceinline__ void bwd_blk_body(const TArgs& a, const float* sD, float* sAcc, double* sX) {
  const int b = blockIdx.x, i = threadIdx.x & 63;
  const int w = kSpans<BS> ? threadIdx.x >> 6 : 0, nw = kSpans<BS> ? (int)(blockDim.x >> 6) : 1;
  const int span = kSpans<BS> ? span_len(a, nw) : a.n, tb = kSpans<BS> ? min(a.n, w * span) : 0;
  const int te = min(a.n, tb + span), base = (i / BS) * BS;
  double lam = 0.0;
  if constexpr (kSpans<BS>) {
    if (nw > 1) {
      double U[BS];
      if (w > 0) {
#pragma unroll
        for (int c = 0; c < BS; ++c) U[c] = i - base == c ? 1.0 : 0.0;
        bwd_blk_steps<BS, STAGED, true>(a, sD, nullptr, b, i, tb, te, lam, U);
        double* x = sX + (size_t)w * (BS + 1) * 64 + i;
#pragma unroll
        for (int c = 0; c < BS; ++c) x[c * 64] = U[c];
        x[BS * 64] = lam;
      }
      __syncthreads();
      lam = 0.0;
      for (int u = nw - 1; u > w; --u) {
        const double* x = sX + (size_t)u * (BS + 1) * 64 + i;
        lam = span_apply<BS>(x[BS * 64], x, 64, lam, base);
      }
    }
  }
  float lam0 = (float)lam;
  bwd_blk_steps<BS, STAGED, false>(a, sD, sAcc + (size_t)w * a.V * (BS + 1) * 64, b, i, tb, te, lam0, nullptr);
}

template <int BS>
__global__ __launch_bounds__(512) void k_bwd_blk(TArgs a) {
  extern __shared__ double s_c[];
  const int b = blockIdx.x, i = threadIdx.x & 63;
  const int w = kSpans<BS> ? threadIdx.x >> 6 : 0, nw = kSpans<BS> ? (int)(blockDim.x >> 6) : 1;
  const bool staged = (size_t)a.V * a.d * (BS + 1) <= (size_t)kStageFloats;
  const int na = a.V * (BS + 1);
  double* sX = s_c;  // (NW, BS + 1, 64): the spans' maps
  float* sAcc = reinterpret_cast<float*>(sX + (size_t)nw * (BS + 1) * 64);  // (NW, V, BS + 1, 64): lane i's column
  float* sD = sAcc + (size_t)nw * na * 64;
  if (staged) stage_blk<BS>(a, nullptr, sD, false);
  for (int q = 0; q < na; ++q) sAcc[((size_t)w * na + q) * 64 + i] = 0.0f;
  __syncthreads();
  if (staged) bwd_blk_body<BS, true>(a, sD, sAcc, sX);
  else bwd_blk_body<BS, false>(a, sD, sAcc, sX);
  __syncthreads();
  if (i < a.d) {  // the sample's partial: its spans in order
    for (int q = w; q < na; q += nw) {
      double s = 0.0;
      for (int u = 0; u < nw; ++u) s += (double)sAcc[((size_t)u * na + q) * 64 + i];
      a.part[((size_t)b * na + q) * a.d + i] = (float)s;
    }
  }
}

// gP and gD from the per-sample partials, in float64: 16 threads per entry sum a run of samples each, eight loads in
// flight, and thread 0 adds the runs in order (one thread per entry took 16 us at 256 samples). The workgroups past the
// entries write gD's zeros outside the blocks.
constexpr int kRedEnt = 16, kRedRun = 16;
__global__ __launch_bounds__(kRedEnt* kRedRun) void k_reduce_blk(TArgs a, int BS, int nent_wg) {
  __shared__ double red[kRedRun][kRedEnt];
  const size_t dd = (size_t)a.d * a.d;
  if ((int)blockIdx.x >= nent_wg) {
    const size_t e = (size_t)(blockIdx.x - nent_wg) * blockDim.x + threadIdx.x;
    if (e >= (size_t)a.V * dd) return;
    const int rc = (int)(e % dd);
    if (rc / a.d / BS != rc % a.d / BS) a.gD[e] = 0.0f;
    return;
  }
  const int x = threadIdx.x % kRedEnt, y = threadIdx.x / kRedEnt;
  const size_t nent = (size_t)a.V * (BS + 1) * a.d, off = (size_t)blockIdx.x * kRedEnt + x;
  const int per = (a.B + kRedRun - 1) / kRedRun, b1 = min(a.B, (y + 1) * per);
  double s = 0.0;
  if (off < nent) {
    int b = y * per;
    for (; b + 8 <= b1; b += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = a.part[(size_t)(b + u) * nent + off];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += (double)v[u];
    }
    for (; b < b1; ++b) s += (double)a.part[(size_t)b * nent + off];
  }
  red[y][x] = s;
  __syncthreads();
  if (y > 0 || off >= nent) return;
  for (int u = 1; u < kRedRun; ++u) s += red[u][x];
  const int i = (int)(off % a.d), q = (int)(off / a.d), g = q / (BS + 1), r = q % (BS + 1);
  if (r == BS) a.gP[(size_t)g * a.d + i] = (float)s;
  else a.gD[((size_t)g * a.d + i) * a.d + (i / BS) * BS + r] = (float)s;
}

}  // namespace tok1

namespace {
int tok1_check(const ews_token1_desc* s) {
  if (!s) return EWS_ERR_NULL;
  if (s->batch < 1 || s->steps < 1 || s->dim < 1 || s->dim > tok1::kMaxD || s->vocab < 1) return EWS_ERR_SHAPE;
  const int bs = s->block;
  if (bs < 0 || bs > 8 || bs == 5 || bs == 7 || (bs > 0 && s->dim % bs != 0)) return EWS_ERR_OPTION;
  // the backward's per-lane accumulators (16 KB per wavefront at most) sit in LDS beside the staged caches (48 KB at
  // most)
  if (bs > 0 && (size_t)s->vocab * (bs + 1) > 64) return EWS_ERR_SHAPE;
  return EWS_OK;
}
// Wavefronts per sample (spans of its steps): eight while that stays under 4096 wavefronts, at least 32 steps each, and
// while their accumulators fit the LDS; one for blocks of 6 and 8.
size_t blk_lds_bytes(const ews_token1_desc* s, int nw, bool bwd) {
  const size_t stage = (size_t)s->vocab * s->dim * (s->block + 1);
  const size_t staged = stage <= (size_t)tok1::kStageFloats ? stage : 0;
  const size_t maps = (size_t)nw * (s->block + 1) * 64;
  return (staged + 2 * maps + (bwd ? maps * s->vocab : 0)) * 4;
}
int blk_waves(const ews_token1_desc* s) {
  int nw = s->block <= 4 ? 8 : 1;  // kSpans
  while (nw > 1 && ((long)s->batch * nw > 4096 || s->steps < 32 * nw || blk_lds_bytes(s, nw, true) > 160 * 1024)) nw /= 2;
  return nw;
}
// launch of a block-diagonal kernel for the descriptor's block size
template <class K>
int blk_launch(K* kern, const ews_token1_desc* s, bool bwd, hipStream_t st, const tok1::TArgs& a) {
  const int nw = blk_waves(s);
  const size_t lds = blk_lds_bytes(s, nw, bwd);
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return EWS_ERR_LAUNCH;
  hipLaunchKernelGGL(kern, dim3(a.B), dim3(64 * nw), lds, st, a);
  return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
}
#define EWS_TOK1_BLK(KERNEL, S, BWD, ST, A)                                         \
  ((S)->block == 1   ? blk_launch(&KERNEL<1>, S, BWD, ST, A)                        \
   : (S)->block == 2 ? blk_launch(&KERNEL<2>, S, BWD, ST, A)                        \
   : (S)->block == 3 ? blk_launch(&KERNEL<3>, S, BWD, ST, A)                        \
   : (S)->block == 4 ? blk_launch(&KERNEL<4>, S, BWD, ST, A)                        \
   : (S)->block == 6 ? blk_launch(&KERNEL<6>, S, BWD, ST, A)                        \
                     : blk_launch(&KERNEL<8>, S, BWD, ST, A))
size_t al256t(size_t x) { return (x + 255) & ~(size_t)255; }
tok1::TArgs tok1_args(const ews_token1_desc* s) {
  tok1::TArgs a{};
  a.B = s->batch;
  a.n = s->steps;
  a.d = s->dim;
  a.V = s->vocab;
  a.nch = (int)(((size_t)a.B * a.n + tok1::kChunk - 1) / tok1::kChunk);
  return a;
}
}  // namespace
}  // namespace ews

extern "C" {

size_t ews_token1_workspace_bytes(const ews_token1_desc* desc) {
  if (ews::tok1_check(desc) != EWS_OK) return 0;
  const ews::tok1::TArgs a = ews::tok1_args(desc);
  if (desc->block > 0) return ews::al256t((size_t)a.B * a.V * (desc->block + 1) * a.d * 4);  // per-sample partials
  const size_t dd = (size_t)a.d * a.d;
  return ews::al256t((size_t)a.V * dd * 4) + ews::al256t((size_t)a.B * a.n * a.d * 4) +
         ews::al256t((size_t)a.V * a.nch * (dd + a.d) * 4);
}

int ews_token1_scan(const ews_token1_desc* desc, const int32_t* tokens, const uint8_t* mask, const float* P_cache,
                    const float* D_cache, float* out, void* workspace, ews_stream_t stream) {
  const int rc = ews::tok1_check(desc);
  if (rc != EWS_OK) return rc;
  if (!tokens || !P_cache || !D_cache || !out || !workspace) return EWS_ERR_NULL;
  ews::tok1::TArgs a = ews::tok1_args(desc);
  a.tokens = tokens;
  a.mask = mask;
  a.P = P_cache;
  a.D = D_cache;
  a.Dt = (float*)workspace;
  a.out = out;
  hipStream_t st = (hipStream_t)stream;
  if (desc->block > 0) {
    using ews::blk_launch;
    return EWS_TOK1_BLK(ews::tok1::k_fwd_blk, desc, false, st, a);
  }
  const size_t nd = (size_t)a.V * a.d * a.d;
  hipLaunchKernelGGL(ews::tok1::k_transpose, dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, st, a);
  if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;
  hipLaunchKernelGGL(ews::tok1::k_fwd, dim3(a.B), dim3(64), 0, st, a);
  return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
}

int ews_token1_scan_backward(const ews_token1_desc* desc, const int32_t* tokens, const uint8_t* mask,
                             const float* P_cache, const float* D_cache, const float* out, const float* grad_out,
                             float* grad_P, float* grad_D, void* workspace, ews_stream_t stream) {
  const int rc = ews::tok1_check(desc);
  if (rc != EWS_OK) return rc;
  if (!tokens || !P_cache || !D_cache || !out || !grad_out || !grad_P || !grad_D || !workspace) return EWS_ERR_NULL;
  ews::tok1::TArgs a = ews::tok1_args(desc);
  a.tokens = tokens;
  a.mask = mask;
  a.P = P_cache;
  a.D = D_cache;
  a.rows = out;
  a.gout = grad_out;
  a.gP = grad_P;
  a.gD = grad_D;
  const size_t dd = (size_t)a.d * a.d;
  hipStream_t st = (hipStream_t)stream;
  if (desc->block > 0) {
    a.part = (float*)workspace;
    using ews::blk_launch;
    const int brc = EWS_TOK1_BLK(ews::tok1::k_bwd_blk, desc, true, st, a);
    if (brc != EWS_OK) return brc;
    constexpr int rt = ews::tok1::kRedEnt * ews::tok1::kRedRun;
    const int ne = (int)(((size_t)a.V * (desc->block + 1) * a.d + ews::tok1::kRedEnt - 1) / ews::tok1::kRedEnt);
    const int nz = (int)(((size_t)a.V * dd + rt - 1) / rt);
    hipLaunchKernelGGL(ews::tok1::k_reduce_blk, dim3(ne + nz), dim3(rt), 0, st, a, desc->block, ne);
    return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
  }
  char* w = (char*)workspace;
  a.lam = (float*)(w + ews::al256t((size_t)a.V * dd * 4));
  a.part = (float*)(w + ews::al256t((size_t)a.V * dd * 4) + ews::al256t((size_t)a.B * a.n * a.d * 4));
  hipLaunchKernelGGL(ews::tok1::k_bwd_lam, dim3(a.B), dim3(64), 0, st, a);
  if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;
  hipLaunchKernelGGL(ews::tok1::k_grads, dim3(a.V, a.nch), dim3(256), 0, st, a);
  if (hipGetLastError() != hipSuccess) return EWS_ERR_LAUNCH;
  const size_t W = (size_t)a.V * (dd + a.d);
  hipLaunchKernelGGL(ews::tok1::k_reduce, dim3((unsigned)((W + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? EWS_OK : EWS_ERR_LAUNCH;
}

}  // extern "C"
