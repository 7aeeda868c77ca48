// Host build of the small-step polynomials (csrc/ews_numerics.h) for CPU tests.
#include "ews_numerics.h"

using ews::cf;

extern "C" {
int shim_degrees(int which) { return which == 0 ? ews::kPolyPhi : ews::kPolyD; }
float shim_radius() { return ews::kPolyR; }
int shim_small(float umax, float hmax) { return ews::poly_small(umax, hmax); }
float shim_max(int which) { return which == 0 ? ews::kPolyMaxU : ews::kPolyMaxH; }
// phi(h u), its d/dh, exp[0, h u, h v] and its d/dh: out n x 8 (re, im)
void shim_poly(int n, const float* h, const float* u, const float* v, float* out) {
  for (int i = 0; i < n; ++i) {
    const cf uu{u[2 * i], u[2 * i + 1]}, vv{v[2 * i], v[2 * i + 1]};
    cf cp[ews::kPolyPhi + 1], cd[ews::kPolyD + 1], dp, dd;
    ews::poly_phi(uu, cp);
    ews::poly_dd3(uu, vv, cd);
    const cf p = ews::poly_val_d<ews::kPolyPhi>(cp, h[i], dp), d = ews::poly_val_d<ews::kPolyD>(cd, h[i], dd);
    const float r[8] = {p.re, p.im, dp.re, dp.im, d.re, d.im, dd.re, dd.im};
    for (int j = 0; j < 8; ++j) out[8 * i + j] = r[j];
  }
}
// node cotangents of the steps (h_i, g_i) under one (u, v) through the moments, out (phi, x, y): 6 floats
void shim_moments(int n, const float* h, const float* g, const float* u, const float* v, float* out) {
  cf mp[ews::kPolyPhi] = {}, md[ews::kPolyD] = {}, gx, gy;
  for (int i = 0; i < n; ++i) {
    float p = h[i];
    for (int m = 0; m < ews::kPolyD; ++m) {
      const cf gi{g[2 * i], g[2 * i + 1]};
      if (m < ews::kPolyPhi) mp[m] = ews::fma_r(p, gi, mp[m]);
      md[m] = ews::fma_r(p, gi, md[m]);
      p *= h[i];
    }
  }
  const cf uu{u[0], u[1]}, vv{v[0], v[1]}, gp = ews::poly_phi_node(uu, mp);
  ews::poly_dd3_node(uu, vv, md, gx, gy);
  const float r[6] = {gp.re, gp.im, gx.re, gx.im, gy.re, gy.im};
  for (int j = 0; j < 6; ++j) out[j] = r[j];
}
}
