// The traversal's slab test (gi_internal.h) on the host: an empty slot is
// never hit, whatever the direction's signs and the ray's limit; a box at a
// finite distance within the limit always is.
#include <cfloat>
#include <cmath>
#include <cstdio>

#include "../../globillum_amd/csrc/gi_internal.h"

using namespace gi;

// The near and the far plane of an axis by the direction's sign, as the
// kernels take them.
static bool hit(const WideNode &nd, int k, const float o[3], const float inv[3], float lim) {
  const float *lo[3] = {nd.lox, nd.loy, nd.loz}, *hi[3] = {nd.hix, nd.hiy, nd.hiz};
  float tn = 0.0f, tf = slab_limit(lim);
  for (int a = 0; a < 3; ++a) {
    const float b = -(o[a] * inv[a]);
    const float l = std::fmaf(lo[a][k], inv[a], b), h = std::fmaf(hi[a][k], inv[a], b);
    tn = std::fmax(tn, inv[a] < 0 ? h : l);
    tf = std::fmin(tf, inv[a] < 0 ? l : h);
  }
  return slab_hit(tn, tf);
}

int main() {
  const float limits[] = {INFINITY, NAN,   FLT_MAX, std::nextafterf(FLT_MAX, 0.f), kMaxLim, std::nextafterf(kMaxLim, 0.f),
                          1e30f,    1.0f, 0.0f,    -1.0f,                         -FLT_MAX, -INFINITY};
  int checks = 0, bad = 0;
  for (int s = 0; s < 8; ++s)
    for (float lim : limits)
      for (float scale : {1e-30f, 1e-3f, 1.0f, 1e30f})
        for (float at : {0.0f, -7.5f, 1e4f}) {
          const float o[3] = {at, 0.5f * at, -at};
          const float inv[3] = {s & 1 ? -scale : scale, s & 2 ? -2 * scale : 2 * scale, s & 4 ? -3 * scale : 3 * scale};
          WideNode nd;
          set_empty_slot(nd, 2);
          ++checks;
          if (hit(nd, 2, o, inv, lim)) ++bad, std::printf("empty slot hit: signs %d lim %g scale %g\n", s, lim, scale);
        }
  // a slab entered at t = FLT_MAX exactly, or nearer, along +x from 0
  for (float t : {FLT_MAX, std::nextafterf(FLT_MAX, 0.f), kMaxLim, 1e20f, 1.0f, 0.0f})
    for (float lim : limits) {
      WideNode nd;
      nd.lox[0] = t, nd.hix[0] = INFINITY, nd.loy[0] = nd.loz[0] = -1.0f, nd.hiy[0] = nd.hiz[0] = 1.0f;
      const float o[3] = {0, 0, 0}, inv[3] = {1.0f, FLT_MAX, FLT_MAX};
      const bool within = std::isnan(lim) || lim >= t;
      ++checks;
      if (within && !hit(nd, 0, o, inv, lim)) ++bad, std::printf("box at %g missed: lim %g\n", t, lim);
    }
  std::printf("%d checks, %d bad\n", checks, bad);
  return bad != 0;
}
