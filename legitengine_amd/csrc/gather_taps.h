// The taps of the gather's trilinear sampler.  Arithmetic only, host and
// device (tests/csrc/check_taps.cpp calls it on the CPU): no HIP header.
#pragma once
#include <math.h>

#ifndef LGX_HD  // included by host code alone
#define LGX_HD inline
#endif

namespace lgx {

// Vulkan clamp-to-edge bilinear taps of a point s in one level: u = s W - 1/2,
// taps floor(u) and the next, each clamped, weights frac(u), and the blends'
// products and sums rounded one by one.  Nothing here may round otherwise: the
// depths of a flat surface tie the horizon test of :254, and another last bit
// is another set of hits (a fused blend: 1 to 18 % of the hit counts; pairs
// of neighbours with saturating weights, one fetch for two texels, are also
// wrong beside a far or infinite texel at a border).
template <class T> struct TapPos {
  T al, be;
  int x0, x1, y0, y1;
  LGX_HD TapPos(T sx, T sy, int lw, int lh) {
    const T u = sx * T(lw) - T(0.5), v = sy * T(lh) - T(0.5);
    const T fu = floor(u), fv = floor(v);
    al = u - fu;
    be = v - fv;
    const int i = (int)fu, j = (int)fv;
    x0 = clamp(i, lw);
    x1 = clamp(i + 1, lw);
    y0 = clamp(j, lh);
    y1 = clamp(j + 1, lh);
  }
  LGX_HD T mix(T p00, T p10, T p01, T p11) const {
    const T top = lerp(al, p00, p10), bot = lerp(al, p01, p11);
    return lerp(be, top, bot);
  }
  static LGX_HD T lerp(T w, T a, T b) { return a * (T(1) - w) + b * w; }

 private:
  static LGX_HD int clamp(int k, int n) {
    const int lo = k < 0 ? 0 : k;
    return lo > n - 1 ? n - 1 : lo;
  }
};

}  // namespace lgx
