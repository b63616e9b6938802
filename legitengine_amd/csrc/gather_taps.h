// The taps of the gather's trilinear sampler.  Arithmetic only, host and
// device (tests/csrc/check_taps.cpp calls it on the CPU): no HIP header.
#pragma once
#include <math.h>

#ifndef LGX_HD  // included by host code alone
#define LGX_HD inline
#endif

namespace lgx {

// The four texels of a pair of neighbouring columns and rows (both the same
// one in a level of one column or row).
template <class T> struct Quad {
  T p00, p10, p01, p11;
};

// Vulkan clamp-to-edge bilinear taps of a point s in one level (u = s W -
// 1/2, taps floor(u) and the next, weights frac(u)).  At a border, where both
// taps are the edge texel, the pair is moved inside and the weight saturates,
// so the two texels of a row are always neighbours and come in one fetch.
template <class T> struct TapPos {
  T al, be;
  int x, y;
  LGX_HD TapPos(T sx, T sy, int lw, int lh) {
    const T u = sx * T(lw) - T(0.5), v = sy * T(lh) - T(0.5);
    const T fu = fmax(fmin(floor(u), T(lw - 2)), T(0)), fv = fmax(fmin(floor(v), T(lh - 2)), T(0));
    al = fmin(fmax(u - fu, T(0)), T(1));
    be = fmin(fmax(v - fv, T(0)), T(1));
    x = (int)fu;
    y = (int)fv;
  }
  // a (1 - w) + b w: exact at w = 0 and w = 1 for finite a and b, where
  // a + w (b - a) rounds at the size of the texel that does not count
  static LGX_HD T lerp(T w, T a, T b) { return fma(w, b, fma(-w, a, a)); }
  LGX_HD T mix(const Quad<T> &q) const { return lerp(be, lerp(al, q.p00, q.p10), lerp(al, q.p01, q.p11)); }
};

// The same texels with the taps clamped one by one and the weights as the
// shader's sampler has them: what an infinite texel, which a saturated weight
// does not take out, is sampled with.
template <class T> LGX_HD T clamped_taps(T sx, T sy, int lw, int lh, const Quad<T> &q) {
  const T u = sx * T(lw) - T(0.5), v = sy * T(lh) - T(0.5);
  const T fu = floor(u), fv = floor(v), al = u - fu, be = v - fv;
  const bool r0 = fu >= T(lw - 1), r1 = fu >= T(0), b0 = fv >= T(lh - 1), b1 = fv >= T(0);
  const T p00 = b0 ? (r0 ? q.p11 : q.p01) : (r0 ? q.p10 : q.p00), p10 = b0 ? (r1 ? q.p11 : q.p01) : (r1 ? q.p10 : q.p00);
  const T p01 = b1 ? (r0 ? q.p11 : q.p01) : (r0 ? q.p10 : q.p00), p11 = b1 ? (r1 ? q.p11 : q.p01) : (r1 ? q.p10 : q.p00);
  const T top = p00 * (T(1) - al) + p10 * al, bot = p01 * (T(1) - al) + p11 * al;
  return top * (T(1) - be) + bot * be;
}

template <class T> LGX_HD bool finite_tap(T r) { return fabs(r) < T(INFINITY); }

}  // namespace lgx
