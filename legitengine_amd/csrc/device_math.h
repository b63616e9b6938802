// Arithmetic shared by the device kernels (HIP sources only).
#pragma once
#include <math.h>

#include "lgx_internal.h"

namespace lgx {

template <class T> LGX_D T fast_rsqrt(T v);
template <> LGX_D float fast_rsqrt<float>(float v) { return __builtin_amdgcn_rsqf(v); }
template <> LGX_D double fast_rsqrt<double>(double v) { return 1.0 / sqrt(v); }

// A uniform value held in a vector register (float).
template <class T> LGX_D T vec(T v) {
  if constexpr (sizeof(T) == 4) asm("" : "+v"(v));
  return v;
}

// A value that the compiler takes for a new one (what is formed from it is not
// merged with what was formed before).
template <class T> LGX_D T opaque(T v) {
  asm("" : "+v"(v));
  return v;
}

template <class T> LGX_D T fma_(T a, T b, T c) { return fma(a, b, c); }

template <class T> LGX_D T fast_rcp(T v);
template <> LGX_D float fast_rcp<float>(float v) { return __builtin_amdgcn_rcpf(v); }
template <> LGX_D double fast_rcp<double>(double v) { return 1.0 / v; }

// x / b for several x over one b, correctly rounded: r = RN(1/b) once, then
// per quotient y = RN(x r) and one fused correction with the exact residual
// x - y b (Markstein), which rounds to the IEEE quotient when r is the
// correctly rounded reciprocal (checked against the IEEE division for every
// significand of b, tests/csrc/check_common_div.c; x = -0 gives +0 here, a
// sign that no sum it enters keeps).
template <class T> LGX_D T div_by(T x, T b, T r) {
  if (sizeof(T) == 8) return x / b;
  const T y = x * r;
  const T e = fma(-y, b, x);
  return fma(e, r, y);
}

// RN(1 / b) for 2^-126 <= |b| < 2^126: the hardware's reciprocal (1 ulp) and
// one Newton step, 3 instructions instead of the division's 10
// (tests/csrc/check_device_math.hip compares all significands on the device,
// here and below).
template <class T> LGX_D T recip(T b) {
  if (sizeof(T) == 8) return T(1) / b;
  const T r = fast_rcp(b);
  return fma(fma(-b, r, T(1)), r, r);
}

// len = RN(sqrt(q)) for finite q >= 2^-100, from the hardware's reciprocal
// square root y and one residual correction of q y.  r: 1 / len by a Newton
// step from y, the IEEE quotient but for the lengths (2 - 2^-23) 2^k, where
// it is an ulp below; a quotient by one of those is an ulp off for x a power
// of two and the IEEE one for every other x.  7 instructions for the two
// instead of 27; the three normalisations of a direction's set-up were a
// quarter of it.  (A branch to IEEE operations for other q costs the gather's
// set-up registers; its callers see to the range.)
template <class T> LGX_D void root(T q, T &len, T &r) {
  if (sizeof(T) == 8) {
    len = sqrt(q);
    r = T(1) / len;
    return;
  }
  const T y = fast_rsqrt(q);
  const T g = q * y;
  len = fma(fma(-g, g, q), T(0.5) * y, g);
  r = fma(fma(-len, y, T(1)), y, y);
}
template <class T> LGX_D Vec3<T> normalize3_cr(Vec3<T> v) {
  T len, r;
  root(dot3(v, v), len, r);
  return Vec3<T>{div_by(v.x, len, r), div_by(v.y, len, r), div_by(v.z, len, r)};
}

// oct_decode with the device's exact roots and quotients (the same values).
template <class T> LGX_D Vec3<T> oct_decode_dev(T ex, T ey) {
  Vec3<T> n{ex, ey, T(1) - fabs(ex) - fabs(ey)};
  if (n.z < T(0)) {
    const T ox = (T(1) - fabs(n.y)) * (n.x >= T(0) ? T(1) : T(-1));
    const T oy = (T(1) - fabs(n.x)) * (n.y >= T(0) ? T(1) : T(-1));
    n.x = ox;
    n.y = oy;
  }
  return normalize3_cr(n);
}

// atan2(y, x) for finite arguments (atan2(0, 0) = 0), float: octant
// reduction to t = min(|x|, |y|) / max(|x|, |y|) in [0, 1] and
// atan(t) = t P(t^2) with a degree-7 polynomial fitted to atan(t) / t on
// [0, 1] by iteratively reweighted least squares (max error 4e-8; 1.2e-7
// evaluated in float).  The hit branch of the march calls it on every horizon
// rise, where the library routine's handling of infinities and NaNs (which
// cannot occur there) costs more than the polynomial.
// NONZERO: the caller's vector is not (0, 0).
template <bool NONZERO> LGX_D double atan2_finite(double y, double x) { return atan2(y, x); }
template <bool NONZERO> LGX_D float atan2_finite(float y, float x) {
  const float ax = fabsf(x), ay = fabsf(y);
  const bool steep = ay > ax;
  const float mx = steep ? ay : ax, mn = steep ? ax : ay;
  const float t = NONZERO || mx > 0.f ? mn * __builtin_amdgcn_rcpf(mx) : 0.f;
  const float s = t * t;
  float p = -0.004054928198456764f;
  p = fmaf(p, s, 0.021864214912056923f);
  p = fmaf(p, s, -0.05591406673192978f);
  p = fmaf(p, s, 0.0964231863617897f);
  p = fmaf(p, s, -0.1390867531299591f);
  p = fmaf(p, s, 0.19946573674678802f);
  p = fmaf(p, s, -0.33329862356185913f);
  p = fmaf(p, s, 0.9999993443489075f);
  float r = t * p;
  r = steep ? 1.5707963705062866f - r : r;
  r = x < 0.f ? 3.1415927410125732f - r : r;
  return copysignf(r, y);
}

// The angle th of a vector (x, y) that is not zero, cos 2 th and sin 2 th.
// IEEE: the library's arc tangent and the divisions; else the polynomial and
// the hardware's reciprocal (1 ulp, of a square that is neither subnormal nor
// infinite).
template <bool IEEE, class T> LGX_D void slice_angle(T y, T x, T &th, T &c2, T &s2) {
  const T q = x * x + y * y;
  if constexpr (IEEE) {
    th = atan2(y, x);
    c2 = (x * x - y * y) / q;
    s2 = (T(2) * x * y) / q;
  } else {
    th = atan2_finite<true>(y, x);
    const T iq = fast_rcp(q);
    c2 = (x * x - y * y) * iq;
    s2 = (T(2) * x * y) * iq;
  }
}

}  // namespace lgx
