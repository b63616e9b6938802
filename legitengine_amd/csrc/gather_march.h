// Where the gather's march along a direction ends.  Arithmetic only, host and
// device (tests/csrc/check_gather_limit.cpp calls it on the CPU): no HIP
// header.
#pragma once
#include <math.h>

#ifndef LGX_HD  // included by host code alone
#define LGX_HD inline
#endif

namespace lgx {

// indirectLighting.frag:202-204 the offset at which a ray from (cx, cy) leaves
// the screen (idx, idy: the reciprocals of its direction)
template <class T> LGX_HD T border_path(T cx, T cy, T W, T H, T idx, T idy) {
  const T t1 = (T(0) - cx) * idx, t2 = (W - cx) * idx, t3 = (T(0) - cy) * idy, t4 = (H - cy) * idy;
  return fabs(fmin(fmax(t1, t2), fmax(t3, t4)));
}

// The march takes the steps whose offset is below a limit, instead of a step
// count and four screen tests: the ray leaves the screen at offset `path`, and
// the shader's step count int(log(path / near) / log(ratio)) + 1 (:212) admits
// step j while near ratio^j <= path, i.e. while the offset near
// ratio^(j + lin) + 1 - near (:217) is at most path ratio^lin + 1 - near;
// below near, where the logarithm is negative, the truncation admits step 0
// alone while path > near / ratio (near_min).  A step within rounding of the
// border may fall on either side: its side fade is 0 there.
// first, second: the offsets of steps 0 and 1 (infinity if there is no other).
template <class T> LGX_HD T growth_limit(T path, T near_step, T first) {
  const T rlin = (first - T(1) + near_step) / near_step;
  return fma(path, rlin, T(1) - near_step);
}
template <class T> LGX_HD T march_limit(T path, T near_step, T near_min, T first, T second) {
  const T lim = path >= near_step ? growth_limit(path, near_step, first) : path > near_min ? second : T(0);
  return fmin(lim, path);
}

// With FP32 sums the far borders are taken 2^-20 of the extent early (0.002
// pixels at 1920, where the fade is below 1e-5): whatever the roundings of the
// limit and of a step's position, the position stays below the extent, and so
// does its texel, which then needs no clamp.
template <class T> LGX_HD T inside_far(T lim, T cx, T cy, T W, T H, T dx, T dy, T idx, T idy) {
  const T far = T(1 - 0x1p-20);
  if (dx > T(0)) lim = fmin(lim, (W * far - cx) * idx);
  if (dy > T(0)) lim = fmin(lim, (H * far - cy) * idy);
  return lim;
}

}  // namespace lgx
