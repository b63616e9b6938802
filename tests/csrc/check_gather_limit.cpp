// The end of the gather's march (gather_march.h, in float as the kernels call
// it, on float tables formed as the host forms them) against the shader's rule
// in double, step by step: a step that only one of the two admits lies
//  * in the outermost 2^-20 of the extent, which the FP32 march leaves out, or
//    within rounding of a border: an offset of the path has four roundings and
//    the reciprocal's, together below 2^-21 of it, and no position on screen
//    is farther than the extent.  So at most 2^-20 + 2^-21 of the extent
//    inside, a fade of 1.5e-5.
//  * or within rounding of the step count's end, near ratio^j = path to 2^-19.
// Usage: check_gather_limit [mistake]; mistake 1 ends the march 1 % early, 2
// forgets the path between near / ratio and near, 3 takes the far borders
// 2^-12 early, 4 forgets the step count: each has to be found.  Prints
// "ok <steps admitted> <differences>" or the first step that is wrong.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <vector>

#include "gather_march.h"

using namespace lgx;

static uint64_t g_s = 0x9E3779B97F4A7C15ull;
static uint32_t rnd() {
  g_s ^= g_s << 13;
  g_s ^= g_s >> 7;
  g_s ^= g_s << 17;
  return (uint32_t)(g_s >> 16);
}

static unsigned long long g_admitted, g_different;

static bool check(int w, int h, int footprint, int cap, int pixels, int mistake) {
  const float W = (float)w, H = (float)h, near_step = W / 1000.f, ratio = 2.f * 3.1415f / (float)footprint + 1.f;
  const float near_min = near_step / ratio;
  int steps = (int)(logf(sqrtf(W * W + H * H) / near_step) / logf(ratio)) + 2;
  if (cap && steps > cap) steps = cap;
  if (steps < 1) steps = 1;
  std::vector<float> off(steps);
  for (int i = 0; i < pixels; i++) {
    const uint32_t edge = rnd() % 4;  // half of the pixels next to a border
    int x = (int)(rnd() % w), y = (int)(rnd() % h);
    if (edge == 0) x = rnd() % 2 ? w - 1 - (int)(rnd() % (w < 4 ? w : 4)) : (int)(rnd() % (w < 4 ? w : 4));
    if (edge == 1) y = rnd() % 2 ? h - 1 - (int)(rnd() % (h < 4 ? h : 4)) : (int)(rnd() % (h < 4 ? h : 4));
    const float cx = (float)x + 0.5f, cy = (float)y + 0.5f, lin = (float)(rnd() % 16) / 16.f;
    float dx, dy;
    switch (rnd() % 8) {
      case 0: dx = 1.f, dy = 0.f; break;
      case 1: dx = 0.f, dy = -1.f; break;
      case 2: dx = -1.f, dy = 9.2654e-5f; break;  // (the shader's pi)
      case 3: dx = 1e-7f, dy = 1.f; break;
      default: {
        const float a = 2.f * 3.1415f * (float)(rnd() & 0xffffffu) * 0x1p-24f;
        dx = cosf(a), dy = sinf(a);
      }
    }
    const float idx = 1.f / dx, idy = 1.f / dy;
    for (int j = 0; j < steps; j++) off[j] = near_step * powf(ratio, (float)j + lin) + 1.f - near_step;
    const float path = border_path(cx, cy, W, H, idx, idy), second = steps > 1 ? off[1] : INFINITY;
    float lim = march_limit(path, near_step, mistake == 2 ? near_step : near_min, off[0], second);
    if (mistake == 4) lim = path;
    if (mistake == 1) lim *= 0.99f;
    float early = inside_far(lim, cx, cy, W, H, dx, dy, idx, idy);
    if (mistake == 3) {
      const float far = 1.f - 0x1p-12f;
      if (dx > 0.f) early = fminf(early, (W * far - cx) * idx);
      if (dy > 0.f) early = fminf(early, (H * far - cy) * idy);
    }
    // the rule in double
    auto to = [](double c, double d, double e) { return d > 0 ? (e - c) / d : d < 0 ? -c / d : INFINITY; };
    const double dpath = fmin(to(cx, dx, w), to(cy, dy, h)), dnear = w / 1000.0, dratio = (double)ratio;
    const double iters = trunc(log(dpath / dnear) / log(dratio)) + 1;
    for (int j = 0; j < steps; j++) {
      const double sx = (cx + (double)dx * off[j]) / w, sy = (cy + (double)dy * off[j]) / h;
      const double in = fmin(fmin(sx, 1 - sx), fmin(sy, 1 - sy));
      const bool rule = j < iters && in > 0;
      g_admitted += rule;
      // within rounding of where the step count ends: at step j, and below near at near / ratio
      const bool end = fabs(dnear * pow(dratio, j) / dpath - 1) <= 0x1p-19 || fabs(dnear / dratio / dpath - 1) <= 0x1p-19;
      for (const float l : {lim, early}) {
        const bool march = off[j] < l;
        if (march == rule) continue;
        g_different++;
        if (in > 0x1p-20 + 0x1p-21 && !end) {
          printf("%d x %d footprint %d cap %d: pixel %d %d direction %a %a step %d offset %a limit %a rule %d (inside %g)\n",
                 w, h, footprint, cap, x, y, dx, dy, j, off[j], l, rule, in);
          return false;
        }
      }
    }
  }
  return true;
}

int main(int argc, char **argv) {
  const int mistake = argc > 1 ? atoi(argv[1]) : 0;
  const int sizes[][2] = {{1, 1}, {5, 3}, {97, 61}, {256, 144}, {1000, 562}, {1279, 719}, {2560, 1440}, {7680, 4320}};
  for (auto &s : sizes)
    for (int footprint : {1, 4, 32, 256})
      for (int cap : {0, 1, 7})
        if (!check(s[0], s[1], footprint, cap, 4000, mistake)) return 1;
  printf("ok %llu %llu\n", g_admitted, g_different);
  return 0;
}
