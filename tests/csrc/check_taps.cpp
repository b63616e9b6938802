// The trilinear sampler's taps (gather_taps.h, in float as the kernels call
// it) against clamp-to-edge taps blended in double, over levels of 1 to 9
// texels with values of very different sizes side by side, infinite ones and
// points from outside one border to the other.
//
// Bound for finite texels: a blend a (1 - w) + b w of two fused operations
// rounds twice, each by at most 2^-24 of (1 - w) |a| + w |b|, and there are
// three blends (columns, rows, levels); the weights are taken from the float
// u = s W - 1/2 on both sides, whose fraction is exact from texel to texel.
// So the error is at most 6 2^-24 (and second-order terms) times the blend of
// the absolute values: 6.1 2^-24.  An infinite texel: the same class and sign.
// The form a + w (b - a), which rounds at the larger texel, has to fail here.
// Prints "ok <samples> <samples at infinite texels> <samples that the other
// form misses>", or the first difference.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include "gather_taps.h"

using namespace lgx;

static uint64_t g_s = 0x9E3779B97F4A7C15ull;
static uint32_t rnd() {
  g_s ^= g_s << 13;
  g_s ^= g_s >> 7;
  g_s ^= g_s << 17;
  return (uint32_t)(g_s >> 16);
}
static float unit() { return (float)(rnd() & 0xffffffu) * 0x1p-24f; }

struct Level {
  int w, h;
  float t[81];
};
static void fill(Level &l, bool inf) {
  l.w = 1 + rnd() % 9;
  l.h = 1 + rnd() % 9;
  for (int i = 0; i < l.w * l.h; i++) {
    static const float big[4] = {1.f, 65504.f, 1e8f, 1e-3f};
    l.t[i] = (0.5f + unit()) * big[rnd() % 4];
    if (inf && rnd() % 6 == 0) l.t[i] = INFINITY;
  }
}
static Quad<float> quad(const Level &l, const TapPos<float> &p) {
  const int x1 = l.w > 1 ? p.x + 1 : p.x, y1 = l.h > 1 ? p.y + 1 : p.y;
  return {l.t[p.y * l.w + p.x], l.t[p.y * l.w + x1], l.t[y1 * l.w + p.x], l.t[y1 * l.w + x1]};
}
// clamped taps in double, and the blend of their absolute values
static void exact(const Level &l, float sx, float sy, double &v) {
  const float u = sx * (float)l.w - 0.5f, w = sy * (float)l.h - 0.5f;
  const float fu = floorf(u), fv = floorf(w);
  const double a = (double)u - fu, b = (double)w - fv;
  auto cl = [](int k, int n) { return k < 0 ? 0 : k > n - 1 ? n - 1 : k; };
  const int x0 = cl((int)fu, l.w), x1 = cl((int)fu + 1, l.w), y0 = cl((int)fv, l.h), y1 = cl((int)fv + 1, l.h);
  auto at = [&](int x, int y) { return (double)l.t[y * l.w + x]; };
  auto lerp = [](double w1, double p, double q) { return p * (1 - w1) + q * w1; };
  v = lerp(b, lerp(a, at(x0, y0), at(x1, y0)), lerp(a, at(x0, y1), at(x1, y1)));
}
static float point(int n) {
  switch (rnd() % 4) {
    case 0: return unit() * 0.5f / n;                        // the first half texel
    case 1: return 1.f - unit() * 0.5f / n;                  // the last
    case 2: return ((float)(rnd() % n) + 0.5f) / (float)n;  // a texel's centre
    default: return unit() * 1.002f - 0.001f;
  }
}

int main() {
  unsigned long long n = 0, at_inf = 0, missed = 0;
  for (int i = 0; i < 4000000; i++) {
    const bool inf = i % 4 == 0;
    Level l0, l1;
    fill(l0, inf);
    fill(l1, inf);
    const float sx = point(rnd() % 2 ? l0.w : l1.w), sy = point(rnd() % 2 ? l0.h : l1.h), f = unit();
    const bool blend = rnd() % 4 != 0 && f > 0.f;
    const TapPos<float> p0(sx, sy, l0.w, l0.h), p1(sx, sy, l1.w, l1.h);
    if (p0.x < 0 || p0.y < 0 || p0.x > (l0.w > 1 ? l0.w - 2 : 0) || p0.y > (l0.h > 1 ? l0.h - 2 : 0)) {
      printf("pair outside the level: %d %d of %d x %d at %a %a\n", p0.x, p0.y, l0.w, l0.h, sx, sy);
      return 1;
    }
    const Quad<float> q0 = quad(l0, p0), q1 = quad(l1, p1);
    // (as the kernels sample: blends, and tap by tap what is not finite)
    float got = p0.mix(q0);
    if (blend) got = TapPos<float>::lerp(f, got, p1.mix(q1));
    if (!finite_tap(got)) {
      got = clamped_taps(sx, sy, l0.w, l0.h, q0);
      if (blend) got = got * (1.f - f) + clamped_taps(sx, sy, l1.w, l1.h, q1) * f;
    }
    double want, other = 0;
    exact(l0, sx, sy, want);
    if (blend) {
      exact(l1, sx, sy, other);
      want = want * (1 - (double)f) + other * (double)f;
    }
    n++;
    if (!(fabs(want) < INFINITY)) {
      at_inf++;
      if (isnan(want) != isnan(got) || (!isnan(want) && got != (float)want)) {
        printf("infinite texel: %a, wanted %a (%d x %d, %a %a)\n", got, want, l0.w, l0.h, sx, sy);
        return 1;
      }
      continue;
    }
    const double bound = 6.1 * 0x1p-24 * want;  // (all texels are positive)
    if (!(fabs((double)got - want) <= bound)) {
      printf("%a, wanted %a (%d x %d, %a %a, blend %d)\n", got, want, l0.w, l0.h, sx, sy, blend);
      return 1;
    }
    auto diff = [](float w1, float a, float b) { return fmaf(w1, b - a, a); };
    auto mix = [&](const TapPos<float> &p, const Quad<float> &q) {
      return diff(p.be, diff(p.al, q.p00, q.p10), diff(p.al, q.p01, q.p11));
    };
    const float d = blend ? diff(f, mix(p0, q0), mix(p1, q1)) : mix(p0, q0);
    missed += !(fabs((double)d - want) <= bound);
  }
  printf("ok %llu %llu %llu\n", n, at_inf, missed);
  return 0;
}
