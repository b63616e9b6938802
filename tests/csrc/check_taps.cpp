// The trilinear sampler's taps (gather_taps.h, in float as the kernels call
// it) against clamp-to-edge taps blended in double, over levels of 1 to 9
// texels with values of very different sizes side by side, infinite ones and
// points from outside one border to the other.
//
// First, bit for bit, the shader's float arithmetic written out: flat surfaces
// tie the horizon test, and another last bit is another set of hits.
// Bound for finite texels: a blend a (1 - w) + b w rounds 1 - w, two products
// and a sum, together at most 3 2^-24 of (1 - w) |a| + w |b|, and there are
// three blends (columns, rows, levels); the weights are taken from the float
// u = s W - 1/2 on both sides, whose fraction is exact but below 0, where it
// rounds once more per axis.  So the error is at most 11 2^-24 (and
// second-order terms) times the blend of the absolute values: 11.1 2^-24.  An
// infinite texel: the same class and sign.  The form a + w (b - a), which
// rounds at the larger texel, and pairs of neighbours with saturating weights
// have to fail here.  Prints "ok <samples> <samples at infinite texels>
// <samples that the difference form misses> <that the pairs miss>", or the
// first difference.
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
struct Quad {
  float p00, p10, p01, p11;
};
static Quad quad(const Level &l, int x0, int x1, int y0, int y1) {
  return {l.t[y0 * l.w + x0], l.t[y0 * l.w + x1], l.t[y1 * l.w + x0], l.t[y1 * l.w + x1]};
}
static Quad quad(const Level &l, const TapPos<float> &p) { return quad(l, p.x0, p.x1, p.y0, p.y1); }
static float mix(const TapPos<float> &p, const Quad &q) { return p.mix(q.p00, q.p10, q.p01, q.p11); }
// a pair of neighbours moved inside, with saturating weights
static float paired(const Level &l, float sx, float sy) {
  const float u = sx * (float)l.w - 0.5f, v = sy * (float)l.h - 0.5f;
  const float fu = fmaxf(fminf(floorf(u), (float)(l.w - 2)), 0.f), fv = fmaxf(fminf(floorf(v), (float)(l.h - 2)), 0.f);
  const float al = fminf(fmaxf(u - fu, 0.f), 1.f), be = fminf(fmaxf(v - fv, 0.f), 1.f);
  const int x = (int)fu, y = (int)fv;
  const Quad q = quad(l, x, l.w > 1 ? x + 1 : x, y, l.h > 1 ? y + 1 : y);
  auto lerp = [](float w, float a, float b) { return fmaf(w, b - a, a); };
  return lerp(be, lerp(al, q.p00, q.p10), lerp(al, q.p01, q.p11));
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
// the same in float, every operation rounded by itself
static float written_out(const Level &l, float sx, float sy) {
  const float u = sx * (float)l.w - 0.5f, v = sy * (float)l.h - 0.5f;
  const float a = u - floorf(u), b = v - floorf(v);
  auto at = [&](int dx, int dy) {
    const int x = (int)floorf(u) + dx, y = (int)floorf(v) + dy;
    return l.t[(y < 0 ? 0 : y >= l.h ? l.h - 1 : y) * l.w + (x < 0 ? 0 : x >= l.w ? l.w - 1 : x)];
  };
  const float ca = 1.f - a, cb = 1.f - b;
  const float t0 = at(0, 0) * ca, t1 = at(1, 0) * a, b0 = at(0, 1) * ca, b1 = at(1, 1) * a;
  const float top = t0 + t1, bot = b0 + b1, top_w = top * cb, bot_w = bot * b;
  return top_w + bot_w;
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
  unsigned long long n = 0, at_inf = 0, missed = 0, pairs = 0;
  for (int i = 0; i < 4000000; i++) {
    const bool inf = i % 4 == 0;
    Level l0, l1;
    fill(l0, inf);
    fill(l1, inf);
    const float sx = point(rnd() % 2 ? l0.w : l1.w), sy = point(rnd() % 2 ? l0.h : l1.h), f = unit();
    const bool blend = rnd() % 4 != 0 && f > 0.f;
    const TapPos<float> p0(sx, sy, l0.w, l0.h), p1(sx, sy, l1.w, l1.h);
    const int in[4] = {p0.x0, p0.x1, p0.y0, p0.y1}, of[4] = {l0.w, l0.w, l0.h, l0.h};
    for (int k = 0; k < 4; k++)
      if (in[k] < 0 || in[k] >= of[k]) {
        printf("tap outside the level: %d of %d at %a %a\n", in[k], of[k], sx, sy);
        return 1;
      }
    const Quad q0 = quad(l0, p0), q1 = quad(l1, p1);
    float got = mix(p0, q0);
    if (blend) got = TapPos<float>::lerp(f, got, mix(p1, q1));
    float same = written_out(l0, sx, sy);
    if (blend) same = same * (1.f - f) + written_out(l1, sx, sy) * f;
    if (!(got == same || (isnan(got) && isnan(same)))) {
      printf("%a, written out %a (%d x %d, %a %a, blend %d)\n", got, same, l0.w, l0.h, sx, sy, blend);
      return 1;
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
    const double bound = 11.1 * 0x1p-24 * want;  // (all texels are positive)
    if (!(fabs((double)got - want) <= bound)) {
      printf("%a, wanted %a (%d x %d, %a %a, blend %d)\n", got, want, l0.w, l0.h, sx, sy, blend);
      return 1;
    }
    auto diff = [](float w1, float a, float b) { return fmaf(w1, b - a, a); };
    auto differences = [&](const TapPos<float> &p, const Quad &q) {
      return diff(p.be, diff(p.al, q.p00, q.p10), diff(p.al, q.p01, q.p11));
    };
    const float d = blend ? diff(f, differences(p0, q0), differences(p1, q1)) : differences(p0, q0);
    missed += !(fabs((double)d - want) <= bound);
    const float e = blend ? diff(f, paired(l0, sx, sy), paired(l1, sx, sy)) : paired(l0, sx, sy);
    pairs += !(fabs((double)e - want) <= bound);
  }
  printf("ok %llu %llu %llu %llu\n", n, at_inf, missed, pairs);
  return 0;
}
