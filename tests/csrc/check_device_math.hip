// The device's short arithmetic (device_math.h) on the GPU:
//   angles    the trilinear gather's slice angles against the double arc tangent
// Prints "<name> <compared> <differences>" per check; exit status 0 if there
// are none.
#include <stdio.h>

#include "device_math.h"

using namespace lgx;

namespace {

LGX_D bool same(float a, float b) {
  return a == b || (a != a && b != b);
}
LGX_D uint32_t hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  return x ^ x >> 16;
}

struct Count {
  unsigned long long n, bad;
  float at[4];
};
LGX_D void tally(Count *c, bool ok, float a = 0.f, float b = 0.f) {
  atomicAdd(&c->n, 1ull);
  if (!ok && atomicAdd(&c->bad, 1ull) == 0) {
    c->at[0] = a;
    c->at[1] = b;
  }
}
LGX_D float make(uint32_t m, int e) { return ldexpf(1.f + (float)m * 0x1p-23f, e); }  // (denormal below -126)

// a slice's angle: within 3 2^-23 of the double arc tangent (a correctly rounded one is within 2^-24; the library's
// documentation gives it 2 ulp), the quotients those of the divisions
__global__ void angle_kernel(int e, Count *c) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const float y = make(hash(2 * i) & 0x7fffffu, e + (int)(hash(i + 77) % 41u) - 20);
  const float x = make(hash(2 * i + 1) & 0x7fffffu, e) * (i & 1 ? -1.f : 1.f);
  float th, c2, s2;
  slice_angle<true>(y, x, th, c2, s2);
  const double want = atan2((double)y, (double)x);
  const float q = x * x + y * y;
  tally(c, fabs((double)th - want) <= 3 * 0x1p-23 * want && same(c2, (x * x - y * y) / q) && same(s2, (2.f * x * y) / q), y, x);
}

Count *g_dev;
bool report(const char *name, int idx) {
  Count h;
  if (hipMemcpy(&h, g_dev + idx, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) {
    printf("%s: %s\n", name, hipGetErrorString(hipGetLastError()));
    return false;
  }
  printf("%s %llu %llu", name, h.n, h.bad);
  if (h.bad) printf(" (%a %a)", h.at[0], h.at[1]);
  printf("\n");
  fflush(stdout);
  return h.n && !h.bad;
}

}  // namespace

int main() {
  constexpr int kChecks = 8;
  if (hipMalloc(&g_dev, kChecks * sizeof(Count)) != hipSuccess || hipMemset(g_dev, 0, kChecks * sizeof(Count)) != hipSuccess) {
    printf("no device memory\n");
    return 2;
  }
  bool ok = true;
  for (int e : {-40, -8, 0, 30}) angle_kernel<<<16384, 256>>>(e, g_dev);
  ok &= report("angles", 0);
  return ok && hipDeviceSynchronize() == hipSuccess ? 0 : 1;
}
