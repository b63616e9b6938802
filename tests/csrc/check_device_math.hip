// The device's short roots, reciprocals and quotients (device_math.h) against
// the IEEE operations they stand for, on the GPU:
//   recip     every significand and sign at binades from the first to the last
//             that it covers
//   root      every significand at binades of both parities, first and last
//             included: the length, and some quotients by it
//   odd       the lengths whose reciprocal is not the correctly rounded one:
//             (2 - 2^-23) 2^k, an ulp below
//   odd_quotients  every significand divided by each of those: the IEEE
//             quotient, but for an ulp at the powers of two
//   vectors   normalize3_cr against the quotients by the root
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

__global__ void recip_kernel(int e, Count *c) {
  unsigned long long bad = 0;
  const float b = make(blockIdx.x * 256 + threadIdx.x, e);
  for (int s = 0; s < 2; s++) {
    const float x = s ? -b : b;
    if (!same(recip(x), 1.f / x)) bad++;
  }
  tally(c, !bad, b);
}

// odd: lengths whose reciprocal is off, at most cap of them
__global__ void root_kernel(int e, Count *c, Count *q, float *odd, unsigned *odd_n, unsigned cap) {
  const uint32_t m = blockIdx.x * 256 + threadIdx.x;
  const float v = make(m, e);
  float len, r;
  root(v, len, r);
  const float want = sqrtf(v);
  tally(c, same(len, want), v);
  if (r != 1.f / want) {
    // (a length of another form, or farther off, is a difference of `root`)
    const uint32_t b = __builtin_bit_cast(uint32_t, want), d = __builtin_bit_cast(uint32_t, 1.f / want);
    if ((b & 0x7fffffu) != 0x7fffffu || __builtin_bit_cast(uint32_t, r) + 1 != d) tally(c, false, v, r);
    const unsigned at = atomicAdd(odd_n, 1u);
    if (at < cap) {
      odd[2 * at] = len;
      odd[2 * at + 1] = r;
    }
  }
  unsigned bad = 0;
  for (uint32_t i = 0; i < 16; i++) {
    const float x = make(hash(m * 16 + i) & 0x7fffffu, e / 2 - (int)(i & 7));
    if (!same(div_by(x, len, r), x / len) && r == 1.f / want) bad++;
  }
  tally(q, !bad, v);
}
__global__ void quotient_kernel(const float *odd, Count *c) {
  const float len = odd[2 * blockIdx.y], r = odd[2 * blockIdx.y + 1];
  const float x = make(blockIdx.x * 256 + threadIdx.x, 0);
  const float got = div_by(x, len, r), want = x / len;
  const int ulp = __builtin_bit_cast(int, got) - __builtin_bit_cast(int, want);
  tally(c, ulp == 0 || (x == 1.f && ulp == -1), x, len);
}

__global__ void vector_kernel(float scale, Count *c) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  float v[3];
  for (int k = 0; k < 3; k++) {
    v[k] = ((float)(hash(3 * i + k) >> 8) * 0x1p-23f - 1.f) * scale;
    if ((hash(i * 7 + k + 99) & 15u) < 3) v[k] = 0.f;
  }
  if (v[0] == 0.f && v[1] == 0.f && v[2] == 0.f) v[0] = scale;
  const Vec3<float> a{v[0], v[1], v[2]}, n = normalize3_cr(a);
  const float len = sqrtf(dot3(a, a));
  tally(c, same(n.x, v[0] / len) && same(n.y, v[1] / len) && same(n.z, v[2] / len), v[0], len);
}

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
  constexpr int kChecks = 8, kSig = (1 << 23) / 256;  // workgroups for all significands
  constexpr unsigned kCap = 4096;
  float *odd;
  unsigned *odd_n, n = 0;
  if (hipMalloc(&g_dev, kChecks * sizeof(Count)) != hipSuccess || hipMalloc(&odd, 2 * kCap * sizeof(float)) != hipSuccess ||
      hipMalloc(&odd_n, sizeof(unsigned)) != hipSuccess || hipMemset(g_dev, 0, kChecks * sizeof(Count)) != hipSuccess ||
      hipMemset(odd_n, 0, sizeof(unsigned)) != hipSuccess) {
    printf("no device memory\n");
    return 2;
  }
  bool ok = true;
  for (int e : {-126, -125, -60, -1, 0, 1, 60, 124, 125}) recip_kernel<<<kSig, 256>>>(e, g_dev);
  ok &= report("recip", 0);
  for (int e : {-100, -99, -42, -1, 0, 1, 2, 63, 124, 125, 126, 127})
    root_kernel<<<kSig, 256>>>(e, g_dev + 1, g_dev + 2, odd, odd_n, kCap);
  ok &= report("root", 1);
  ok &= report("root_quotients", 2);
  if (hipMemcpy(&n, odd_n, sizeof(n), hipMemcpyDeviceToHost) != hipSuccess || !n || n > kCap) {
    printf("odd %u\n", n);
    return 1;
  }
  printf("odd %u\n", n);
  for (unsigned at = 0; at < n; at += 64)
    quotient_kernel<<<dim3(kSig, n - at < 64 ? n - at : 64), 256>>>(odd + 2 * at, g_dev + 3);
  ok &= report("odd_quotients", 3);
  for (float s : {1e-14f, 1e-3f, 1.f, 1e3f, 1e10f, 5e18f}) vector_kernel<<<4096, 256>>>(s, g_dev + 4);
  ok &= report("vectors", 4);
  for (int e : {-40, -8, 0, 30}) angle_kernel<<<16384, 256>>>(e, g_dev + 5);
  ok &= report("angles", 5);
  return ok && hipDeviceSynchronize() == hipSuccess ? 0 : 1;
}
