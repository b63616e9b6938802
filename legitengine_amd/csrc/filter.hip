// Denoise and composite passes.
//
//  * lgx_bilateral: the geometry-aware filter whose weights are written (and
//    commented out) in denoiser.frag:87-110: w = exp(-|d - dc| * 10.5) *
//    exp(-|n - nc|^2 * 20) over the taps [-r, r)^2 (y outer, x inner), at
//    pixel centres with clamp to edge, colour / (sumW + 1e-7).  The output
//    tile of a workgroup plus its halo of irradiance, radial depth and decoded
//    normals is staged in LDS once, so each texel is read from memory about
//    once per pass instead of (2r)^2 times.
//  * lgx_regression_denoise: the live DenoiserPass (denoiser.frag:72-185).
//  * lgx_composite: finalGatherer.frag:42-58.
#include <math.h>

#include "device_math.h"
#include "lgx_internal.h"

namespace lgx {

struct BilatArgs {
  const float4 *in;
  int in_pitch;
  const float *depth;
  int depth_pitch;
  const void *normal;
  int normal_pitch;
  float4 *out;
  int out_pitch;
  int w, h, r;
  float ds, ns;
};

constexpr int kBilatMaxR = 8, kBilatTW = 32;

// One row of taps (n = 2r of them, geometry and colour in LDS) for the
// outputs LO..HI of a thread's column.
template <int R, int LO, int HI>
LGX_D void bilat_row(const float4 *geo, const float4 *col, int n, float kd, float kn, const float4 (&gc)[R], float4 (&acc)[R]) {
#pragma unroll 4
  for (int x = 0; x < n; x++) {
    const float4 gs = geo[x], c = col[x];
#pragma unroll
    for (int k = LO; k <= HI; k++) {
      // exp(-|dd| ds) exp(-|dn|^2 ns) = exp2(-|dd| kd - |dn|^2 kn): one
      // hardware exp2 (1 ulp) per tap.  kd and kn (of any sign) multiply the
      // differences, which are exact for neighbours: of values scaled first
      // every product would round at its own size
      const float dx = gs.y - gc[k].y, dy = gs.z - gc[k].z, dz = gs.w - gc[k].w;
      const float dn2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
      const float w = __builtin_amdgcn_exp2f(fmaf(-dn2, kn, -fabsf(gs.x - gc[k].x) * kd));
      acc[k].x = fmaf(c.x, w, acc[k].x);
      acc[k].y = fmaf(c.y, w, acc[k].y);
      acc[k].z = fmaf(c.z, w, acc[k].z);
      acc[k].w = fmaf(c.w, w, acc[k].w);
    }
  }
}
// the same for the uniform range lo..hi
template <int R, int LO = 0, int HI = 0>
LGX_D void bilat_rows(int lo, int hi, const float4 *geo, const float4 *col, int n, float kd, float kn, const float4 (&gc)[R],
                      float4 (&acc)[R]) {
  if (lo == LO && hi == HI)
    bilat_row<R, LO, HI>(geo, col, n, kd, kn, gc, acc);
  else if constexpr (HI + 1 < R)
    bilat_rows<R, LO, HI + 1>(lo, hi, geo, col, n, kd, kn, gc, acc);
  else if constexpr (LO + 1 < R)
    bilat_rows<R, LO + 1, LO + 1>(lo, hi, geo, col, n, kd, kn, gc, acc);
}

// A workgroup filters 32 x 8R pixels, a thread R pixels of one column, whose
// windows overlap in all but R - 1 of their rows: a tap read from LDS serves
// up to R outputs.  Bound by VALU issue (1.19 instructions a CU-cycle by
// counters; the taps' mix alone can reach 1.37): 14 instructions a tap with
// one exp2 (20 and their scalar operands before), about 330 a pixel for
// staging and the quotients.  More outputs a thread read less LDS and lose as
// much to the fewer workgroups that fit it.  2560x1440, r = 4: 133 -> 94 us a
// call.
template <int NFMT, int R> __global__ __launch_bounds__(256) void bilateral_kernel(const BilatArgs a) {
  extern __shared__ __align__(16) float4 s_bilat[];
  const int r = a.r, n = 2 * r;
  constexpr int TW = kBilatTW, TH = 256 / TW * R;
  const int sw = TW + n - 1, sh = TH + n - 1;  // taps reach -r .. r-1
  float4 *s_geo = s_bilat, *s_col = s_bilat + sw * sh;  // (depth, normal xyz), colour
  const int x0 = blockIdx.x * TW - r, y0 = blockIdx.y * TH - r;
  const float kd = vec(a.ds * 1.44269504f), kn = vec(a.ns * 1.44269504f);
  // Four texels of the tile a thread at a time, all their loads in flight
  // together: a load per row waited for its own round trip to memory, which
  // the few workgroups that fit a CU's LDS do not hide.
  const int total = sw * sh;
  const uint32_t inv = ((1u << 20) + sw - 1) / (uint32_t)sw;  // i / sw for i < 4096, sw in 16 .. 79
  // 32-bit byte offsets from the tile's first image row
  const int yb = max(y0, 0);
  const char *b_in = (const char *)(a.in + (size_t)yb * a.in_pitch);
  const char *b_n = (const char *)a.normal + (size_t)yb * a.normal_pitch * (NFMT == LGX_RG16F ? 4 : 8);
  const char *b_d = (const char *)(a.depth + (size_t)yb * a.depth_pitch);
  for (int i0 = threadIdx.x; i0 < total; i0 += 4 * 256) {
    float4 c[4];
    float2 nt[4];
    float d[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int i = min(i0 + u * 256, total - 1);
      const int ly = (int)(((uint32_t)i * inv) >> 20), lx = i - ly * sw;
      const uint32_t gx = (uint32_t)min(max(x0 + lx, 0), a.w - 1), row = (uint32_t)(min(max(y0 + ly, 0), a.h - 1) - yb);
      c[u] = *(const float4 *)(b_in + (row * (uint32_t)a.in_pitch + gx) * 16u);
      const float4 t = Texel<NFMT>::load(b_n + (row * (uint32_t)a.normal_pitch + gx) * (NFMT == LGX_RG16F ? 4u : 8u), 0);
      nt[u] = make_float2(t.x, t.y);
      d[u] = *(const float *)(b_d + (row * (uint32_t)a.depth_pitch + gx) * 4u);
    }
    // (a normal whose squared length overflows: uniform, no wave of unit normals goes there)
    float longest = 0.f;
#pragma unroll
    for (int u = 0; u < 4; u++) longest = fmaxf(longest, fabsf(nt[u].x) + fabsf(nt[u].y));
    const bool ieee = __builtin_amdgcn_ballot_w64(longest > 1e18f) != 0;
    auto stage = [&](auto decode) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = i0 + u * 256;
        if (i < total) {
          const Vec3<float> nv = decode(nt[u].x, nt[u].y);
          s_geo[i] = make_float4(d[u], nv.x, nv.y, nv.z);
          s_col[i] = make_float4(c[u].x, c[u].y, c[u].z, 1.0f);
        }
      }
    };
    if (ieee)
      stage([](float x, float y) { return oct_decode<float>(x, y); });
    else
      stage([](float x, float y) { return oct_decode_dev<float>(x, y); });
  }
  __syncthreads();
  const int tx = threadIdx.x % TW, ty = threadIdx.x / TW * R;
  float4 gc[R], acc[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    gc[k] = s_geo[(ty + k + r) * sw + tx + r];
    acc[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // window row j holds the taps of outputs k with 0 <= j - k < 2r
  for (int j = 0; j < n + R - 1; j++) {
    const int at = (ty + j) * sw + tx;
    bilat_rows<R>(max(j - n + 1, 0), min(j, R - 1), s_geo + at, s_col + at, n, kd, kn, gc, acc);
  }
  const int px = blockIdx.x * TW + tx, py = blockIdx.y * TH + ty;
  if (px >= a.w) return;
#pragma unroll
  for (int k = 0; k < R; k++) {
    if (py + k >= a.h) break;
    // IEEE quotients: an infinite sum stays infinite (1.4 us of the 94 at 2560x1440, r = 4, over one reciprocal and
    // its corrections, which give NaN there)
    const float sum = acc[k].w + 1e-7f;
    a.out[(size_t)(py + k) * a.out_pitch + px] = make_float4(acc[k].x / sum, acc[k].y / sum, acc[k].z / sum, 1.0f);
  }
}

__global__ __launch_bounds__(256) void copy4_kernel(const float4 *in, int ip, float4 *out, int op, int w, int h) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x < w && y < h) out[(size_t)y * op + x] = in[(size_t)y * ip + x];
}

struct RegArgs {
  const float4 *in;
  int in_pitch;
  const float *depth;
  int depth_pitch;
  float4 *out;
  int out_pitch;
  int w, h;
};

__global__ __launch_bounds__(256) void regression_kernel(const RegArgs a) {
  const int px = blockIdx.x * 16 + (threadIdx.x & 15), py = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (px >= a.w || py >= a.h) return;
  float dep[16];
  float3 col[16];
  int i = 0;
  for (int y = -2; y < 2; y++)  // denoiser.frag:116-123
    for (int x = -2; x < 2; x++) {
      const int sx = min(max(px + x, 0), a.w - 1), sy = min(max(py + y, 0), a.h - 1);
      dep[i] = a.depth[(size_t)sy * a.depth_pitch + sx];
      const float4 c = a.in[(size_t)sy * a.in_pitch + sx];
      col[i] = make_float3(c.x, c.y, c.z);
      i++;
    }
  float g00 = 0.f, g01 = 0.f, g11 = 0.f;  // :135-147
  for (int k = 0; k < 16; k++) g00 += dep[k] * dep[k];
  for (int k = 0; k < 16; k++) g01 += dep[k] * 1.0f;
  for (int k = 0; k < 16; k++) g11 += 1.0f * 1.0f;
  g00 += 1e-7f;
  g11 += 1e-7f;
  const float det = g00 * g11 - g01 * g01;  // 2x2 block of inverse(mat4) (:148)
  const float i00 = g11 / det, i01 = -g01 / det, i11 = g00 / det;
  const float dc = a.depth[(size_t)py * a.depth_pitch + px];
  float res[3];
  for (int ch = 0; ch < 3; ch++) {  // :154-184
    float m0 = 0.f, m1 = 0.f;
    for (int k = 0; k < 16; k++) m0 += dep[k] * (&col[k].x)[ch];
    for (int k = 0; k < 16; k++) m1 += 1.0f * (&col[k].x)[ch];
    const float c0 = i00 * m0 + i01 * m1;
    const float c1 = i01 * m0 + i11 * m1;
    res[ch] = c0 * dc + c1 * 1.0f;
  }
  a.out[(size_t)py * a.out_pitch + px] = make_float4(res[0], res[1], res[2], 1.0f);
}

template <int RFMT, int AFMT>
__global__ __launch_bounds__(256) void composite_kernel(const void *rad, int rp, const void *alb, int ap,
                                                        const float4 *ind, int ip, float4 *out, int op, int w, int h) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= w || y >= h) return;
  const float4 d = Texel<RFMT>::load(rad, (size_t)y * rp + x);
  const float4 al = Texel<AFMT>::load(alb, (size_t)y * ap + x);
  const float4 in = ind[(size_t)y * ip + x];
  out[(size_t)y * op + x] = make_float4(d.x + in.x * al.x, d.y + in.y * al.y, d.z + in.z * al.z, d.w + in.w * al.w);
}

}  // namespace lgx

using namespace lgx;

extern "C" int lgx_bilateral(const lgx_bilateral_params *p, const lgx_image *in, const lgx_gbuffer *g,
                             lgx_image *out, lgx_stream_t stream) {
  if (!p || !g || !image_ok(in) || !image_ok(out) || !image_ok(&g->depth) || !image_ok(&g->normal))
    return LGX_EINVAL;
  if (in->format != LGX_RGBA32F || out->format != LGX_RGBA32F || g->depth.format != LGX_R32F) return LGX_EFORMAT;
  if (g->normal.format != LGX_RG16F && g->normal.format != LGX_RG32F) return LGX_EFORMAT;
  if (in->w != out->w || in->h != out->h || g->depth.w != in->w || g->depth.h != in->h || g->normal.w != in->w ||
      g->normal.h != in->h)
    return LGX_ESIZE;
  if (p->radius < 0 || p->radius > kBilatMaxR) return LGX_EUNSUPPORTED;
  if (in->ptr == out->ptr) return LGX_EINVAL;  // taps read neighbours: no in-place
  hipStream_t s = (hipStream_t)stream;
  if (p->radius == 0) {  // denoiser.frag:82-86
    dim3 grid((in->w + 63) / 64, (in->h + 3) / 4);
    hipLaunchKernelGGL(copy4_kernel, grid, dim3(256), 0, s, (const float4 *)in->ptr, in->pitch, (float4 *)out->ptr,
                       out->pitch, in->w, in->h);
    return hip_status(hipGetLastError());
  }
  BilatArgs a{(const float4 *)in->ptr, in->pitch, (const float *)g->depth.ptr, g->depth.pitch, g->normal.ptr,
              g->normal.pitch, (float4 *)out->ptr, out->pitch, in->w, in->h, p->radius, p->depth_sharpness,
              p->normal_sharpness};
  auto launch = [&](auto kern, int R) {
    const int n = 2 * p->radius, TH = 256 / kBilatTW * R;
    const size_t lds = (size_t)(kBilatTW + n - 1) * (TH + n - 1) * 2 * sizeof(float4);
    hipLaunchKernelGGL(kern, dim3((in->w + kBilatTW - 1) / kBilatTW, (in->h + TH - 1) / TH), dim3(256), lds, s, a);
    return hip_status(hipGetLastError());
  };
  const bool h16 = g->normal.format == LGX_RG16F;
  // Two outputs a thread once their 4096 tiles of 32 x 16 keep every CU's five
  // workgroups busy for a few rounds (2560x1440, r = 4: 96 against 101 us a
  // call for one output; 1279x719, r = 3: 23.5 against 20.8 us).
  if ((int64_t)in->w * in->h >= (int64_t)4096 * 512)
    return h16 ? launch(bilateral_kernel<LGX_RG16F, 2>, 2) : launch(bilateral_kernel<LGX_RG32F, 2>, 2);
  return h16 ? launch(bilateral_kernel<LGX_RG16F, 1>, 1) : launch(bilateral_kernel<LGX_RG32F, 1>, 1);
}

extern "C" int lgx_regression_denoise(const lgx_image *in, const lgx_gbuffer *g, int32_t radius, lgx_image *out,
                                      lgx_stream_t stream) {
  if (!g || !image_ok(in) || !image_ok(out) || !image_ok(&g->depth)) return LGX_EINVAL;
  if (in->format != LGX_RGBA32F || out->format != LGX_RGBA32F || g->depth.format != LGX_R32F) return LGX_EFORMAT;
  if (in->w != out->w || in->h != out->h || g->depth.w != in->w || g->depth.h != in->h) return LGX_ESIZE;
  if (in->ptr == out->ptr) return LGX_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  if (radius == 0) {
    dim3 grid((in->w + 63) / 64, (in->h + 3) / 4);
    hipLaunchKernelGGL(copy4_kernel, grid, dim3(256), 0, s, (const float4 *)in->ptr, in->pitch, (float4 *)out->ptr,
                       out->pitch, in->w, in->h);
    return hip_status(hipGetLastError());
  }
  RegArgs a{(const float4 *)in->ptr, in->pitch, (const float *)g->depth.ptr, g->depth.pitch, (float4 *)out->ptr,
            out->pitch, in->w, in->h};
  dim3 grid((in->w + 15) / 16, (in->h + 15) / 16);
  hipLaunchKernelGGL(regression_kernel, grid, dim3(256), 0, s, a);
  return hip_status(hipGetLastError());
}

extern "C" int lgx_composite(const lgx_gbuffer *g, const lgx_image *indirect, lgx_image *out, lgx_stream_t stream) {
  if (!g || !image_ok(indirect) || !image_ok(out) || !image_ok(&g->radiance) || !image_ok(&g->albedo))
    return LGX_EINVAL;
  if (indirect->format != LGX_RGBA32F || out->format != LGX_RGBA32F) return LGX_EFORMAT;
  const int w = out->w, h = out->h;
  if (indirect->w != w || indirect->h != h || g->radiance.w != w || g->radiance.h != h || g->albedo.w != w ||
      g->albedo.h != h)
    return LGX_ESIZE;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((w + 63) / 64, (h + 3) / 4), block(256);
  const int rf = g->radiance.format, af = g->albedo.format;
  const void *rp = g->radiance.ptr, *ap = g->albedo.ptr;
  const float4 *ip = (const float4 *)indirect->ptr;
  float4 *op = (float4 *)out->ptr;
  if (rf == LGX_RGBA16F && af == LGX_RGBA8)
    hipLaunchKernelGGL((composite_kernel<LGX_RGBA16F, LGX_RGBA8>), grid, block, 0, s, rp, g->radiance.pitch, ap,
                       g->albedo.pitch, ip, indirect->pitch, op, out->pitch, w, h);
  else if (rf == LGX_RGBA32F && af == LGX_RGBA32F)
    hipLaunchKernelGGL((composite_kernel<LGX_RGBA32F, LGX_RGBA32F>), grid, block, 0, s, rp, g->radiance.pitch, ap,
                       g->albedo.pitch, ip, indirect->pitch, op, out->pitch, w, h);
  else if (rf == LGX_RGBA16F && af == LGX_RGBA32F)
    hipLaunchKernelGGL((composite_kernel<LGX_RGBA16F, LGX_RGBA32F>), grid, block, 0, s, rp, g->radiance.pitch, ap,
                       g->albedo.pitch, ip, indirect->pitch, op, out->pitch, w, h);
  else if (rf == LGX_RGBA32F && af == LGX_RGBA8)
    hipLaunchKernelGGL((composite_kernel<LGX_RGBA32F, LGX_RGBA8>), grid, block, 0, s, rp, g->radiance.pitch, ap,
                       g->albedo.pitch, ip, indirect->pitch, op, out->pitch, w, h);
  else
    return LGX_EFORMAT;
  return hip_status(hipGetLastError());
}
