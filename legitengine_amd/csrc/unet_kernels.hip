// U-Net denoiser kernels for gfx950: BF16 activations and weights, FP32
// accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).
//
// Replaces the reference's regression DenoiserPass (SSVGIRenderer.h:265-302,
// denoiser.frag:112-184) with a learned filter; the layer graph lives in
// unet.cpp.
//
// Layouts: activations NHWC bf16 with channel counts that are multiples of
// 32 (convolution inputs) or 16 (outputs).  Convolution weights are packed
// per K-chunk: [tap 9][Cin/32][Cout][32], so one lane's MFMA operand (8
// consecutive input channels of one output channel) is a single 16-byte load.
//
// MFMA 16x16x32 operand layout (gfx950, wave64, lane l, item i of 8 / 4):
//   A (16 x 32, row m, col k):  m = l % 16, k = 8 * (l / 16) + i
//   B (32 x 16, row k, col n):  n = l % 16, k = 8 * (l / 16) + i
//   D (16 x 16):                n = l % 16, m = 4 * (l / 16) + i
// The convolution maps M = output channels, N = pixels, K = (tap, Cin):
// A is read from the packed weights, B straight from the NHWC activations
// (16 bytes = 8 channels of one pixel per lane), and each lane's result is 4
// consecutive output channels of one pixel (one 8-byte store).
#include <limits.h>
#include <math.h>

#include <algorithm>

#include "lgx_internal.h"
#include "unet.h"

namespace lgx {
namespace unet {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

LGX_D float bf2f(bf16 v) { return (float)v; }
LGX_D bf16 f2bf(float v) { return (bf16)v; }

// ------------------------------------------------------------ convolution

// The value of the neighbouring lane (lane ^ 1): a DPP quad permutation
// [1, 0, 3, 2], a modifier of one VALU move (no LDS round trip as a shuffle
// through ds_bpermute would take).
LGX_D float lane_xor1(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
}

// One image row of a tensor as a buffer of its own, so a column past the row
// is past the buffer: reads give 0 and stores are dropped without a branch.
LGX_D __amdgpu_buffer_rsrc_t row_rsrc(const bf16 *p, size_t row, int w, int stride) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)(p + row * w * stride), (short)0, w * stride * 2, 0x00020000);
}
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
LGX_D void row_store(__amdgpu_buffer_rsrc_t r, int offset, bf16x4 v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, offset, 0, 0);
}
LGX_D bf16x4 row_load(__amdgpu_buffer_rsrc_t r, int offset) {
  return __builtin_bit_cast(bf16x4, __builtin_amdgcn_raw_buffer_load_b64(r, offset, 0, 0));
}
LGX_D float relu(float v) { return fmaxf(v, 0.f); }  // one instruction; NaN and -0 give +0
// The residual of the inference head at a pixel (the first three of four floats).
LGX_D float4 head_input(const ConvArgs &a, int n, int y, int x) {
  return *(const float4 *)(a.head_in + (((size_t)n * a.h + y) * a.head_in_pitch + x) * a.head_in_floats);
}
// v with the channels zeroed whose mask is not positive (NaN: zeroed)
LGX_D bf16x4 masked(bf16x4 v, bf16x4 m) {
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = bf2f(m[i]) > 0.f ? v[i] : f2bf(0.f);
  return v;
}

// The epilogue of a wave's register tile: WR rows from y0 (uniform) x WP blocks
// of 16 pixels from x0 (lane: pixel col) x MB blocks of 16 channels from co0
// (lane: 4 channels of group kg).  Bias and ReLU, rounded to BF16; then
//  * pool_out: the 2x2 average of the rounded values (rows r, r + 1 are this
//    lane's, columns x, x + 1 are lanes col, col + 1), summed as
//    avgpool_kernel sums: (y, x), (y, x+1), (y+1, x), (y+1, x+1);
//  * UP, channels [0, split): their 2x2 sums in upsample_bwd_kernel's order
//    (the same), masked at half resolution, instead of the full rows;
//  * the rows: channels [0, split) to out0, the rest to out1, zeroed where the
//    mask is not positive.  split is a multiple of 16 (checked on the host),
//    so a block's half is uniform.
// Each value is formed once, columns are checked by the row buffers' range, and
// addresses are a lane offset per pixel block plus constants: with the values
// formed per use and 64-bit addresses per store, the epilogue of a 64-channel
// layer with its pool was 1300 of 1560 VALU instructions a tile, as long as the
// tile's 288 MFMAs.
template <int WR, int WP, int MB, bool UP>
LGX_D void conv_epilogue(const ConvArgs &a, const f32x4 (&acc)[WR][WP][MB], const float (&bias_r)[MB][4], int n, int y0,
                         int x0, int co0, int col, int kg) {
  y0 = __builtin_amdgcn_readfirstlane(y0);
  if (y0 >= a.h) return;
  bf16x4 v[WR][WP][MB];
  if (a.bias) {  // a forward layer: bias and ReLU (checked on the host); uniform
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int pb = 0; pb < WP; pb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          f32x4 f;
#pragma unroll
          for (int i = 0; i < 4; i++) f[i] = relu(acc[r][pb][mb][i] + bias_r[mb][i]);
          v[r][pb][mb] = __builtin_convertvector(f, bf16x4);
        }
  } else {
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int pb = 0; pb < WP; pb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) v[r][pb][mb] = __builtin_convertvector(acc[r][pb][mb], bf16x4);
  }
  const size_t row0 = (size_t)n * a.h + y0;
  if constexpr (WR % 2 == 0) {
    if (a.pool_out || UP) {
      const int hh = a.h >> 1, ww = a.w >> 1, stride = UP ? a.split : a.cout;
      bf16 *const dst = UP ? a.up_out : a.pool_out;
#pragma unroll
      for (int r = 0; r < WR; r += 2) {
        if ((y0 + r) >> 1 >= hh) break;  // uniform
        const size_t hrow = (size_t)n * hh + ((y0 + r) >> 1);
        const __amdgpu_buffer_rsrc_t rs = row_rsrc(dst, hrow, ww, stride);
        const __amdgpu_buffer_rsrc_t ms = row_rsrc(UP ? a.up_mask : dst, hrow, ww, stride);
#pragma unroll
        for (int pb = 0; pb < WP; pb++) {
          const int x = x0 + pb * 16 + col;
          // (odd columns have no pixel here)
          const int at = col & 1 ? (int)0x80000000u : ((x >> 1) * stride + co0 + kg * 4) * 2;
#pragma unroll
          for (int mb = 0; mb < MB; mb++) {
            if (UP && !(co0 + mb * 16 < a.split)) continue;  // uniform
            f32x4 f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const float t = bf2f(v[r][pb][mb][i]), b = bf2f(v[r + 1][pb][mb][i]);
              const float q = ((t + lane_xor1(t)) + b) + lane_xor1(b);
              f[i] = UP ? q : q * 0.25f;
            }
            bf16x4 o = __builtin_convertvector(f, bf16x4);
            if (UP) o = masked(o, row_load(ms, at + mb * 32));
            row_store(rs, at + mb * 32, o);
          }
        }
      }
    }
  }
  // the masks of every row before the stores: for all the compiler knows a
  // store may alias them, and a read after it would wait for its round trip
  const bool any_mask = a.mask0 || a.mask1;
  int at0[WP], at1[WP];  // byte offset of this lane's channels co0.. in a row of out0 / out1
#pragma unroll
  for (int pb = 0; pb < WP; pb++) {
    const int x = x0 + pb * 16 + col;
    at0[pb] = (x * a.split + co0 + kg * 4) * 2;
    at1[pb] = (x * (a.cout - a.split) + co0 - a.split + kg * 4) * 2;
  }
  if (any_mask) {
    bf16x4 m[WR][WP][MB];
#pragma unroll
    for (int r = 0; r < WR; r++)
      if (y0 + r < a.h)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          const bool lo = co0 + mb * 16 < a.split;
          const bf16 *const mask = lo ? a.mask0 : a.mask1;
          if (!mask || (UP && lo)) continue;
          const __amdgpu_buffer_rsrc_t rs = row_rsrc(mask, row0 + r, a.w, lo ? a.split : a.cout - a.split);
#pragma unroll
          for (int pb = 0; pb < WP; pb++) m[r][pb][mb] = row_load(rs, (lo ? at0[pb] : at1[pb]) + mb * 32);
        }
#pragma unroll
    for (int r = 0; r < WR; r++)
      if (y0 + r < a.h)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          const bool lo = co0 + mb * 16 < a.split;
          if (!(lo ? a.mask0 : a.mask1) || (UP && lo)) continue;
#pragma unroll
          for (int pb = 0; pb < WP; pb++) v[r][pb][mb] = masked(v[r][pb][mb], m[r][pb][mb]);
        }
  }
#pragma unroll
  for (int r = 0; r < WR; r++) {
    if (y0 + r >= a.h) break;  // uniform
    const __amdgpu_buffer_rsrc_t r0 = row_rsrc(a.out0, row0 + r, a.w, a.split);
    const __amdgpu_buffer_rsrc_t r1 = row_rsrc(a.out1, row0 + r, a.w, a.cout - a.split);
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const bool lo = co0 + mb * 16 < a.split;  // uniform
      if (UP && lo) continue;                   // stored as 2x2 sums at half resolution
#pragma unroll
      for (int pb = 0; pb < WP; pb++) {
        if (lo)
          row_store(r0, at0[pb] + mb * 32, v[r][pb][mb]);
        else
          row_store(r1, at1[pb] + mb * 32, v[r][pb][mb]);
      }
    }
  }
}

// Forward 3x3 convolution (stride 1, zero padding 1) + bias + ReLU, and the
// same kernel with flipped/transposed weights for the input gradient.
// A wave computes R output rows x PB blocks of 16 pixels x all output
// channels (MB blocks of 16); the 4 waves of a workgroup sit side by side
// along x and share the weight fragments through L1.  Per 32-channel input
// chunk and horizontal tap offset dx, the wave loads the R + 2 input rows it
// needs once and feeds each of them to the three vertical taps, so an
// activation fragment serves up to 3 * MB MFMAs and a weight fragment R * PB.
// Output channels [0, split) go to out0, [split, cout) to out1 (the two
// halves of a concatenated input when computing its gradient); an optional
// mask zeroes outputs whose mask activation is <= 0 (the ReLU derivative of
// the tensor the gradient flows into).
template <int MB, int PB, int R> __global__ __launch_bounds__(256) void conv3x3_kernel(const ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.z, y0 = blockIdx.y * R, x0 = (blockIdx.x * 4 + wave) * (PB * 16);
  // the bias, in LDS for the epilogue (a global read placed after the
  // epilogue's stores would wait for their round trip: they might alias it)
  __shared__ __attribute__((aligned(16))) float s_bias[MB * 16];
  if ((int)threadIdx.x < MB * 16) s_bias[threadIdx.x] = a.bias ? a.bias[threadIdx.x] : 0.f;
  __syncthreads();
  if (x0 >= a.w) return;
  const int col = lane & 15, kg = lane >> 4;
  const int cin = a.ca + a.cb, chunks = cin >> 5;
  f32x4 acc[R][PB][MB];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int pb = 0; pb < PB; pb++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++) acc[r][pb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int cc = 0; cc < chunks; cc++) {
    // the chunk's source is uniform: A (optionally at half resolution) or B
      const bool from_a = cc * 32 < a.ca;
      const bool up = from_a && a.a_up;
    const int cs = from_a ? a.ca : a.cb;
    const int sw = up ? (a.w >> 1) : a.w, sh = up ? (a.h >> 1) : a.h;
    const bf16 *img = (from_a ? a.a : a.b) + (size_t)n * sh * sw * cs + (from_a ? cc * 32 : cc * 32 - a.ca) + kg * 8;
    const bf16 *wchunk = a.wt + ((size_t)cc * a.cout + col) * 32 + kg * 8;
    const size_t wtap = (size_t)chunks * a.cout * 32;
#pragma unroll 1
    for (int dx = -1; dx <= 1; dx++) {
      uint32_t xoff[PB];
      bool xok[PB];
#pragma unroll
      for (int pb = 0; pb < PB; pb++) {
        const int x = x0 + pb * 16 + col + dx;
        xok[pb] = x >= 0 && x < a.w;
        xoff[pb] = (uint32_t)(up ? (x >> 1) : x) * (uint32_t)cs;
      }
      bf16x8 bx[R + 2][PB];
#pragma unroll
      for (int rr = 0; rr < R + 2; rr++) {
        const int yy = y0 - 1 + rr;
        const bool yok = yy >= 0 && yy < a.h;
        const uint32_t roff = (uint32_t)((up ? (yy >> 1) : yy) * sw) * (uint32_t)cs;
#pragma unroll
        for (int pb = 0; pb < PB; pb++) {
          bf16x8 z = {};
          bx[rr][pb] = (yok && xok[pb]) ? *(const bf16x8 *)(img + roff + xoff[pb]) : z;
        }
      }
#pragma unroll
      for (int dy = -1; dy <= 1; dy++) {
        const bf16 *wrow = wchunk + (size_t)((dy + 1) * 3 + (dx + 1)) * wtap;
        bf16x8 aw[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++) aw[mb] = *(const bf16x8 *)(wrow + (size_t)mb * 16 * 32);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
          for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
              acc[r][pb][mb] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[mb], bx[r + 1 + dy][pb], acc[r][pb][mb], 0, 0, 0);
      }
    }
  }
  float bias_r[MB][4];
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const float4 b4 = *(const float4 *)(&s_bias[mb * 16 + kg * 4]);
    bias_r[mb][0] = b4.x;
    bias_r[mb][1] = b4.y;
    bias_r[mb][2] = b4.z;
    bias_r[mb][3] = b4.w;
  }
  conv_epilogue<R, PB, MB, false>(a, acc, bias_r, n, y0, x0, 0, col, kg);
}

// The same convolution with the operands staged in LDS.  A workgroup
// computes a TH = 4*WR row x TW = 16*WP pixel tile for MB*16 output channels
// (a wide layer's channels are split over `splits` tiles), its 4 waves
// stacked vertically.  Per 32-channel input chunk it stages the
// (TH+2) x (TW+2) pixel halo tile (zeros outside the image) and the chunk's
// weights of all 9 taps in LDS; the MFMAs read only LDS while the global
// loads of the next (tile, chunk) are in flight in registers, so global
// latency overlaps the matrix work also across tiles: a workgroup walks
// tiles blockIdx.x, blockIdx.x + gridDim.x, ...  Every output is
// accumulated in the same order as conv3x3_kernel (chunk, dx, dy), so the
// two kernels give bit-identical results.
// With one input chunk and no channel split every tile uses the same
// weights: they stay in LDS from the workgroup's first tile on.

// Raw G-buffer texels of one pixel for the G-buffer-fed first convolution
// (GIN = 1: RG16F normal, RGBA8 albedo; GIN = 2: RG32F, RGBA32F), kept raw
// in registers while in flight and converted when staged.
template <int GIN> struct GinRaw;
template <> struct GinRaw<1> {
  float4 c;
  float d;
  uint32_t n, al;
};
template <> struct GinRaw<2> {
  float4 c;
  float d;
  float2 n;
  float4 al;
};
template <> struct GinRaw<3> {  // the first 9 floats of an input record
  float4 a, b;
  float c;
};
// (GIN = 3 reads image n's records; the G-buffer formats have one image)
template <int GIN> LGX_D GinRaw<GIN> gin_load(const ConvArgs &a, int y, int x, int n = 0) {
  GinRaw<GIN> r;
  if constexpr (GIN == 3) {
    const float *rec = a.gin_x12 + (((size_t)n * a.h + y) * a.w + x) * 12;
    r.a = *(const float4 *)rec;
    r.b = *(const float4 *)(rec + 4);
    r.c = rec[8];
    return r;
  } else {
  r.c = a.gin_noisy[(size_t)y * a.gin_noisy_pitch + x];
  r.d = a.gin_depth[(size_t)y * a.gin_depth_pitch + x];
  if constexpr (GIN == 1) {
    r.n = ((const uint32_t *)a.gin_normal)[(size_t)y * a.gin_normal_pitch + x];
    r.al = ((const uint32_t *)a.gin_albedo)[(size_t)y * a.gin_albedo_pitch + x];
  } else {
    r.n = ((const float2 *)a.gin_normal)[(size_t)y * a.gin_normal_pitch + x];
    r.al = ((const float4 *)a.gin_albedo)[(size_t)y * a.gin_albedo_pitch + x];
  }
  return r;
  }
}
// The first 16 channels of the pixel's input: noisy irradiance rgb, depth, oct
// normal xy, albedo rgb and zeros (a record has 12 floats, the last 3 unused).
template <int GIN> LGX_D void gin_pack(const GinRaw<GIN> &r, bf16x8 &v0, bf16x8 &v1) {
  if constexpr (GIN == 3) {
    v0 = bf16x8{f2bf(r.a.x), f2bf(r.a.y), f2bf(r.a.z), f2bf(r.a.w), f2bf(r.b.x), f2bf(r.b.y), f2bf(r.b.z), f2bf(r.b.w)};
    v1 = bf16x8{};
    v1[0] = f2bf(r.c);
    return;
  } else {
  float nx, ny, ar, ag, ab;
  if constexpr (GIN == 1) {
    nx = h2f((uint16_t)(r.n & 0xffffu));
    ny = h2f((uint16_t)(r.n >> 16));
    const float k = 1.0f / 255.0f;
    ar = (float)(r.al & 0xffu) * k;
    ag = (float)((r.al >> 8) & 0xffu) * k;
    ab = (float)((r.al >> 16) & 0xffu) * k;
  } else {
    nx = r.n.x;
    ny = r.n.y;
    ar = r.al.x;
    ag = r.al.y;
    ab = r.al.z;
  }
  v0 = bf16x8{f2bf(r.c.x), f2bf(r.c.y), f2bf(r.c.z), f2bf(r.d), f2bf(nx), f2bf(ny), f2bf(ar), f2bf(ag)};
  v1 = bf16x8{};
  v1[0] = f2bf(ab);
  }
}

// LDS bytes of conv3x3_lds_kernel<MB, WR, WP> (the layout described in it),
// and the workgroups per CU that LDS allows, at most 3 (168 VGPRs; 4 would
// leave 128, fewer than the tiles' accumulators and operands need): the
// register allocation is held to that occupancy.
constexpr int conv_lds_bytes(int MB, int WR, int WP) {
  return (4 * (((4 * WR + 2) * (16 * WP + 2) * 8 + 127) / 128 * 128) + 4 * 9 * MB * 16 * 8) * 2;
}
constexpr int conv_lds_blocks(int MB, int WR, int WP) {
  return 160 * 1024 / conv_lds_bytes(MB, WR, WP) < 3 ? 160 * 1024 / conv_lds_bytes(MB, WR, WP) : 3;
}

// UP: the epilogue of an input gradient through an upsample (ConvArgs::up_out),
// a separate instantiation so the other convolutions keep their registers.
template <int MB, int WR, int WP, bool UP = false>
__global__ __launch_bounds__(256, conv_lds_blocks(MB, WR, WP)) void conv3x3_lds_kernel(const ConvArgs a, int tiles_x,
                                                                                      int tiles_y, int splits) {
  constexpr int TH = 4 * WR, TW = 16 * WP, IW = TW + 2, IH = TH + 2;
  constexpr int NPIX = IH * IW;                       // input tile pixels (with the halo)
  constexpr int IN_PIECES = (NPIX + 15) / 16 * 16 * 4;  // 16-byte pieces, pixels rounded up to 16
  constexpr int W_PIECES = 9 * MB * 16 * 4;            // of the chunk's weights
  constexpr int IN_PER = (IN_PIECES + 255) / 256, W_PER = (W_PIECES + 255) / 256;
  // LDS layout [channel group kg][pixel or weight row][8 channels], every
  // plane a multiple of 256 bytes (the 64 banks).  A 128-bit LDS access is
  // served 16 lanes at a time, each 8-lane group of a wave with one from
  // the other 16-lane half of its 32 (counters: 2-way conflicts when planes
  // started 16 banks apart, none when 8-lane group g covers bank half
  // g & 1).  Matrix-operand reads (lanes: kg = lane / 16, pixel = lane % 16)
  // therefore put 8-lane groups of different planes on opposite bank halves,
  // and the staging stores use the same rule (see piece()).
  constexpr int PLANE_IN = (NPIX * 8 + 127) / 128 * 128, PLANE_W = 9 * MB * 16 * 8;
  __shared__ __attribute__((aligned(16))) bf16 s_in[4 * PLANE_IN];
  __shared__ __attribute__((aligned(16))) bf16 s_w[4 * PLANE_W];
  static_assert(sizeof(s_in) + sizeof(s_w) == conv_lds_bytes(MB, WR, WP), "LDS layout");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // 16-byte piece q of a tile -> (pixel or weight row, part = channel group):
  // a wave's 64 pieces are 16 consecutive pixels x 4 parts, lane l taking
  // pixel l % 16 of part l / 16 -- the lane pattern of the operand reads
  auto piece = [](int q, int &pix, int &part) {
    pix = ((q >> 6) << 4) + (q & 15);
    part = (q >> 4) & 3;
  };
  const int col = lane & 15, kg = lane >> 4;
  const int chunks = (a.ca + a.cb) >> 5;
  const size_t wtap = (size_t)chunks * a.cout * 32;
  const int T = tiles_x * tiles_y * a.n * splits;
  struct Tile {
    int n, y0, x0, co0;
  };
  // consecutive tile indices: the channel splits of one pixel tile, then x, y, image
  auto tile_of = [&](int t) {
    Tile r;
    r.co0 = (t % splits) * MB * 16;
    int u = t / splits;
    r.x0 = (u % tiles_x) * TW;
    u /= tiles_x;
    r.y0 = (u % tiles_y) * TH;
    r.n = u / tiles_y;
    return r;
  };
  // Loads are unconditional (clamped to an in-image pixel / a valid piece)
  // and padding is applied when staging: a conditional load would make the
  // compiler merge values right after it and wait for the load there,
  // serialising the prefetch with the matrix work.
  bf16x8 pin[IN_PER], pw[W_PER];
  uint32_t valid = 0;  // bit i: piece i of pin lies in the image
  const bool w_resident = chunks == 1 && splits == 1;
  auto fetch = [&](const Tile &tl, int cc, bool with_w) {
    const bool from_a = cc * 32 < a.ca;
    const bool up = from_a && a.a_up;
    const int cs = from_a ? a.ca : a.cb;
    const int sw = up ? (a.w >> 1) : a.w, sh = up ? (a.h >> 1) : a.h;
    const bf16 *img = (from_a ? a.a : a.b) + (size_t)tl.n * sh * sw * cs + (from_a ? cc * 32 : cc * 32 - a.ca);
    valid = 0;
#pragma unroll
    for (int i = 0; i < IN_PER; i++) {
      int p, part;
      piece(min(tid + i * 256, IN_PIECES - 1), p, part);
      p = min(p, NPIX - 1);  // a rounding piece: loaded in bounds, never staged
      const int y = tl.y0 - 1 + p / IW, x = tl.x0 - 1 + p % IW;
      const bool ok = y >= 0 && y < a.h && x >= 0 && x < a.w;
      const int yc = min(max(y, 0), a.h - 1), xc = min(max(x, 0), a.w - 1);
      const uint32_t off = (uint32_t)((up ? (yc >> 1) : yc) * sw + (up ? (xc >> 1) : xc)) * (uint32_t)cs + part * 8;
      pin[i] = *(const bf16x8 *)(img + off);
      valid |= (uint32_t)ok << i;
    }
    if (!with_w) return;
    const bf16 *wsrc = a.wt + ((size_t)cc * a.cout + tl.co0) * 32;
#pragma unroll
    for (int i = 0; i < W_PER; i++) {
      int row, part;
      piece(min(tid + i * 256, W_PIECES - 1), row, part);
      const int tap = row / (MB * 16), co = row % (MB * 16);
      pw[i] = *(const bf16x8 *)(wsrc + tap * wtap + (co * 4 + part) * 8);
    }
  };
  int t = blockIdx.x;
  if (t >= T) return;  // the whole workgroup, before any barrier
  Tile cur = tile_of(t);
  fetch(cur, 0, true);
  bool stage_w = true;  // false once resident weights are staged
  for (;;) {
    f32x4 acc[WR][WP][MB];
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int pb = 0; pb < WP; pb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[r][pb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The tile's bias, read before the matrix work and kept in registers: a
    // global read placed after the tile's stores would wait for their memory
    // round trip (for all the compiler knows they may alias it).  The read is
    // unconditional like the tile loads (a layer without bias reads its
    // weights instead and never adds the values).
    float bias_r[MB][4];
    const float *bsrc = a.bias ? a.bias : (const float *)a.wt;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
      const float4 b4 = *(const float4 *)(bsrc + cur.co0 + mb * 16 + kg * 4);
      bias_r[mb][0] = b4.x;
      bias_r[mb][1] = b4.y;
      bias_r[mb][2] = b4.z;
      bias_r[mb][3] = b4.w;
    }
    for (int cc = 0; cc < chunks; cc++) {
#pragma unroll
      for (int i = 0; i < IN_PER; i++) {
        const int q = tid + i * 256;
        const bf16x8 z = {};
        int p, part;
        piece(q, p, part);
        if (q < IN_PIECES && p < NPIX) *(bf16x8 *)(s_in + part * PLANE_IN + p * 8) = ((valid >> i) & 1u) ? pin[i] : z;
      }
      if (stage_w) {
#pragma unroll
        for (int i = 0; i < W_PER; i++) {
          const int q = tid + i * 256;
          int row, part;
          piece(q, row, part);
          if (q < W_PIECES) *(bf16x8 *)(s_w + part * PLANE_W + row * 8) = pw[i];
        }
        stage_w = !w_resident;
      }
      __syncthreads();
      // in flight during the matrix work below: the next chunk, or the next tile's first
      if (cc + 1 < chunks)
        fetch(cur, cc + 1, true);
      else if (t + (int)gridDim.x < T)
        fetch(tile_of(t + (int)gridDim.x), 0, !w_resident);
#pragma unroll
      for (int dx = 0; dx < 3; dx++) {
        bf16x8 bx[WR + 2][WP];
#pragma unroll
        for (int rr = 0; rr < WR + 2; rr++)
#pragma unroll
          for (int pb = 0; pb < WP; pb++)
            bx[rr][pb] = *(const bf16x8 *)(s_in + kg * PLANE_IN + ((wave * WR + rr) * IW + pb * 16 + col + dx) * 8);
#pragma unroll
        for (int dy = 0; dy < 3; dy++) {
          const int tap = dy * 3 + dx;
          bf16x8 aw[MB];
#pragma unroll
          for (int mb = 0; mb < MB; mb++)
            aw[mb] = *(const bf16x8 *)(s_w + kg * PLANE_W + ((tap * MB + mb) * 16 + col) * 8);
#pragma unroll
          for (int r = 0; r < WR; r++)
#pragma unroll
            for (int pb = 0; pb < WP; pb++)
#pragma unroll
              for (int mb = 0; mb < MB; mb++)
                acc[r][pb][mb] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[mb], bx[r + dy][pb], acc[r][pb][mb], 0, 0, 0);
        }
      }
      __syncthreads();  // the next stash overwrites the tiles
    }
    conv_epilogue<WR, WP, MB, UP>(a, acc, bias_r, cur.n, cur.y0 + wave * WR, cur.x0, cur.co0, col, kg);
    t += gridDim.x;
    if (t >= T) break;
    cur = tile_of(t);
  }
}

// conv_epilogue for a tile whose channel blocks are paired: the 16 rows of block
// mb are channels 32 (mb / 2) + 8 kg + 4 (mb & 1) + i, so a lane holds 8
// consecutive channels of a pixel in two blocks and a pixel's 32 channels are
// one 64-byte run of four lanes' 16-byte stores (8-byte stores wrote 32-byte
// runs, twice as many).  Every store is issued (rows past the image go to an
// empty buffer): at least kStores, which the caller's wait counts on.
template <int WR, int WP, int MB, bool UP> constexpr int epilogue_stores() {
  return WR * WP * MB / 2 / (UP ? 2 : 1);
}
// The channel of a row of block mb.  Pairs from 64 channels a workgroup on (128
// bytes a pixel: 45 us against 58 for the 1080p layer 64 + 64 -> 64); with 32
// channels the 8-byte stores are the faster ones (67 us against 76 for the
// full-size 32 -> 32 layer, 125 against 142 for 96 -> 32).
constexpr bool conv_pairs(int MB) { return MB % 4 == 0; }
LGX_D int pair_row(bool pairs, int mb, int row) {
  return pairs ? (mb >> 1) * 32 + (row >> 2) * 8 + (mb & 1) * 4 + (row & 3) : mb * 16 + row;
}
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
LGX_D void row_store8(__amdgpu_buffer_rsrc_t r, int offset, bf16x8 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, offset, 0, 0);
}
LGX_D bf16x8 row_load8(__amdgpu_buffer_rsrc_t r, int offset) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, 0));
}
LGX_D bf16x8 masked8(bf16x8 v, bf16x8 m) {
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = bf2f(m[i]) > 0.f ? v[i] : f2bf(0.f);
  return v;
}
// Element i (a constant) as a float, from the packed words: the compiler turns bf2f(v[i]) of a converted
// vector into a conversion of that element of its own.
LGX_D float unpack8(bf16x8 v, int i) {
  const uint32_t u = __builtin_bit_cast(u32x4, v)[i >> 1];
  return __builtin_bit_cast(float, i & 1 ? u & 0xffff0000u : u << 16);
}
template <int WR, int WP, int MB, bool UP>
LGX_D void conv_epilogue_pairs(const ConvArgs &a, const f32x4 (&acc)[WR][WP][MB], const float (&bias_r)[MB][4], int n,
                               int y0, int x0, int co0, int col, int kg) {
  constexpr int MP = MB / 2;
  y0 = __builtin_amdgcn_readfirstlane(y0);
  bf16x8 v[WR][WP][MP];
#pragma unroll
  for (int r = 0; r < WR; r++)
#pragma unroll
    for (int pb = 0; pb < WP; pb++)
#pragma unroll
      for (int mp = 0; mp < MP; mp++) {
        f32x8 f;
        if (a.bias) {  // a forward layer: bias and ReLU (checked on the host); uniform
#pragma unroll
          for (int i = 0; i < 8; i++) f[i] = relu(acc[r][pb][2 * mp + (i >> 2)][i & 3] + bias_r[2 * mp + (i >> 2)][i & 3]);
        } else {
#pragma unroll
          for (int i = 0; i < 8; i++) f[i] = acc[r][pb][2 * mp + (i >> 2)][i & 3];
        }
        v[r][pb][mp] = __builtin_convertvector(f, bf16x8);
      }
  const size_t row0 = (size_t)n * a.h + y0;
  if constexpr (WR % 2 == 0) {
    if (a.pool_out || UP) {
      const int hh = a.h >> 1, ww = a.w >> 1, stride = UP ? a.split : a.cout;
      bf16 *const dst = UP ? a.up_out : a.pool_out;
#pragma unroll
      for (int r = 0; r < WR; r += 2) {
        const bool in = (y0 + r) >> 1 < hh;  // uniform
        const size_t hrow = in ? (size_t)n * hh + ((y0 + r) >> 1) : 0;
        const __amdgpu_buffer_rsrc_t rs = row_rsrc(dst, hrow, in ? ww : 0, stride);
        const __amdgpu_buffer_rsrc_t ms = row_rsrc(UP ? a.up_mask : dst, hrow, in ? ww : 0, stride);
#pragma unroll
        for (int pb = 0; pb < WP; pb++) {
          const int x = x0 + pb * 16 + col;
          // (odd columns have no pixel here)
          const int at = col & 1 ? (int)0x80000000u : ((x >> 1) * stride + co0 + kg * 8) * 2;
#pragma unroll
          for (int mp = 0; mp < MP; mp++) {
            if (UP && !(co0 + mp * 32 < a.split)) continue;  // uniform
            f32x8 f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
              const float t = bf2f(v[r][pb][mp][i]), b = bf2f(v[r + 1][pb][mp][i]);
              const float q = ((t + lane_xor1(t)) + b) + lane_xor1(b);
              f[i] = UP ? q : q * 0.25f;
            }
            bf16x8 o = __builtin_convertvector(f, bf16x8);
            if (UP) o = masked8(o, row_load8(ms, at + mp * 64));
            row_store8(rs, at + mp * 64, o);
          }
        }
      }
    }
  }
  int at0[WP], at1[WP];  // byte offset of this lane's channels co0.. in a row of out0 / out1
#pragma unroll
  for (int pb = 0; pb < WP; pb++) {
    const int x = x0 + pb * 16 + col;
    at0[pb] = (x * a.split + co0 + kg * 8) * 2;
    at1[pb] = (x * (a.cout - a.split) + co0 - a.split + kg * 8) * 2;
  }
  if (a.mask0 || a.mask1) {  // all masks before the stores (a read after a store would wait for its round trip)
    bf16x8 m[WR][WP][MP];
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int mp = 0; mp < MP; mp++) {
        const bool lo = co0 + mp * 32 < a.split;
        const bf16 *const mask = lo ? a.mask0 : a.mask1;
        if (!mask || (UP && lo)) continue;
        const bool in = y0 + r < a.h;
        const __amdgpu_buffer_rsrc_t rs = row_rsrc(mask, in ? row0 + r : 0, in ? a.w : 0, lo ? a.split : a.cout - a.split);
#pragma unroll
        for (int pb = 0; pb < WP; pb++) m[r][pb][mp] = row_load8(rs, (lo ? at0[pb] : at1[pb]) + mp * 64);
      }
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int mp = 0; mp < MP; mp++) {
        const bool lo = co0 + mp * 32 < a.split;
        if (!(lo ? a.mask0 : a.mask1) || (UP && lo)) continue;
#pragma unroll
        for (int pb = 0; pb < WP; pb++) v[r][pb][mp] = masked8(v[r][pb][mp], m[r][pb][mp]);
      }
  }
#pragma unroll
  for (int r = 0; r < WR; r++) {
    const bool in = y0 + r < a.h;
    const __amdgpu_buffer_rsrc_t r0 = row_rsrc(a.out0, in ? row0 + r : 0, in ? a.w : 0, a.split);
    const __amdgpu_buffer_rsrc_t r1 = row_rsrc(a.out1, in ? row0 + r : 0, in ? a.w : 0, a.cout - a.split);
#pragma unroll
    for (int mp = 0; mp < MP; mp++) {
      const bool lo = co0 + mp * 32 < a.split;  // uniform
      if (UP && lo) continue;                   // stored as 2x2 sums at half resolution
#pragma unroll
      for (int pb = 0; pb < WP; pb++) {
        if (lo)
          row_store8(r0, at0[pb] + mp * 64, v[r][pb][mp]);
        else
          row_store8(r1, at1[pb] + mp * 64, v[r][pb][mp]);
      }
    }
  }
}

// The same convolution with its operands moved to LDS by direct loads
// (buffer_load ... lds: no registers and no LDS store instructions).  A
// workgroup of NW waves computes NW WR rows x 16 WP pixels for MB 16-channel
// blocks and walks tiles; while the MFMAs read one input buffer the next
// stage (the tile's next 32-channel chunk, or the next tile's first) lands in
// the other, with one barrier a stage.  Weights of all chunks stay in LDS
// when they fit (wres), else they move with their chunk.
//
// LDS layout: 64 bytes a pixel (or output channel), the 16-byte channel group g
// of pixel p in place g ^ 2 (p / 4 % 2).  A wave's direct load fills 1 KB, four
// lanes to a pixel, so it reads whole 64-byte runs of memory (with a pixel's
// groups 16 lanes apart, each lane of a quad read another cache line); the
// exchange of places puts the lanes of an operand read that are served
// together (8 of one group and the 8 others of the next one) on all 64 banks
// from any first pixel; g ^ (p / 4 % 4) does so only from every fourth, and
// half of the LDS cycles were conflicts (96 -> 32 at 1080p 131 us, now 126).
// Pixels outside the image are offsets outside the buffer, which load as zeros.  Accumulation order is conv3x3_kernel's.
//
// What bounds it: the epilogue and the outputs' stores (about 40 % of a layer;
// without them 64 -> 64 at 960 x 540 takes 33 us instead of 46), then the matrix
// work; the input loads are hidden.  conv3x3_lds_kernel holds the next stage
// in registers, which the wide tiles do not have to spare, and issues every
// element's LDS store: at 960 x 540 its best tile takes 63 us for 64 -> 64
// against 45 here, 113 against 91 for 192 -> 64 and 57 against 40 for 128 -> 64,
// at 480 x 270 47 against 36 for 128 -> 128.
constexpr int dma_in_blocks(int WR, int WP, int NW) { return ((NW * WR + 2) * (16 * WP + 2) + 15) / 16; }
constexpr int dma_act_bytes(int WR, int WP, int NW, bool head) { return head ? NW * WR * WP * 16 * 64 + 512 : 0; }
// LDS bytes with `slots` weight chunks
constexpr int dma_lds_bytes(int MB, int WR, int WP, int NW, bool head, int slots) {
  return (2 * dma_in_blocks(WR, WP, NW) + 9 * MB * slots) * 1024 + dma_act_bytes(WR, WP, NW, head);
}

template <int MB, int WR, int WP, int NW, int OCC, bool HEAD, bool UP>
__global__ __launch_bounds__(64 * NW, OCC) void conv3x3_dma_kernel(const ConvArgs a, int tiles_x, int tiles_y, int splits,
                                                                   int wres) {
  constexpr int TH = NW * WR, TW = 16 * WP, IW = TW + 2, IH = TH + 2, NPIX = IH * IW;
  constexpr int NBLK = (NPIX + 15) / 16, NI = (NBLK + NW - 1) / NW, WBLK = 9 * MB, NJ = (WBLK + NW - 1) / NW;
  constexpr bool PAIRS = conv_pairs(MB);
  extern __shared__ __align__(16) char s_dma[];
  char *const s_w = s_dma + 2 * NBLK * 1024;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kg = lane >> 4;
  const int chunks = (a.ca + a.cb) >> 5;
  typedef __attribute__((address_space(3))) void LdsVoid;
  const uint32_t logical = xcd_remap(blockIdx.x, gridDim.x);
  const int co0 = (int)(logical % (uint32_t)splits) * MB * 16, step = (int)gridDim.x / splits;
  const int T = tiles_x * tiles_y * a.n;
  int t = (int)(logical / (uint32_t)splits);
  if (t >= T) return;  // the whole workgroup, before any barrier
  struct Tile {
    int n, y0, x0;
  };
  auto tile_of = [&](int u) {
    Tile r;
    r.x0 = (u % tiles_x) * TW;
    u /= tiles_x;
    r.y0 = (u % tiles_y) * TH;
    r.n = u / tiles_y;
    return r;
  };
  // this lane's pixel of the wave's i-th input block (row, column of the halo tile) and its channel group
  const int part = ((lane & 3) ^ (lane >> 4 & 1) * 2) * 16;
  int prow[NI], pcol[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int p = (wave + NW * i) * 16 + (lane >> 2);
    prow[i] = p < NPIX ? p / IW : 1 << 20;  // a pixel past the tile: outside every image
    pcol[i] = p % IW;
  }
  // byte offsets of the wave's pieces in the source of chunk cc (a chunk of the
  // same tile and source only moves the base), then the loads
  uint32_t voff[NI];
  auto dma_in = [&](int buf, const Tile &tl, int cc) {
    const bool from_a = cc * 32 < a.ca;
    const int up = from_a && a.a_up ? 1 : 0;
    const int cs = from_a ? a.ca : a.cb;
    const int sw = a.w >> up, sh = a.h >> up;
    const int yb = max(tl.y0 - 1, 0) >> up;  // offsets count from the tile's first row
    const int ch = from_a ? cc * 32 : cc * 32 - a.ca;
    const bf16 *base = (from_a ? a.a : a.b) + ((size_t)tl.n * sh + yb) * sw * cs + ch;
    const size_t left = ((size_t)(sh - yb) * sw * cs - ch) * 2;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)base, (short)0, (int)(left < 0x7fffffffu ? left : 0x7fffffffu), 0x00020000);
    if (cc == 0 || cc * 32 == a.ca) {
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const int y = tl.y0 - 1 + prow[i], x = tl.x0 - 1 + pcol[i];
        const bool ok = (uint32_t)y < (uint32_t)a.h && (uint32_t)x < (uint32_t)a.w;
        const uint32_t off = (uint32_t)(((y >> up) - yb) * sw + (x >> up)) * (uint32_t)(cs * 2) + (uint32_t)part;
        voff[i] = ok ? off : 0x80000000u;
      }
    }
#pragma unroll
    for (int i = 0; i < NI; i++)
      if (wave + NW * i < NBLK)  // uniform
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsVoid *)(s_dma + (buf * NBLK + wave + NW * i) * 1024), 16,
                                                 (int)voff[i], 0, 0, 0);
  };
  const __amdgpu_buffer_rsrc_t wrs =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.wt, (short)0, 9 * chunks * a.cout * 64, 0x00020000);
  const int wrow = pair_row(PAIRS, 0, lane >> 2) * 64;  // (block mb: pair_row(PAIRS, mb, 0) rows on)
  auto dma_w = [&](int slot, int cc) {
#pragma unroll
    for (int i = 0; i < NJ; i++) {
      const int b = wave + NW * i;
      if (b >= WBLK) continue;  // uniform
      const int tap = b / MB, mb = b % MB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (LdsVoid *)(s_w + (slot * WBLK + b) * 1024), 16,
                                               wrow + part, ((tap * chunks + cc) * a.cout + co0 + pair_row(PAIRS, mb, 0)) * 64, 0, 0);
    }
  };
  // LDS offset of the input operand at pixel (wave WR + rr) IW + dx + col, group kg; 16 pixels on is 1 KB on
  int in_off[WR + 2][3];
#pragma unroll
  for (int rr = 0; rr < WR + 2; rr++)
#pragma unroll
    for (int dx = 0; dx < 3; dx++) {
      const int p = (wave * WR + rr) * IW + dx + col;
      in_off[rr][dx] = p * 64 + (kg ^ (p >> 2 & 1) * 2) * 16;
    }
  Tile cur = tile_of(t);
  char *const s_act = s_w + (wres ? chunks : 2) * WBLK * 1024;
  // the head's weights and bias, in LDS: read from memory they would wait behind the next stage's loads
  float *const s_head = (float *)(s_act + NW * WR * TW * 64);
  if (HEAD && threadIdx.x < 99) s_head[threadIdx.x] = threadIdx.x < 96 ? a.head_w[threadIdx.x] : a.head_b[threadIdx.x - 96];
  if (wres)
    for (int cc = 0; cc < chunks; cc++) dma_w(cc, cc);
  else
    dma_w(0, 0);
  float bias_r[MB][4];
  const float *bsrc = a.bias ? a.bias : (const float *)a.wt;  // (never added without a bias)
#pragma unroll
  for (int mb = 0; mb < MB; mb++) {
    const float4 b4 = *(const float4 *)(bsrc + co0 + pair_row(PAIRS, mb, kg * 4));
    bias_r[mb][0] = b4.x;
    bias_r[mb][1] = b4.y;
    bias_r[mb][2] = b4.z;
    bias_r[mb][3] = b4.w;
  }
  dma_in(0, cur, 0);
  __syncthreads();  // (waits for the loads)
  int buf = 0;
  for (;;) {
    f32x4 acc[WR][WP][MB];
#pragma unroll
    for (int r = 0; r < WR; r++)
#pragma unroll
      for (int pb = 0; pb < WP; pb++)
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[r][pb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int tn = t + step;
    // HEAD: this lane's pixels (lane, lane + 64, .. of the wave's), their residuals ahead of the next stage's loads
    constexpr int NP = HEAD ? WR * TW / 64 : 1;
    float4 head_c[NP];
    if constexpr (HEAD)
#pragma unroll
      for (int k = 0; k < NP; k++) {
        const int p = lane + k * 64, y = min(cur.y0 + wave * WR + p / TW, a.h - 1), x = min(cur.x0 + p % TW, a.w - 1);
        head_c[k] = head_input(a, cur.n, y, x);
      }
    for (int cc = 0; cc < chunks; cc++) {
      // the next stage into the other buffer: every wave is past the barrier that ended its last use
      const bool more = cc + 1 < chunks || tn < T;
      if (more) {
        const int nc = cc + 1 < chunks ? cc + 1 : 0;
        dma_in(buf ^ 1, cc + 1 < chunks ? cur : tile_of(tn), nc);
        if (!wres) dma_w(buf ^ 1, nc);
      }
      const char *in = s_dma + buf * NBLK * 1024;
      const char *w = s_w + (wres ? cc : buf) * WBLK * 1024 + col * 64 + (kg ^ (col >> 2 & 1) * 2) * 16;
      // Taps in the order (dx, dy).  The operands of a tap are read while the
      // previous one's MFMAs run: its weights, and the next column's rows a
      // third at a time.  (Left to the compiler the reads sit right before
      // their use, and every tap waits for LDS.)
      constexpr int ROWS = WR + 2;
      bf16x8 bx[2][ROWS][WP], aw[2][MB];
      auto read_row = [&](int dx, int rr) {
#pragma unroll
        for (int pb = 0; pb < WP; pb++) bx[dx & 1][rr][pb] = *(const bf16x8 *)(in + in_off[rr][dx] + pb * 1024);
      };
      auto read_w = [&](int s) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
          aw[s & 1][mb] = *(const bf16x8 *)(w + (((s % 3) * 3 + s / 3) * MB + mb) * 1024);
      };
      read_w(0);
#pragma unroll
      for (int rr = 0; rr < ROWS; rr++) read_row(0, rr);
#pragma unroll
      for (int s = 0; s < 9; s++) {
        const int dx = s / 3, dy = s % 3;
        if (s + 1 < 9) read_w(s + 1);
        if (dx + 1 < 3) {
#pragma unroll
          for (int rr = dy * ROWS / 3; rr < (dy + 1) * ROWS / 3; rr++) read_row(dx + 1, rr);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < WR; r++)
#pragma unroll
          for (int pb = 0; pb < WP; pb++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
              acc[r][pb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[s & 1][mb], bx[dx & 1][r + dy][pb],
                                                                       acc[r][pb][mb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (cc + 1 == chunks) {
        if constexpr (HEAD) {
          // the inference head: each wave's activations (BF16, as the unfused
          // path stores them) through LDS of its own, then a lane per pixel
          // forms in + b + W act, channel by channel.  1920 x 1080: 65 us, 55
          // without the head (the residual's read is waited for before the
          // tile's first MFMA); with 80 bytes a pixel in LDS only one
          // workgroup fits a CU (108), and with the head's weights read
          // from memory per tile, behind the next stage's loads, 118.
          static_assert(!HEAD || (MB == 2 && WR * WP % 4 == 0), "a lane per pixel");
          char *act = s_act + wave * (WR * TW * 64);
#pragma unroll
          for (int r = 0; r < WR; r++)
#pragma unroll
            for (int pb = 0; pb < WP; pb++)
#pragma unroll
              for (int mb = 0; mb < MB; mb++) {
                typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
                bf16x4 o;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                  const float v = acc[r][pb][mb][i] + bias_r[mb][i];
                  o[i] = f2bf(v > 0.f ? v : 0.f);
                }
                // (the 16-byte place of channels 8 c .. 8 c + 7 of pixel p is c ^ (p / 4 % 4))
                *(bf16x4 *)(act + (r * TW + pb * 16 + col) * 64 + ((mb * 2 + (kg >> 1)) ^ (col >> 2)) * 16 + (kg & 1) * 8) = o;
              }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          // (a buffer from the wave's first row: one store a pixel whatever lies outside, which the wait counts on)
          const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
              (void *)(a.head_out + ((size_t)cur.n * a.h + cur.y0 + wave * WR) * a.head_out_pitch), (short)0, 0x7fffffff,
              0x00020000);
#pragma unroll
          for (int k = 0; k < NP; k++) {
            const int p = lane + k * 64, r = p / TW, x = cur.x0 + p % TW;
            const float4 c = head_c[k];
            const f32x4 hb = *(const f32x4 *)(s_head + 96);
            float o[3] = {c.x + hb[0], c.y + hb[1], c.z + hb[2]};
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const bf16x8 v = *(const bf16x8 *)(act + p * 64 + (q ^ (p >> 2 & 3)) * 16);
              f32x4 hw[3][2];
#pragma unroll
              for (int k3 = 0; k3 < 3; k3++)
#pragma unroll
                for (int i = 0; i < 2; i++) hw[k3][i] = *(const f32x4 *)(s_head + k3 * 32 + q * 8 + i * 4);
#pragma unroll
              for (int i = 0; i < 8; i++) {
                const float f = bf2f(v[i]);
#pragma unroll
                for (int k3 = 0; k3 < 3; k3++) o[k3] += hw[k3][i >> 2][i & 3] * f;
              }
            }
            const f32x4 out = {o[0], o[1], o[2], 1.f};
            const bool in = cur.y0 + wave * WR + r < a.h && x < a.w;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, out), rs,
                                                   in ? (r * a.head_out_pitch + x) * 16 : (int)0x80000000u, 0, 0);
          }
        } else {
          if constexpr (PAIRS)
            conv_epilogue_pairs<WR, WP, MB, UP>(a, acc, bias_r, cur.n, cur.y0 + wave * WR, cur.x0, co0, col, kg);
          else
            conv_epilogue<WR, WP, MB, UP>(a, acc, bias_r, cur.n, cur.y0 + wave * WR, cur.x0, co0, col, kg);
        }
      }
      if (more) {  // the next stage has landed, and every wave has read this one
        // A wait for the direct loads alone: the epilogue's stores were issued
        // after them (memory operations of a wave retire from this counter in
        // order), and waiting for those too would hold every tile for a
        // store's round trip.  (conv_epilogue skips rows past the image: no count.)
        if (cc + 1 < chunks || (!PAIRS && !HEAD))
          asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        else if constexpr (HEAD)
          asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NP) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(epilogue_stores<WR, WP, MB, UP>()) : "memory");
      }
      buf ^= 1;
    }
    if (tn >= T) break;
    t = tn;
    cur = tile_of(t);
  }
}

// The first two convolutions in one kernel (inference and the training
// forward): the first one's output goes to HBM only when the backward pass
// needs it, which is about half of the two layers' traffic.
//
// One wave is one workgroup and walks down a strip 30 output columns wide,
// two rows an iteration: the strip's records (34 columns, packed from the
// G-buffer or the FP32 records by gin_pack) and the first
// layer's output (32 columns, two 16-pixel blocks) live in LDS rings of four
// rows, so each row of either is formed once, and nothing waits at a
// barrier.  A strip is cut into segments of `len` row pairs so that there are
// about as many waves as fit the chip; a segment forms two extra rows of the
// first layer.
//
// First layer: its records have 9 channels, padded to 16, so one tap per
// 32-deep MFMA would leave half of K zero; here taps 2p and 2p + 1 share an
// MFMA (k = 16 * (tap & 1) + channel; the tenth tap is zero): 5 MFMAs per
// output block instead of 9.  (conv3x3 on the packed records, one tap per
// MFMA, rounds the partial sums differently.)  Second layer: conv3x3's order
// (dx, dy), its weights in registers, with the 2x2 pool.
//
// What bounds it: issue.  An iteration has 112 MFMAs (1800 cycles) and 350 other
// vector instructions, which the two waves of a SIMD overlap in part.  From
// the G-buffer at 1920 x 1080: 71 us, where 225 MB of traffic take 44 at a
// copy's rate; with workgroups of four waves that staged an 8 x 32 tile,
// formed its halo and met at two barriers a tile, 141.  From records with
// both layers kept (16 x 256 x 256): 60 us for 270 MB, 81 before.
//
// LDS: two halves (8 KB apart) of two rows each; iteration k writes half k & 1
// and reads both.  In a half: records, [plane of 8 channels][row][pixel],
// then first-layer outputs, the same with four planes; planes are 1280 bytes
// (a multiple of the banks, as in conv3x3_lds_kernel), rows 640.
constexpr int kPairCols = 30;           // output columns of a strip
constexpr int kPairRow = 640, kPairPlane = 2 * kPairRow, kPairOut = 2 * kPairPlane, kPairHalf = 8192;
// zeros the tenth tap reads (with its zero weights: no 0 * inf), at row and block steps of 640 and 256 bytes
constexpr int kPairZero = 2 * kPairHalf;
template <int GIN, bool KEEP>
__global__ __launch_bounds__(64, 2) void conv_first_pair_kernel(const ConvArgs a0, const ConvArgs a1, int strips,
                                                                int segs, int len) {
  __shared__ __attribute__((aligned(256))) char s[2 * kPairHalf + 1024];
  const int lane = threadIdx.x, col = lane & 15, kg = lane >> 4;
  const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
  const int x0 = (int)(id % (uint32_t)strips) * kPairCols, seg = (int)(id / (uint32_t)strips) % segs,
            n = (int)(id / (uint32_t)(strips * segs));
  const int ys = seg * len * 2, pairs = min(len, (a0.h + 1) / 2 - seg * len), h = a0.h, w = a0.w;
  const bf16x8 zero8 = {};
  // First-layer weights: the A operand of pair p, block mb holds tap 2p + (kg >> 1), channels 8 * (kg & 1)
  // .. + 7; its rows are ordered (pair_row) so that a lane's outputs are channels 8 kg .. 8 kg + 7.
  bf16x8 w0[5][2], w1[9][2];
#pragma unroll
  for (int p = 0; p < 5; p++)
#pragma unroll
    for (int mb = 0; mb < 2; mb++) {
      const int tap = 2 * p + (kg >> 1);
      w0[p][mb] = tap < 9 ? *(const bf16x8 *)(a0.wt + ((size_t)tap * 32 + pair_row(true, mb, col)) * 32 + (kg & 1) * 8)
                          : zero8;
    }
#pragma unroll
  for (int tap = 0; tap < 9; tap++)
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
      w1[tap][mb] = *(const bf16x8 *)(a1.wt + ((size_t)tap * 32 + pair_row(true, mb, col)) * 32 + kg * 8);
  // A first-layer column outside the image has bias -inf: ReLU makes every sum (NaN, too) the zero that the
  // second layer's padding is.
  float bias0[2][8], bias1[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float b = a0.bias[kg * 8 + i];
#pragma unroll
    for (int pb = 0; pb < 2; pb++) {
      const int x = x0 - 1 + pb * 16 + col;
      bias0[pb][i] = x >= 0 && x < w ? b : -INFINITY;
    }
    bias1[i] = a1.bias[kg * 8 + i];
  }
  // this lane's record column (lanes past 33 repeat the last and store nothing)
  const int rpx = min(lane, 33), rx = x0 - 2 + rpx, rxc = min(max(rx, 0), w - 1);
  const bool rx_in = rx >= 0 && rx < w;
  GinRaw<GIN> raw[2];
  auto fetch = [&](int y) {  // rows y, y + 1 (clamped into the image)
#pragma unroll
    for (int i = 0; i < 2; i++) raw[i] = gin_load<GIN>(a0, min(max(y + i, 0), h - 1), rxc, n);
  };
  // rows y, y + 1 into a half: zero outside the image (the first layer's padding); a segment's own pixels
  // also to rec_out when asked (32 channels, the upper 16 zero: the training backward reads them)
  auto stage = [&](int y, int half, bool own) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const bool in = rx_in && y + i >= 0 && y + i < h;
      bf16x8 v0, v1;
      gin_pack<GIN>(raw[i], v0, v1);
      v0 = in ? v0 : zero8;
      v1 = in ? v1 : zero8;
      if (lane < 34) {
        *(bf16x8 *)(s + half + i * kPairRow + rpx * 16) = v0;
        *(bf16x8 *)(s + half + kPairPlane + i * kPairRow + rpx * 16) = v1;
      }
    }
    if constexpr (KEEP) {  // four lanes a pixel, 16 pixels a store, so that a store is one run of memory
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const int part = lane & 3, px = 2 + (lane >> 2);
      const char *from = part < 2 ? s + half + part * kPairPlane + px * 16 : s + kPairZero;
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const bool in = own && y + i < h;
        const __amdgpu_buffer_rsrc_t rs = row_rsrc(a0.rec_out, in ? (size_t)n * h + y + i : 0, in ? w : 0, 32);
#pragma unroll
        for (int j = 0; j < 2; j++)
          row_store8(rs, px + j * 16 < 2 + kPairCols ? (x0 - 2 + px + j * 16) * 64 + part * 16 : (int)0x80000000u,
                     *(const bf16x8 *)(from + i * kPairRow + j * 256));
      }
    }
  };
  // this lane's kept first-layer columns (1 .. 30, the strip's own) in a row of out0
  int keep_at[2];
#pragma unroll
  for (int pb = 0; pb < 2; pb++) {
    const int c = pb * 16 + col, x = x0 - 1 + c;
    keep_at[pb] = c >= 1 && c <= kPairCols ? x * 64 + kg * 16 : (int)0x80000000u;
  }
  // First layer, rows y (from record rows lo 0, lo 1, hi 0) and y + 1 (lo 1, hi 0, hi 1), to half hi.
  auto first = [&](int y, int lo, int hi, bool own0, bool own1) {
    const int lane_off = col * 16 + (kg & 1) * kPairPlane;
    const int up = kg >> 1;  // the upper tap of a pair
    const char *const alo = s + lo + lane_off + up * 16, *const ahi = s + hi + lane_off + up * 16;
    // taps 2 and 3: (row, dx 2) and (row + 1, dx 0)
    const char *const b0 = s + lo + lane_off + (up ? kPairRow : 32);
    const char *const b1 = s + lane_off + (up ? hi : lo + kPairRow + 32);
    const char *const c8 = up ? s + kPairZero : ahi + 32;
    auto operand = [&](int st, int pb) {
      const int p = st >> 1, r = st & 1;
      const char *at;
      if (p == 0) at = alo + r * kPairRow;                       // taps 0, 1: row r
      else if (p == 1) at = r ? b1 : b0;                         // taps 2, 3
      else if (p == 2) at = r ? ahi + 16 : alo + kPairRow + 16;  // taps 4, 5: row r + 1
      else if (p == 3) at = ahi + r * kPairRow;                  // taps 6, 7: row r + 2
      else at = c8 + r * kPairRow;                               // tap 8 and, in the upper lanes, zeros
      return *(const bf16x8 *)(at + pb * 256);
    };
    f32x4 acc[2][2][2];
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int pb = 0; pb < 2; pb++)
#pragma unroll
        for (int mb = 0; mb < 2; mb++) acc[r][pb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int D = 4;
    bf16x8 bx[D][2];
#pragma unroll
    for (int st = 0; st < D - 1; st++)
#pragma unroll
      for (int pb = 0; pb < 2; pb++) bx[st][pb] = operand(st, pb);
#pragma unroll
    for (int st = 0; st < 10; st++) {
      if (st + D - 1 < 10)
#pragma unroll
        for (int pb = 0; pb < 2; pb++) bx[(st + D - 1) % D][pb] = operand(st + D - 1, pb);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int pb = 0; pb < 2; pb++) {
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
          acc[st & 1][pb][mb] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[st >> 1][mb], bx[st % D][pb], acc[st & 1][pb][mb], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // bias, ReLU, BF16 (conv_epilogue's rounding), zero outside the image (the second layer's padding)
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const bool row_in = y + r >= 0 && y + r < h;
      const bool own = KEEP && (r ? own1 : own0) && row_in;
      const __amdgpu_buffer_rsrc_t rs = row_rsrc(KEEP ? a0.out0 : nullptr, own ? (size_t)n * h + y + r : 0, own ? w : 0, 32);
      bf16x8 v[2];
#pragma unroll
      for (int pb = 0; pb < 2; pb++) {
        f32x8 f;
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = relu(acc[r][pb][i >> 2][i & 3] + bias0[pb][i]);
        v[pb] = __builtin_convertvector(f, bf16x8);
      }
      if (!row_in) v[0] = v[1] = zero8;
#pragma unroll
      for (int pb = 0; pb < 2; pb++) {
        *(bf16x8 *)(s + hi + kPairOut + kg * kPairPlane + r * kPairRow + (pb * 16 + col) * 16) = v[pb];
        if (KEEP) row_store8(rs, keep_at[pb], v[pb]);
      }
    }
  };
  // this lane's output columns (30 of 32) in the rows of the output and of the pool
  int out_at[2], pool_at[2];
#pragma unroll
  for (int pb = 0; pb < 2; pb++) {
    const int c = pb * 16 + col, x = x0 + c;
    out_at[pb] = c < kPairCols ? x * 64 + kg * 16 : (int)0x80000000u;
    pool_at[pb] = c < kPairCols && !(col & 1) ? (x >> 1) * 64 + kg * 16 : (int)0x80000000u;
  }
  // Second layer, output rows y, y + 1 from first-layer rows lo 0, lo 1, hi 0, hi 1, and their pool.
  auto second = [&](int y, int lo, int hi) {
    const char *const base = s + kPairOut + kg * kPairPlane + col * 16;
    auto operand = [&](int st, int pb) {
      const int dx = st >> 2, rr = st & 3;
      return *(const bf16x8 *)(base + (rr < 2 ? lo : hi) + (rr & 1) * kPairRow + (pb * 16 + dx) * 16);
    };
    f32x4 acc[2][2][2];
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int pb = 0; pb < 2; pb++)
#pragma unroll
        for (int mb = 0; mb < 2; mb++) acc[r][pb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int D = 4;
    bf16x8 bx[D][2];
#pragma unroll
    for (int st = 0; st < D - 1; st++)
#pragma unroll
      for (int pb = 0; pb < 2; pb++) bx[st][pb] = operand(st, pb);
#pragma unroll
    for (int st = 0; st < 12; st++) {
      const int dx = st >> 2, rr = st & 3;
      if (st + D - 1 < 12)
#pragma unroll
        for (int pb = 0; pb < 2; pb++) bx[(st + D - 1) % D][pb] = operand(st + D - 1, pb);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 2; r++) {
        const int dy = rr - r;
        if (dy < 0 || dy > 2) continue;
#pragma unroll
        for (int pb = 0; pb < 2; pb++)
#pragma unroll
          for (int mb = 0; mb < 2; mb++)
            acc[r][pb][mb] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[dy * 3 + dx][mb], bx[st % D][pb], acc[r][pb][mb], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    bf16x8 v[2][2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const bool in = y + r < h;
      const __amdgpu_buffer_rsrc_t rs = row_rsrc(a1.out0, in ? (size_t)n * h + y + r : 0, in ? w : 0, 32);
#pragma unroll
      for (int pb = 0; pb < 2; pb++) {
        f32x8 f;
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = relu(acc[r][pb][i >> 2][i & 3] + bias1[i]);
        v[r][pb] = __builtin_convertvector(f, bf16x8);
        row_store8(rs, out_at[pb], v[r][pb]);
      }
    }
    const bool in = (y >> 1) < (h >> 1);
    const __amdgpu_buffer_rsrc_t ps =
        row_rsrc(a1.pool_out, in ? (size_t)n * (h >> 1) + (y >> 1) : 0, in ? w >> 1 : 0, 32);
#pragma unroll
    for (int pb = 0; pb < 2; pb++) {
      f32x8 f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float t = unpack8(v[0][pb], i), b = unpack8(v[1][pb], i);
        f[i] = (((t + lane_xor1(t)) + b) + lane_xor1(b)) * 0.25f;
      }
      const bf16x8 o = __builtin_convertvector(f, bf16x8);
      row_store8(ps, pool_at[pb], o);
    }
  };
  // Lanes read what other lanes of the wave wrote: LDS serves a wave in
  // order, the fence keeps the compiler to that order too.
  auto fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  *(bf16x8 *)(s + kPairZero + lane * 16) = zero8;
  fetch(ys - 2);
  stage(ys - 2, kPairHalf, false);
  fetch(ys);
  stage(ys, 0, true);
  fetch(ys + 2);
  fence();
  first(ys - 1, kPairHalf, 0, false, true);
  fence();
  for (int k = 1; k <= pairs; k++) {
    const int hi = (k & 1) * kPairHalf, lo = kPairHalf - hi, y = ys + 2 * k;
    stage(y, hi, k < pairs);
    fetch(y + 2);  // (in flight during the matrix work; past the segment: clamped rows nothing reads)
    fence();
    first(y - 1, lo, hi, true, k < pairs);
    fence();
    second(y - 2, lo, hi);
    fence();
  }
}

// Weight and bias gradient of a 3x3 convolution:
//   dW[tap][ci][co] = sum_p X[p + shift(tap)][ci] * dY[p][co],  db[co] = sum_p dY[p][co]
// A wave owns 32 output channels x NC blocks of 16 channels of one 32-channel
// group of the input, all 9 taps (MFMA rows: output channels, columns: input
// channels, K: 32 pixels of a row), and walks down a 32-pixel strip.  Step r
// has the input row r (34 pixels) and the gradient row r + 1: the input row's
// operands of the three horizontal taps serve the gradient rows r - 1, r and
// r + 1, which are kept in registers, so a step is 18 NC MFMAs on 2 + 3 NC
// operands.  The rows land in LDS by direct loads, in a ring of four steps of
// the wave's own: nothing waits at a barrier.  The bias gradient (input
// group 0) is one more MFMA a block, with a column of ones.
//
// LDS is [pixel][32 channels], as in memory; a transposing read
// (ds_read_b64_tr_b16) gives 16 lanes 4 consecutive pixels of a channel each,
// so there is no transposition on the way in, and a tap's shift is an address.
// A lane group's pixels are kg 4 + 0 .. 3 and 16 more on (K in any order, the
// same for both operands).  The 32-byte halves of pixels 4 to 7 of every 8 are
// exchanged, which puts the 8 pixels that 32 lanes read on all banks.
//
// The pixels (strips x rows) of an image batch are one list, divided evenly
// over the waves; a wave's share is one or more pieces of strips.  Each
// workgroup adds its 8 waves' sums and stores them (no atomics) to its own slot
// of the scratch buffer, part[group][slot][tap][ci % 32][co] and
// part_b[slot][co]; wgrad_reduce_kernel adds the slots in a fixed order.
//
// What bounds it (16 x 256 x 256): 96 -> 32 at full size 56 us, of which 27 are
// its MFMAs, 9 the direct loads that do not overlap, and 10 a launch's start,
// first loads and last sums.  Staging pixel pairs through registers into
// transposed rows and shifting operands by elements, with one workgroup's
// waves at two barriers a round, it was bound by LDS: 157 us; the ten layers
// 570 and 66 for their sums, now 284 and 23.
constexpr int kWgradWaves = 8, kWgradSlot = 34 * 64 + 32 * 64, kWgradRing = 4 * kWgradSlot;
constexpr int kWgradLds = kWgradWaves * kWgradRing;
template <int NC> constexpr int wgrad_sums() { return 18 * NC + 2; }  // f32x4 a lane, with the bias
// The operands of one step: per operand 8 pixels of the lane's channel, kg 4 + 0 .. 3 and 16 (1 KB) on.  In
// assembly, with its wait: before the builtin of this read the compiler waits for every direct load in
// flight, the next steps' too (wgrad 96 -> 32 at 256 x 256 x 16: 78 us).
template <int NC>
LGX_D void wgrad_operands(int at, const int (&xoff)[3][NC], const int (&doff)[2], bf16x8 (&b)[3][NC], bf16x8 (&d)[2]) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  s16x4 v[3 * NC + 2][2];
  int p[3 * NC + 2];
#pragma unroll
  for (int k = 0; k < 3 * NC; k++) p[k] = at + xoff[k / NC][k % NC];
#pragma unroll
  for (int k = 0; k < 2; k++) p[3 * NC + k] = at + doff[k];
  if constexpr (NC == 2) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %16 offset:1024\n\t"
        "ds_read_b64_tr_b16 %2, %17\n\tds_read_b64_tr_b16 %3, %17 offset:1024\n\t"
        "ds_read_b64_tr_b16 %4, %18\n\tds_read_b64_tr_b16 %5, %18 offset:1024\n\t"
        "ds_read_b64_tr_b16 %6, %19\n\tds_read_b64_tr_b16 %7, %19 offset:1024\n\t"
        "ds_read_b64_tr_b16 %8, %20\n\tds_read_b64_tr_b16 %9, %20 offset:1024\n\t"
        "ds_read_b64_tr_b16 %10, %21\n\tds_read_b64_tr_b16 %11, %21 offset:1024\n\t"
        "ds_read_b64_tr_b16 %12, %22\n\tds_read_b64_tr_b16 %13, %22 offset:1024\n\t"
        "ds_read_b64_tr_b16 %14, %23\n\tds_read_b64_tr_b16 %15, %23 offset:1024\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1]), "=&v"(v[2][0]), "=&v"(v[2][1]),
          "=&v"(v[3][0]), "=&v"(v[3][1]), "=&v"(v[4][0]), "=&v"(v[4][1]), "=&v"(v[5][0]), "=&v"(v[5][1]),
          "=&v"(v[3 * NC][0]), "=&v"(v[3 * NC][1]), "=&v"(v[3 * NC + 1][0]), "=&v"(v[3 * NC + 1][1])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[3 * NC]), "v"(p[3 * NC + 1])
        : "memory");
  } else {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %10\n\tds_read_b64_tr_b16 %1, %10 offset:1024\n\t"
        "ds_read_b64_tr_b16 %2, %11\n\tds_read_b64_tr_b16 %3, %11 offset:1024\n\t"
        "ds_read_b64_tr_b16 %4, %12\n\tds_read_b64_tr_b16 %5, %12 offset:1024\n\t"
        "ds_read_b64_tr_b16 %6, %13\n\tds_read_b64_tr_b16 %7, %13 offset:1024\n\t"
        "ds_read_b64_tr_b16 %8, %14\n\tds_read_b64_tr_b16 %9, %14 offset:1024\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1]), "=&v"(v[2][0]), "=&v"(v[2][1]),
          "=&v"(v[3][0]), "=&v"(v[3][1]), "=&v"(v[4][0]), "=&v"(v[4][1])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4])
        : "memory");
  }
  auto whole = [&](int k) {
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(v[k][0], v[k][1], 0, 1, 2, 3, 4, 5, 6, 7));
  };
#pragma unroll
  for (int k = 0; k < 3 * NC; k++) b[k / NC][k % NC] = whole(k);
#pragma unroll
  for (int k = 0; k < 2; k++) d[k] = whole(3 * NC + k);
}
template <int NC> LGX_D void wgrad_task(const WgradArgs &a, int task) {
  extern __shared__ __align__(16) char s_wg[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kg = lane >> 4;
  const int groups = (a.ca + a.cb) >> 5, units = groups * (a.cout >> 5), slots = a.slots;
  // the units of one share of the pixels are neighbours (the same rows, in one XCD's L2)
  const int slot = task / units, g = task % units % groups, co0 = task % units / groups * 32;
  const bool from_a = g * 32 < a.ca;
  const int up = from_a && a.a_up ? 1 : 0;
  const int cs = from_a ? a.ca : a.cb, ch = from_a ? g * 32 : g * 32 - a.ca;
  const bf16 *const src = from_a ? a.a : a.b;
  const int sw = a.w >> up, sh = a.h >> up, bands = (a.w + 31) >> 5;
  const int items = a.n * bands * a.h;  // (checked on the host)
  int i0 = (slot * kWgradWaves + wave) * a.rows;
  const int i1 = min(items, i0 + a.rows);
  typedef __attribute__((address_space(3))) void LdsVoid;
  char *const ring = s_wg + wave * kWgradRing;
  const int ring_at = (int)(uintptr_t)(LdsVoid *)ring;  // in LDS
  struct Piece {  // dY rows [ys, ye) of a strip; at most cap rows, so that offsets in it stay below 2 GB
    int n, x0, ys, ye;
  };
  auto piece_at = [&](int i) {
    const int strip = i / a.h, ys = i % a.h;
    return Piece{strip / bands, strip % bands * 32, ys, min(min(a.h, ys + (i1 - i)), ys + a.cap)};
  };
  // Direct loads of one step: input row r (2 KB and the last two pixels, 8 lanes) and gradient row r + 1.
  // Rows outside the image or the piece, and steps past the end, are past their buffer: zeros.  Five loads,
  // always: the wait below counts them.  A piece has its buffers (from input row ys - 1, or 0, and gradient
  // row ys) and lane offsets, a step only its two row offsets: with whole addresses formed per step the
  // scalar work was as long as the matrix work.
  const int part = ((lane & 3) ^ (lane >> 4 & 1) * 2) * 16;
  const int xstep = sw * cs * 2, dstep = a.w * a.cout * 2;
  int fi = i0, fr = 0, fy = 0, xsize = 0, dsize = 0, xlane[3], dlane[2];
  Piece fp = {0, 0, 0, 0};
  __amdgpu_buffer_rsrc_t xr, dr;
  auto open = [&] {  // the piece at fi
    fp = piece_at(min(fi, items - 1));
    fr = fp.ys - 1;
    fy = max(fr, 0) >> up;
    xsize = (int)min((long)(sh - fy) * xstep - ch * 2, 0x7fffffffL);
    dsize = (int)min((long)(a.h - fp.ys) * dstep - co0 * 2, 0x7fffffffL);
    xr = __builtin_amdgcn_make_buffer_rsrc((void *)(src + ((size_t)fp.n * sh + fy) * sw * cs + ch), (short)0, xsize,
                                           0x00020000);
    dr = __builtin_amdgcn_make_buffer_rsrc((void *)(a.dy + ((size_t)fp.n * a.h + fp.ys) * a.w * a.cout + co0), (short)0,
                                           dsize, 0x00020000);
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const int x = fp.x0 - 1 + b * 16 + (lane >> 2);
      xlane[b] = (uint32_t)x < (uint32_t)a.w ? (x >> up) * cs * 2 + part : (int)0x80000000u;
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const int x = fp.x0 + b * 16 + (lane >> 2);
      dlane[b] = x < a.w ? x * a.cout * 2 + part : (int)0x80000000u;
    }
  };
  char *dst = ring;  // the slot the loads below fill
  auto load_x = [&](int b0, int b1) {
    const int row = fi < i1 && (uint32_t)fr < (uint32_t)a.h ? ((fr >> up) - fy) * xstep : xsize;
#pragma unroll
    for (int b = b0; b < b1; b++)
      if (b < 2 || lane < 8)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (LdsVoid *)(dst + b * 1024), 16, xlane[b], row, 0, 0);
  };
  auto load_d = [&](int b) {
    const int row = fi < i1 && fr + 1 < fp.ye ? (fr + 1 - fp.ys) * dstep : dsize;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(dr, (LdsVoid *)(dst + 34 * 64 + b * 1024), 16, dlane[b], row, 0, 0);
  };
  auto next = [&] {
    if (++fr > fp.ye && fi < i1) {
      fi += fp.ye - fp.ys;
      if (fi < i1) open();
    }
  };
  open();
  // lane offsets of the operands: input pixels dx + kg 4 + .., half cb; gradient pixels kg 4 + .., half mb
  int xoff[3][NC], doff[2];
#pragma unroll
  for (int dx = 0; dx < 3; dx++) {
    const int p = dx + kg * 4 + (col >> 2);
#pragma unroll
    for (int cb = 0; cb < NC; cb++) xoff[dx][cb] = p * 64 + (cb ^ (p >> 2 & 1)) * 32 + (col & 3) * 8;
  }
#pragma unroll
  for (int mb = 0; mb < 2; mb++) {
    const int p = kg * 4 + (col >> 2);
    doff[mb] = 34 * 64 + p * 64 + (mb ^ (p >> 2 & 1)) * 32 + (col & 3) * 8;
  }
  f32x4 acc[9][NC][2], accb[2];
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
#pragma unroll
      for (int mb = 0; mb < 2; mb++) acc[t][cb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int mb = 0; mb < 2; mb++) accb[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones, d[3][2];  // d: gradient rows r - 1, r, r + 1
#pragma unroll
  for (int i = 0; i < 8; i++) ones[i] = f2bf(1.f);
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int mb = 0; mb < 2; mb++) d[k][mb] = bf16x8{};
  for (int k = 0; k < 3; k++) {
    dst = ring + k * kWgradSlot;
    load_x(0, 3);
    load_d(0);
    load_d(1);
    next();
  }
  int at = 0;
  while (i0 < i1) {
    const Piece p = piece_at(i0);
    i0 += p.ye - p.ys;
    for (int r = p.ys - 1; r <= p.ye; r++) {
      // this step's five loads have landed (ten later ones are in flight); the slot the next loads go to
      // was read in the last step
      asm volatile("s_waitcnt vmcnt(10) lgkmcnt(0)" ::: "memory");
      dst = ring + (at == 0 ? 3 * kWgradSlot : at - kWgradSlot);
      const int x = ring_at + at;
      at = at == 3 * kWgradSlot ? 0 : at + kWgradSlot;
      bf16x8 b[3][NC];
      wgrad_operands<NC>(x, xoff, doff, b, d[2]);
      // vertical tap t: gradient row r + 1 - t, while it is in the piece (uniform)
      auto taps = [&](int t) {
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int cb = 0; cb < NC; cb++)
#pragma unroll
            for (int mb = 0; mb < 2; mb++)
              acc[t * 3 + dx][cb][mb] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[2 - t][mb], b[dx][cb], acc[t * 3 + dx][cb][mb], 0, 0, 0);
      };
      load_x(0, 2);
      if (r > p.ys) taps(2);
      load_x(2, 3);
      load_d(0);
      if (r >= p.ys && r < p.ye) taps(1);
      load_d(1);
      next();
      if (r + 1 < p.ye) {
        taps(0);
        if (g == 0)
#pragma unroll
          for (int mb = 0; mb < 2; mb++)
            accb[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[2][mb], ones, accb[mb], 0, 0, 0);
      }
#pragma unroll
      for (int mb = 0; mb < 2; mb++) {
        d[0][mb] = d[1][mb];
        d[1][mb] = d[2][mb];
      }
    }
  }
  // The waves' sums in a fixed order, through LDS, which holds four waves': waves 4 .. 7 to waves 0 .. 3, then
  // each wave adds the four of an eighth of the sums and stores it.
  constexpr int SUMS = wgrad_sums<NC>();
  f32x4 *const all = (f32x4 *)s_wg + lane;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int round = 0; round < 2; round++) {
    __syncthreads();
    f32x4 *const mine = all + (size_t)(wave & 3) * SUMS * 64;
    if ((wave >> 2) != round) {  // round 0: waves 4 .. 7, round 1: waves 0 .. 3
#pragma unroll
      for (int k = 0; k < 18 * NC; k++) mine[k * 64] = acc[k / (2 * NC)][k / 2 % NC][k % 2];
#pragma unroll
      for (int k = 0; k < 2; k++) mine[(18 * NC + k) * 64] = accb[k];
    }
    __syncthreads();
    if (round == 0 && wave < 4) {
#pragma unroll
      for (int k = 0; k < 18 * NC; k++) acc[k / (2 * NC)][k / 2 % NC][k % 2] += mine[k * 64];
#pragma unroll
      for (int k = 0; k < 2; k++) accb[k] += mine[(18 * NC + k) * 64];
    }
  }
  float *out = a.part + ((size_t)g * slots + slot) * (9 * 32 * a.cout) + co0 + kg * 4;
  for (int k = wave; k < SUMS; k += kWgradWaves) {
    const f32x4 v = ((all[k * 64] + all[(SUMS + k) * 64]) + all[(2 * SUMS + k) * 64]) + all[(3 * SUMS + k) * 64];
    if (k < 18 * NC)  // tap, input block, output block
      *(f32x4 *)&out[(k / (2 * NC) * 32 + k / 2 % NC * 16 + col) * a.cout + k % 2 * 16] = v;
    else if (g == 0 && col == 0)
      *(f32x4 *)&a.part_b[(size_t)slot * a.cout + co0 + (k - 18 * NC) * 16 + kg * 4] = v;
  }
}

// The weight gradients of layers l .. t.n - 1: workgroup -> layer -> task (a unit's share).
__global__ __launch_bounds__(64 * kWgradWaves, 2) void conv3x3_wgrad_kernel(const WgradTable t, int l) {
  const int id = (int)xcd_remap(blockIdx.x, gridDim.x) + t.first[l];
  while (id >= t.first[l + 1]) l++;
  const WgradArgs &a = t.l[l];
  if (a.cin_log <= 16)  // the other half of the only group's channels is padding
    wgrad_task<1>(a, id - t.first[l]);
  else
    wgrad_task<2>(a, id - t.first[l]);
}

// The fixed-order sums of the workgroups' partial sums, all layers in one
// launch.  A workgroup of a layer's weight gradient,
//   dw[co][ci][tap] = sum over slots of part[g][slot][tap][ci % 32][co]
// written in the master layout for ci < cin_log (g = ci / 32), has 16 float4
// elements x 16 slices; slice k sums slots k, k + 16, ... and the slice sums are
// added in order (256 slots: with 4 slices of 64 loads each, 100 us for the
// ten layers instead of 23).  A layer's last workgroup: the bias gradient, db[co] =
// sum over slots of part_b[slot][co], the same way.  Neither result depends on
// the order in which workgroups ran.
constexpr int kReduceEl = 16, kReduceSl = 16;
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const WgradTable t) {
  int l = 0;
  while ((int)blockIdx.x >= t.reduce[l + 1]) l++;
  const WgradArgs &a = t.l[l];
  const int blk = (int)blockIdx.x - t.reduce[l], cout = a.cout, slots = a.slots;
  __shared__ f32x4 red[kReduceSl][kReduceEl];
  const int el = threadIdx.x % kReduceEl, sl = threadIdx.x / kReduceEl;
  const bool bias = (int)blockIdx.x + 1 == t.reduce[l + 1];  // uniform per workgroup
  if (bias) {
    float *const rb = (float *)red;
    const int co = (int)threadIdx.x % cout, k0 = (int)threadIdx.x / cout, step = 256 / cout;
    float sb = 0.f;
    for (int k = k0; k < slots; k += step) sb += a.part_b[(size_t)k * cout + co];
    rb[threadIdx.x] = sb;
    __syncthreads();
    if (k0) return;
    for (int k = 1; k < step; k++) sb += rb[k * cout + co];
    a.db[co] = sb;
    return;
  }
  const int per4 = 9 * 32 * cout / 4;
  const int e = blk * kReduceEl + el;  // (a workgroup is in one group, and whole)
  const int g = e / per4, f = e % per4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const f32x4 *src = (const f32x4 *)a.part + (size_t)g * slots * per4 + f;
  for (int k = sl; k < slots; k += kReduceSl) acc += src[(size_t)k * per4];
  red[sl][el] = acc;
  __syncthreads();
  if (sl) return;
  f32x4 v = red[0][el];
#pragma unroll
  for (int k = 1; k < kReduceSl; k++) v += red[k][el];
  const int tap = f * 4 / (32 * cout), rem = f * 4 % (32 * cout), ci = g * 32 + rem / cout, co = rem % cout;
  if (ci < a.cin_log)
#pragma unroll
    for (int i = 0; i < 4; i++) a.dw[((size_t)(co + i) * a.cin_log + ci) * 9 + tap] = v[i];
}

// ------------------------------------------------------------ glue kernels

__global__ __launch_bounds__(256) void avgpool_kernel(const bf16 *x, int n, int h, int w, int c, bf16 *y) {
  // y[n][h/2][w/2][c] = mean of the 2x2 children
  const int hh = h >> 1, ww = w >> 1;
  const size_t total = (size_t)n * hh * ww * (c / 8);
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const int q = (int)(e % (c / 8));
    size_t p = e / (c / 8);
    const int xx = (int)(p % ww);
    p /= ww;
    const int yy = (int)(p % hh);
    const int nn = (int)(p / hh);
    const size_t b00 = (((size_t)nn * h + 2 * yy) * w + 2 * xx) * c + q * 8;
    const bf16x8 v0 = *(const bf16x8 *)(x + b00), v1 = *(const bf16x8 *)(x + b00 + c);
    const bf16x8 v2 = *(const bf16x8 *)(x + b00 + (size_t)w * c), v3 = *(const bf16x8 *)(x + b00 + (size_t)w * c + c);
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = f2bf((bf2f(v0[i]) + bf2f(v1[i]) + bf2f(v2[i]) + bf2f(v3[i])) * 0.25f);
    *(bf16x8 *)(y + (((size_t)nn * hh + yy) * ww + xx) * c + q * 8) = o;
  }
}

// dx[p] = mask(act[p] > 0) * (dx_in[p] + dpool[p/2] / 4): the gradient of a
// tensor feeding both a concatenation (dx_in) and an average pool (dpool).
// Rows (image nn, row yy) over blockIdx.y, their pixels x 8-channel groups
// over the threads: 32-bit index arithmetic, no division in the loop (c / 8
// is a power of two).
__global__ __launch_bounds__(256) void pool_bwd_add_kernel(const bf16 *dx_in, const bf16 *dpool, const bf16 *act, int n,
                                                           int h, int w, int c, bf16 *dx) {
  const int cq = c / 8, cs = __builtin_ctz((unsigned)cq);
  for (int row = blockIdx.y; row < n * h; row += gridDim.y) {
  const int yy = row % h, nn = row / h;
  const size_t r0 = (size_t)row * w * c, rp = ((size_t)nn * (h >> 1) + (yy >> 1)) * (w >> 1) * c;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < w * cq; e += gridDim.x * 256) {
    const int q = e & (cq - 1), xx = e >> cs;
    const size_t i0 = r0 + (size_t)xx * c + q * 8, ip = rp + (size_t)(xx >> 1) * c + q * 8;
    const bf16x8 a = *(const bf16x8 *)(dx_in + i0), b = *(const bf16x8 *)(dpool + ip), m = *(const bf16x8 *)(act + i0);
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = bf2f(m[i]) > 0.f ? f2bf(bf2f(a[i]) + 0.25f * bf2f(b[i])) : f2bf(0.f);
    *(bf16x8 *)(dx + i0) = o;
  }
  }
}

// Gradient through a nearest x2 upsample: dhalf[q] = mask(act[q] > 0) * sum of its 4 children.
__global__ __launch_bounds__(256) void upsample_bwd_kernel(const bf16 *dfull, const bf16 *act, int n, int hh, int ww, int c,
                                                           bf16 *dhalf) {
  const int h = hh * 2, w = ww * 2;
  const size_t total = (size_t)n * hh * ww * (c / 8);
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const int q = (int)(e % (c / 8));
    size_t p = e / (c / 8);
    const int xx = (int)(p % ww);
    p /= ww;
    const int yy = (int)(p % hh);
    const int nn = (int)(p / hh);
    const size_t b00 = (((size_t)nn * h + 2 * yy) * w + 2 * xx) * c + q * 8;
    const bf16x8 v0 = *(const bf16x8 *)(dfull + b00), v1 = *(const bf16x8 *)(dfull + b00 + c);
    const bf16x8 v2 = *(const bf16x8 *)(dfull + b00 + (size_t)w * c);
    const bf16x8 v3 = *(const bf16x8 *)(dfull + b00 + (size_t)w * c + c);
    const size_t oi = (((size_t)nn * hh + yy) * ww + xx) * c + q * 8;
    const bf16x8 m = *(const bf16x8 *)(act + oi);
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; i++)
      o[i] = bf2f(m[i]) > 0.f ? f2bf(bf2f(v0[i]) + bf2f(v1[i]) + bf2f(v2[i]) + bf2f(v3[i])) : f2bf(0.f);
    *(bf16x8 *)(dhalf + oi) = o;
  }
}

// Training: the 1x1 head, the loss and the head's backward in one pass (the
// head's output is not stored).  One pixel per thread: out = x + b_h + W_h
// act, summed channel by channel; mean L1: g = sign(out - target) /
// count per channel, mean squared error (l2): g = 2 (out - target) / count;
// dd1 = mask(d1 > 0) W_h^T g (per channel, the three products in channel
// order).  A thread keeps 3 x 32 head-weight partial sums; they are reduced
// over the lanes of a wave with shuffles, over the waves in LDS, and added to
// dW_h, db_h and the loss once per workgroup.
__global__ __launch_bounds__(256) void head_train_kernel(const bf16 *__restrict__ d1, const float *__restrict__ x12,
                                                         const float4 *__restrict__ target, const float *__restrict__ wh,
                                                         const float *__restrict__ bh, size_t npix, float inv_count,
                                                         int l2, bf16 *__restrict__ dd1, float *dwh, float *dbh,
                                                         float *loss) {
  __shared__ float red[4][100];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float aw[3][32], ab[3] = {0.f, 0.f, 0.f}, al = 0.f;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int i = 0; i < 32; i++) aw[c][i] = 0.f;
  for (size_t p = (size_t)blockIdx.x * 256 + threadIdx.x; p < npix; p += (size_t)gridDim.x * 256) {
    bf16x8 v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = *(const bf16x8 *)(d1 + p * 32 + q * 8);
    const float4 t = target[p];
    float o[3];
#pragma unroll
    for (int c = 0; c < 3; c++) o[c] = x12[p * 12 + c] + bh[c];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float f = bf2f(v[q][i]);
#pragma unroll
        for (int c = 0; c < 3; c++) o[c] += wh[c * 32 + q * 8 + i] * f;
      }
    const float df[3] = {o[0] - t.x, o[1] - t.y, o[2] - t.z};
    float g[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      g[c] = (l2 ? 2.f * df[c] : (df[c] > 0.f ? 1.f : (df[c] < 0.f ? -1.f : 0.f))) * inv_count;
      al += l2 ? df[c] * df[c] : fabsf(df[c]);
      ab[c] += g[c];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      bf16x8 o8;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float f = bf2f(v[q][i]);
        float sacc = 0.f;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          sacc += wh[c * 32 + q * 8 + i] * g[c];
          aw[c][q * 8 + i] += g[c] * f;
        }
        o8[i] = f > 0.f ? f2bf(sacc) : f2bf(0.f);
      }
      *(bf16x8 *)(dd1 + p * 32 + q * 8) = o8;
    }
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
      for (int i = 0; i < 32; i++) aw[c][i] += __shfl_xor(aw[c][i], m);
      ab[c] += __shfl_xor(ab[c], m);
    }
    al += __shfl_xor(al, m);
  }
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
#pragma unroll
      for (int i = 0; i < 32; i++) red[wave][c * 32 + i] = aw[c][i];
      red[wave][96 + c] = ab[c];
    }
    red[wave][99] = al;
  }
  __syncthreads();
  if (threadIdx.x < 100) {
    const float v = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
    if (threadIdx.x < 96) atomicAdd(&dwh[threadIdx.x], v);
    else if (threadIdx.x < 99) atomicAdd(&dbh[threadIdx.x - 96], v);
    else if (loss) atomicAdd(loss, v * inv_count);
  }
}

// Adam on the FP32 master parameters (Kingma & Ba 2015, bias-corrected);
// every updated weight of the convolutions is also written to its BF16
// forward and input-gradient layouts (pack_weights_kernel's placement; the
// zero padding channels are never written).
__global__ __launch_bounds__(256) void adam_pack_kernel(float *p, const float *g, float *m, float *v, size_t n, float lr,
                                                        float b1, float b2, float eps, float bc1, float bc2,
                                                        const PackTable pk) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    p[i] = pi;
#pragma unroll 1
    for (int l = 0; l < pk.n; l++) {
      const PackLayer &L = pk.l[l];
      if (i < L.off || i >= L.off + (size_t)L.cout * L.cin_log * 9) continue;
      const size_t r = i - L.off;
      const int tap = (int)(r % 9), ci = (int)((r / 9) % L.cin_log), co = (int)(r / 9 / L.cin_log);
      const bf16 b = f2bf(pi);
      L.wf[(((size_t)tap * (L.cin_pad / 32) + ci / 32) * L.cout + co) * 32 + (ci & 31)] = b;
      if (L.wt) L.wt[(((size_t)(8 - tap) * (L.cout / 32) + co / 32) * L.cin_pad + ci) * 32 + (co & 31)] = b;
      break;
    }
  }
}

__global__ __launch_bounds__(256) void fill_kernel(float *p, size_t n, float v) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = v;
}

// Pack master weights W[co][ci][3][3] (FP32, ci < cin_log) into the forward
// layout [tap][cin_pad/32][cout][32] and, when wt != null, the input-gradient
// layout: the same convolution read as cout -> cin_pad with flipped taps,
// [tap'][cout/32][cin_pad][32] with tap' = 8 - tap.
__global__ __launch_bounds__(256) void pack_weights_kernel(const float *w, int cout, int cin_log, int cin_pad, bf16 *wf,
                                                           bf16 *wt) {
  const size_t total = (size_t)cout * cin_pad * 9;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const int tap = (int)(e % 9);
    const int ci = (int)((e / 9) % cin_pad);
    const int co = (int)(e / 9 / cin_pad);
    const float v = ci < cin_log ? w[((size_t)co * cin_log + ci) * 9 + tap] : 0.f;
    wf[(((size_t)tap * (cin_pad / 32) + ci / 32) * cout + co) * 32 + (ci & 31)] = f2bf(v);
    if (wt) wt[(((size_t)(8 - tap) * (cout / 32) + co / 32) * cin_pad + ci) * 32 + (co & 31)] = f2bf(v);
  }
}

// MFMA operand-layout probe: D = A * B for a 16x32 A and 32x16 B given in
// row-major order, computed by one wave with the layout stated above.
__global__ __launch_bounds__(64) void mfma_probe_kernel(const float *A, const float *B, float *D) {
  const int l = threadIdx.x, col = l & 15, kg = l >> 4;
  bf16x8 a, b;
  for (int i = 0; i < 8; i++) {
    a[i] = f2bf(A[col * 32 + kg * 8 + i]);
    b[i] = f2bf(B[(kg * 8 + i) * 16 + col]);
  }
  f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  for (int i = 0; i < 4; i++) D[(kg * 4 + i) * 16 + col] = d[i];
}

// ------------------------------------------------------------ launchers

static unsigned grid_for(size_t work, size_t per_block) {
  size_t g = (work + per_block - 1) / per_block;
  if (g > 65535u * 16u) g = 65535u * 16u;
  return (unsigned)(g ? g : 1);
}

// Register tiles (R rows, PB pixel blocks) offered per output-channel block
// count MB, accumulators R * PB * MB * 4 VGPRs <= 128; entry 0 is the
// default, the others are the autotuner's candidates.  Which tile a layer gets
// is measured at the network's shape (1920 x 1080, us: best register tile /
// best conv3x3_lds_kernel tile / best conv3x3_dma_kernel tile): 32 -> 32 at full
// size 84 / 57 / 55; 32 -> 64 at half size 51 / 36 / 26; 128 -> 64 99 / 57 /
// 40; 64 -> 128 at a quarter 63 / 27 / 23; 192 -> 64 at half size 213 / 113 /
// 91.  The input gradient 32 -> 96 (16 x 256 x 256: 151 / 90 / 82) is fastest
// with 16 columns a tile, whose registers let four waves share a SIMD; others
// are not (32 -> 32 at full size 59 with it).  The smallest images go the other
// way (quarter size of 256 x 256: 12.4 / 13.5 / 19): the direct-load tiles are
// the largest, and too few of them
// fill the chip.
struct ConvTile {
  int r, pb, lds;  // lds: 1 conv3x3_lds_kernel, 2 conv3x3_dma_kernel with WR = r, WP = pb
  int mbw;         // lds: output-channel blocks per workgroup (cout / (16 * mbw) splits)
  int per_cu;      // lds: workgroups per CU walking the tiles, 0 = one workgroup per tile
  int nw;          // dma: waves per workgroup
};
static constexpr ConvTile kTiles1[] = {{4, 2, 0, 1, 0}, {2, 4, 0, 1, 0}, {4, 4, 0, 1, 0}, {1, 4, 0, 1, 0}};
static constexpr ConvTile kTiles2[] = {{4, 2, 0, 2, 0}, {2, 4, 0, 2, 0}, {4, 4, 0, 2, 0},   {1, 4, 0, 2, 0},
                                   {2, 4, 1, 2, 0}, {2, 2, 1, 2, 0}, {1, 4, 1, 2, 0},   {2, 4, 1, 2, 2},
                                   {2, 2, 1, 2, 3}, {1, 4, 1, 2, 3}, {2, 2, 2, 2, 2, 4}, {2, 2, 2, 2, 1, 8}};
static constexpr ConvTile kTiles4[] = {{2, 2, 0, 4, 0}, {4, 2, 0, 4, 0}, {2, 4, 0, 4, 0}, {1, 4, 0, 4, 0},   {2, 2, 1, 4, 0},
                                   {1, 4, 1, 4, 0}, {1, 2, 1, 4, 0}, {2, 2, 1, 4, 2}, {1, 2, 1, 4, 3},   {2, 4, 1, 2, 0},
                                   {2, 2, 1, 2, 3}, {2, 2, 2, 4, 1, 4}, {2, 2, 2, 4, 1, 8}};
static constexpr ConvTile kTiles6[] = {{2, 2, 0, 6, 0}, {1, 4, 0, 6, 0}, {1, 2, 0, 6, 0},
                                   {2, 4, 1, 2, 0}, {2, 2, 1, 2, 3}, {2, 2, 2, 2, 2, 4}, {2, 1, 2, 2, 2, 8}};
static constexpr ConvTile kTiles8[] = {{1, 2, 0, 8, 0}, {2, 2, 0, 8, 0}, {1, 4, 0, 8, 0},   {2, 2, 1, 4, 0},
                                   {1, 2, 1, 4, 3}, {2, 2, 1, 4, 2}, {2, 2, 2, 4, 1, 4}, {2, 2, 2, 4, 1, 8}};
static constexpr ConvTile kTiles12[] = {{1, 2, 0, 12, 0}, {2, 1, 0, 12, 0},   {2, 2, 1, 4, 0},
                                    {1, 2, 1, 4, 3},  {2, 2, 2, 4, 1, 4}, {2, 2, 2, 4, 1, 8}};

static const ConvTile *conv_tiles(int mb, int *count) {
#define LGX_TILES(T) \
  *count = (int)(sizeof(T) / sizeof(T[0])); \
  return T
  switch (mb) {
    case 1: LGX_TILES(kTiles1);
    case 2: LGX_TILES(kTiles2);
    case 4: LGX_TILES(kTiles4);
    case 6: LGX_TILES(kTiles6);
    case 8: LGX_TILES(kTiles8);
    case 12: LGX_TILES(kTiles12);
    default: *count = 0; return nullptr;
  }
#undef LGX_TILES
}

// The tile of a network that was not autotuned, from the pixels of the layer's output.  Direct-load tiles from
// where they fill the chip, below that the LDS tiles with the most workgroups: a pass with
// them takes 1.00 to 1.02 times the autotuned one from 16 x 16 to 2560 x 1440 (1.10 at 2 x 512 x 512); with the
// tables' first entries 1280 x 720 took 523 us instead of 274 and 2560 x 1440 1746 instead of 941.
// (Named by their shapes, which must be in the tables: an index would follow another tile's insertion.)
template <size_t N> constexpr int tile_index(const ConvTile (&tiles)[N], const ConvTile &t) {
  for (size_t i = 0; i < N; i++)
    if (tiles[i].r == t.r && tiles[i].pb == t.pb && tiles[i].lds == t.lds && tiles[i].mbw == t.mbw &&
        tiles[i].per_cu == t.per_cu && tiles[i].nw == t.nw)
      return (int)i;
  return -1;
}
int conv3x3_default_tile(int cout, long pixels) {
  constexpr int dma2 = tile_index(kTiles2, {2, 2, 2, 2, 2, 4});
  constexpr int lds4 = tile_index(kTiles4, {1, 2, 1, 4, 3}), dma4 = tile_index(kTiles4, {2, 2, 2, 4, 1, 4}),
                wide4 = tile_index(kTiles4, {2, 2, 2, 4, 1, 8});
  constexpr int lds6 = tile_index(kTiles6, {2, 2, 1, 2, 3}), dma6 = tile_index(kTiles6, {2, 1, 2, 2, 2, 8});
  constexpr int lds8 = tile_index(kTiles8, {1, 2, 1, 4, 3}), wide8 = tile_index(kTiles8, {2, 2, 2, 4, 1, 8});
  constexpr int dma12 = tile_index(kTiles12, {2, 2, 2, 4, 1, 4}), wide12 = tile_index(kTiles12, {2, 2, 2, 4, 1, 8});
  static_assert(dma2 >= 0 && lds4 >= 0 && dma4 >= 0 && wide4 >= 0 && lds6 >= 0 && dma6 >= 0 && lds8 >= 0 &&
                    wide8 >= 0 && dma12 >= 0 && wide12 >= 0,
                "not in its table");
  switch (cout) {
    case 32: return dma2;
    case 64: return pixels >= 200000 ? wide4 : pixels >= 40000 ? dma4 : lds4;
    case 96: return pixels >= 200000 ? dma6 : lds6;
    case 128: return pixels >= 40000 ? wide8 : lds8;
    case 192: return pixels >= 40000 ? wide12 : dma12;
    default: return 0;
  }
}

int conv3x3_head_tile() {
  constexpr int t = tile_index(kTiles2, {2, 2, 2, 2, 2, 4});
  static_assert(t >= 0, "not in its table");
  return t;
}

int conv3x3_tile_pool(int cout, int tile) {
  int n = 0;
  if (cout % 16) return 0;
  const ConvTile *t = conv_tiles(cout / 16, &n);
  return t && tile >= 0 && tile < n && t[tile].lds && t[tile].r % 2 == 0;
}

int conv3x3_tiles(int cout) {
  int n = 0;
  if (cout % 16) return 0;
  (void)conv_tiles(cout / 16, &n);
  return n;
}

template <int MB, int PB, int R> static void launch_conv(const ConvArgs &a, hipStream_t s) {
  dim3 grid((a.w + 4 * PB * 16 - 1) / (4 * PB * 16), (a.h + R - 1) / R, a.n), block(256);
  hipLaunchKernelGGL((conv3x3_kernel<MB, PB, R>), grid, block, 0, s, a);
}

static int cu_count() {
  static int cus = 0;
  if (!cus) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) ==
                                                hipSuccess && v > 0)
      cus = v;
    else
      cus = 256;
  }
  return cus;
}

template <int MBW, int WR, int WP> static void launch_conv_lds(const ConvArgs &a, int per_cu, hipStream_t s) {
  const int tx = (a.w + 16 * WP - 1) / (16 * WP), ty = (a.h + 4 * WR - 1) / (4 * WR), splits = a.cout / (16 * MBW);
  const long tiles = (long)tx * ty * a.n * splits;
  long grid = per_cu > 0 ? std::min(tiles, (long)per_cu * cu_count()) : tiles;
  if constexpr (WR % 2 == 0) {
    if (a.up_out) {
      hipLaunchKernelGGL((conv3x3_lds_kernel<MBW, WR, WP, true>), dim3((unsigned)grid), dim3(256), 0, s, a,
                         tx, ty, splits);
      return;
    }
  }
  hipLaunchKernelGGL((conv3x3_lds_kernel<MBW, WR, WP>), dim3((unsigned)grid), dim3(256), 0, s, a, tx, ty,
                     splits);
}

// Weights resident when two input buffers and all chunks' weights leave room
// for `per_cu` workgroups' LDS; a tile shape that does not fit either way is
// an error (none of the network's layers).
template <int MBW, int WR, int WP, int NW> static hipError_t launch_conv_dma(const ConvArgs &a, int per_cu, hipStream_t s) {
  const int tx = (a.w + 16 * WP - 1) / (16 * WP), ty = (a.h + NW * WR - 1) / (NW * WR), splits = a.cout / (16 * MBW);
  const int chunks = (a.ca + a.cb) / 32, cap = 160 * 1024 / per_cu;
  const bool head = a.head_out != nullptr;
  const int wres = dma_lds_bytes(MBW, WR, WP, NW, head, chunks) <= cap ? 1 : 0;
  const int lds = dma_lds_bytes(MBW, WR, WP, NW, head, wres ? chunks : 2);
  if (lds > 160 * 1024 || (conv_pairs(MBW) && a.split % 32)) return hipErrorInvalidValue;
  const long tiles = (long)tx * ty * a.n;
  const long grid = std::min(tiles, std::max(1L, (long)per_cu * cu_count() / splits)) * splits;
  constexpr int OCC = NW * ((NW == 4 && MBW == 2 && WR * WP == 4) || WR * WP == 2 ? 2 : 1) / 4;
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * NW), (size_t)lds, s, a, tx, ty, splits, wres);
    return hipGetLastError();
  };
  if constexpr (MBW == 2 && NW == 4) {
    if (head) return launch(conv3x3_dma_kernel<MBW, WR, WP, NW, OCC, true, false>);
  }
  if (head) return hipErrorInvalidValue;
  if (a.up_out) return launch(conv3x3_dma_kernel<MBW, WR, WP, NW, OCC, false, true>);
  return launch(conv3x3_dma_kernel<MBW, WR, WP, NW, OCC, false, false>);
}

template <int MB> static hipError_t conv_mb(const ConvArgs &a, const ConvTile &t, hipStream_t s) {
#define LGX_CASE(RR, PP) \
  if (!t.lds && t.r == RR && t.pb == PP) { \
    launch_conv<MB, PP, RR>(a, s); \
    return hipGetLastError(); \
  }
#define LGX_LDS(MBW, RR, PP) \
  if (t.lds == 1 && t.mbw == MBW && t.r == RR && t.pb == PP) { \
    launch_conv_lds<MBW, RR, PP>(a, t.per_cu, s); \
    return hipGetLastError(); \
  }
  if constexpr (MB <= 2) {
    LGX_CASE(4, 2) LGX_CASE(2, 4) LGX_CASE(4, 4) LGX_CASE(1, 4)
  } else if constexpr (MB <= 4) {
    LGX_CASE(2, 2) LGX_CASE(4, 2) LGX_CASE(2, 4) LGX_CASE(1, 4)
  } else if constexpr (MB <= 8) {
    LGX_CASE(2, 2) LGX_CASE(1, 4) LGX_CASE(1, 2)  // covers the MB = 6 and MB = 8 tables
  } else {
    LGX_CASE(1, 2) LGX_CASE(2, 1)
  }
#define LGX_DMA(MBW, RR, PP, NW) \
  if (t.lds == 2 && t.mbw == MBW && t.r == RR && t.pb == PP && t.nw == NW) \
    return launch_conv_dma<MBW, RR, PP, NW>(a, t.per_cu, s);
  if constexpr (MB == 6) {
    LGX_DMA(2, 2, 1, 8)
  }
  if constexpr (MB % 2 == 0) {
    LGX_DMA(2, 2, 2, 4) LGX_DMA(2, 2, 2, 8)
    LGX_LDS(2, 2, 4) LGX_LDS(2, 2, 2) LGX_LDS(2, 1, 4)
  }
  if constexpr (MB % 4 == 0) {
    LGX_DMA(4, 2, 2, 4) LGX_DMA(4, 2, 2, 8)
    LGX_LDS(4, 2, 2) LGX_LDS(4, 1, 4) LGX_LDS(4, 1, 2)
  }
#undef LGX_CASE
#undef LGX_LDS
#undef LGX_DMA
  return hipErrorInvalidValue;
}

hipError_t conv3x3(const ConvArgs &a, hipStream_t s) {
  if (a.cout % 16 || (a.bias != nullptr) != (a.relu != 0)) return hipErrorInvalidValue;
  if (a.head_out && (a.cout != 32 || !a.head_in || a.tile != conv3x3_head_tile())) return hipErrorInvalidValue;
  if (a.gin_fmt) return hipErrorInvalidValue;  // records packed while staging: conv_first_pair
  if (a.pool_out && (a.head_out || a.mask0 || a.mask1 || !conv3x3_tile_pool(a.cout, a.tile)))
    return hipErrorInvalidValue;
  if (a.up_out && (a.head_out || a.pool_out || a.mask0 || !a.up_mask || a.split < 16 || a.h % 2 || a.w % 2 ||
                   !conv3x3_tile_pool(a.cout, a.tile)))
    return hipErrorInvalidValue;
  if (a.split < 0 || a.split > a.cout || a.split % 16) return hipErrorInvalidValue;  // whole 16-channel blocks
  const int mb = a.cout / 16;
  int n = 0;
  const ConvTile *tiles = conv_tiles(mb, &n);
  if (!tiles || a.tile < 0 || a.tile >= n) return hipErrorInvalidValue;
  const ConvTile &t = tiles[a.tile];
  switch (mb) {
    case 1: return conv_mb<1>(a, t, s);
    case 2: return conv_mb<2>(a, t, s);
    case 4: return conv_mb<4>(a, t, s);
    case 6: return conv_mb<6>(a, t, s);
    case 8: return conv_mb<8>(a, t, s);
    case 12: return conv_mb<12>(a, t, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t conv_first_pair(const ConvArgs &a0, const ConvArgs &a1, hipStream_t s) {
  if (a0.gin_fmt < 1 || a0.gin_fmt > 3 || (a0.gin_fmt == 3 ? !a0.gin_x12 : a0.n != 1) || a0.n < 1 ||
      a0.cout != 32 || !a0.wt || !a0.bias || a1.n != a0.n || a1.cout != 32 || a1.split != 32 || !a1.out0 ||
      !a1.pool_out || !a1.wt || !a1.bias || a1.h != a0.h || a1.w != a0.w || a0.h < 1 || a0.w < 1 ||
      (a0.out0 != nullptr) != (a0.gin_fmt == 3) || (a0.rec_out != nullptr) != (a0.gin_fmt == 3))
    return hipErrorInvalidValue;
  // Row pairs per segment: of the lengths that fill one to four rounds of the waves that are resident at once
  // (2 per SIMD) the one that ends first, a segment's first rows counted as 0.4 of an iteration.
  const int strips = (a0.w + kPairCols - 1) / kPairCols, pairs = (a0.h + 1) / 2;
  const long waves = 8L * cu_count(), columns = (long)strips * a0.n;
  int len = pairs, segs = 1;
  long best = LONG_MAX;
  for (long r = 1; r <= 4; r++) {
    const long want = std::min((long)pairs, std::max(1L, r * waves / columns)), l = (pairs + want - 1) / want,
               k = (pairs + l - 1) / l, cost = (columns * k + waves - 1) / waves * (5 * l + 2);
    if (cost < best) {
      best = cost;
      len = (int)l;
      segs = (int)k;
    }
  }
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)((long)strips * segs * a0.n)), dim3(64), 0, s, a0, a1, strips, segs, len);
  };
  if (a0.gin_fmt == 1)
    launch(conv_first_pair_kernel<1, false>);
  else if (a0.gin_fmt == 2)
    launch(conv_first_pair_kernel<2, false>);
  else
    launch(conv_first_pair_kernel<3, true>);
  return hipGetLastError();
}

// Rows of a strip per wave of conv3x3_wgrad_kernel: at least 2.
static constexpr int kWgradMinRows = 2;

size_t conv3x3_wgrad_scratch_bytes() {
  // a task has 9 x 32 x 32 sums, and at most 32 channels' bias slots; a launch's tasks are at most the CUs or,
  // with one each, the units of its layers (52 in the network)
  return (size_t)kWgradLaunches * (cu_count() + 64) * (9 * 32 * 32 + 32) * 4;
}

// The units of a launch's layers are divided into tasks of about equal work, as many as there are CUs (a workgroup's
// LDS takes a CU): the least work T per task for which the sum over layers of units * ceil(work of a unit / T)
// fits.  A launch has about 10 us of its own (its start, the first loads, the last sums).
hipError_t conv3x3_wgrad(WgradTable &t, float *part, size_t part_bytes, hipStream_t s) {
  if (t.done < 0 || t.n <= t.done || t.n > 10 || !part) return hipErrorInvalidValue;
  const int l0 = t.done;
  long items[10], units[10], most = 0;
  for (int l = l0; l < t.n; l++) {
    const WgradArgs &a = t.l[l];
    if (a.cout != 32 && a.cout != 64 && a.cout != 128) return hipErrorInvalidValue;
    if ((a.ca + a.cb) % 32 || a.ca % 32 || a.n < 1 || a.h < 1 || a.w < 1 || !a.dw || !a.db || a.cin_log < 1 ||
        a.cin_log > a.ca + a.cb || (a.cin_log <= 16 && a.ca + a.cb != 32))
      return hipErrorInvalidValue;
    items[l] = (long)a.n * ((a.w + 31) / 32) * a.h;  // rows of strips
    if (items[l] > INT_MAX / 2) return hipErrorInvalidValue;
    units[l] = (long)(a.ca + a.cb) / 32 * (a.cout / 32);
    most = std::max(most, items[l]);
  }
  // (a unit with half of the matrix work counts half, though its loads are the same)
  auto slots_of = [&](int l, long T) {
    const long per = kWgradWaves * std::max((long)kWgradMinRows, (T * (t.l[l].cin_log <= 16 ? 2 : 1) + kWgradWaves - 1) / kWgradWaves);
    return (items[l] + per - 1) / per;
  };
  auto tasks_of = [&](long T) {
    long k = 0;
    for (int l = l0; l < t.n; l++) k += units[l] * slots_of(l, T);
    return k;
  };
  long lo = 0, hi = most;  // hi fits, or is the fewest tasks there are
  while (hi - lo > 1) {
    const long mid = (lo + hi) / 2;
    (tasks_of(mid) <= cu_count() ? hi : lo) = mid;
  }
  size_t used = t.used;
  int blocks = t.first[l0], sums = t.reduce[l0];
  const int block0 = blocks;
  for (int l = l0; l < t.n; l++) {
    WgradArgs &a = t.l[l];
    long slots = slots_of(l, hi);
    a.rows = (int)((items[l] + slots * kWgradWaves - 1) / (slots * kWgradWaves));
    slots = (items[l] + (long)a.rows * kWgradWaves - 1) / ((long)a.rows * kWgradWaves);
    a.slots = (int)slots;
    // a piece's rows (two more are read) within 2 GB of its first
    a.cap = (int)std::max(1L, std::min((long)a.h, 0x7fffffffL / ((long)a.w * 2 * std::max({a.ca, a.cb, a.cout})) - 3));
    a.part = part + used;
    used += (size_t)units[l] * slots * 9 * 32 * 32;
    a.part_b = part + used;
    used += (size_t)slots * a.cout;
    t.first[l] = blocks;
    t.reduce[l] = sums;
    blocks += (int)(units[l] * slots);
    sums += (int)(units[l] * 9 * 32 * 32 / 4 / kReduceEl) + 1;
  }
  t.first[t.n] = blocks;
  t.reduce[t.n] = sums;
  if (used * 4 > part_bytes) return hipErrorInvalidValue;
  const size_t lds = std::max(kWgradLds, wgrad_sums<2>() * 1024 * kWgradWaves / 2);
  t.used = used;
  t.done = t.n;
  hipLaunchKernelGGL(conv3x3_wgrad_kernel, dim3((unsigned)(blocks - block0)), dim3(64 * kWgradWaves), lds, s, t, l0);
  return hipGetLastError();
}

hipError_t conv3x3_wgrad_sums(const WgradTable &t, hipStream_t s) {
  if (t.n < 1 || t.done != t.n) return hipErrorInvalidValue;
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)t.reduce[t.n]), dim3(256), 0, s, t);
  return hipGetLastError();
}

hipError_t avgpool(const bf16 *x, int n, int h, int w, int c, bf16 *y, hipStream_t s) {
  hipLaunchKernelGGL(avgpool_kernel, dim3(grid_for((size_t)n * (h / 2) * (w / 2) * (c / 8), 256)), dim3(256), 0, s, x,
                     n, h, w, c, y);
  return hipGetLastError();
}
hipError_t pool_bwd_add(const bf16 *dx_in, const bf16 *dpool, const bf16 *act, int n, int h, int w, int c, bf16 *dx,
                        hipStream_t s) {
  if (c % 8 || (c / 8) & (c / 8 - 1) || h < 2 || w < 2) return hipErrorInvalidValue;
  const unsigned bx = (unsigned)std::min((w * (c / 8) + 255) / 256, 64);
  hipLaunchKernelGGL(pool_bwd_add_kernel, dim3(bx, (unsigned)std::min(n * h, 65535)), dim3(256), 0, s, dx_in, dpool,
                     act, n, h, w, c, dx);
  return hipGetLastError();
}
hipError_t upsample_bwd(const bf16 *dfull, const bf16 *act, int n, int hh, int ww, int c, bf16 *dhalf, hipStream_t s) {
  hipLaunchKernelGGL(upsample_bwd_kernel, dim3(grid_for((size_t)n * hh * ww * (c / 8), 256)), dim3(256), 0, s, dfull,
                     act, n, hh, ww, c, dhalf);
  return hipGetLastError();
}
hipError_t head_train(const bf16 *d1, const float *x12, const float4 *target, const float *wh, const float *bh,
                      size_t npix, float inv_count, int l2, bf16 *dd1, float *dwh, float *dbh, float *loss,
                      hipStream_t s) {
  // persistent: about two workgroups per CU, so as many atomic sums per head parameter
  const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(2 * cu_count(), (npix + 255) / 256));
  hipLaunchKernelGGL(head_train_kernel, dim3(blocks), dim3(256), 0, s, d1, x12, target, wh, bh, npix, inv_count, l2,
                     dd1, dwh, dbh, loss);
  return hipGetLastError();
}
hipError_t adam_pack(float *p, const float *g, float *m, float *v, size_t n, float lr, float b1, float b2, float eps,
                     float bc1, float bc2, const PackTable &pk, hipStream_t s) {
  hipLaunchKernelGGL(adam_pack_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, g, m, v, n, lr, b1, b2, eps, bc1,
                     bc2, pk);
  return hipGetLastError();
}

hipError_t fill(float *p, size_t n, float v, hipStream_t s) {
  hipLaunchKernelGGL(fill_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}
hipError_t pack_weights(const float *w, int cout, int cin_log, int cin_pad, bf16 *wf, bf16 *wt, hipStream_t s) {
  hipLaunchKernelGGL(pack_weights_kernel, dim3(grid_for((size_t)cout * cin_pad * 9, 256)), dim3(256), 0, s, w, cout,
                     cin_log, cin_pad, wf, wt);
  return hipGetLastError();
}
hipError_t mfma_probe(const float *A, const float *B, float *D, hipStream_t s) {
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, s, A, B, D);
  return hipGetLastError();
}

}  // namespace unet
}  // namespace lgx
