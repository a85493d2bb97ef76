// Parallel- and fan-beam 2D projector / backprojector for gfx950.
//
// The reference runs all four 2D kernels on the CUDA texture unit (linear
// filter, border addressing, unnormalised coordinates).  gfx950 has no image
// sampler, so the texture fetch is done in software: the coordinate c handed
// to the sampler is formed exactly as the reference forms it
// (physical_to_index(p) + 0.5f), then b = c - 0.5f, i = floor(b), weights
// b - i (exact, not 8-bit), neighbours outside the array read 0.
//
// The 2D problems are small (a 512^2 image is 1 MiB), so the samplers test
// bounds per neighbour instead of reading a zero-apron copy.  With f32 storage the two
// x neighbours of a row are adjacent: when both lie inside the row, one 8-byte load reads
// them (dword aligned; the target's vector loads do not need natural alignment), which
// halves the loads of a sample without changing any value.
#include "common.h"

namespace pyronn {

typedef float f32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

// img[i], img[i + 1] as one load
__device__ __forceinline__ f32x2_a4 load_pair(const float *__restrict__ img, size_t i) {
  return *reinterpret_cast<const f32x2_a4 *>(img + i);
}

constexpr float kPi = 3.14159265359f;  // par_backprojector_2D_CudaKernel.cu.cc:32

// helper_grid.h:23-31
__device__ __forceinline__ float i2p(float i, float o, float s) { return fmaf(i, s, o); }
__device__ __forceinline__ float p2i(float p, float o, float s) { return (p - o) / s; }

// 1 / s when s is a positive power of two well inside the normal range, else 0.  For
// such s, x / s and x * (1 / s) are the correctly rounded value of the same real number,
// so they are equal for every x; the kernels then multiply instead of dividing.
__device__ __forceinline__ float pow2_reciprocal(float s) {
  const unsigned b = __float_as_uint(s);
  const unsigned e = (b >> 23) & 0xffu;
  return ((b & 0x807fffffu) == 0u && e > 1u && e < 253u) ? __uint_as_float((254u - e) << 23) : 0.0f;
}
// physical_to_index with the division replaced by the exact product when POW2
template <bool POW2>
__device__ __forceinline__ float p2i_k(float p, float o, float s, float inv) {
  return POW2 ? (p - o) * inv : (p - o) / s;
}

// The four neighbours a lane read last (consecutive march samples usually share them).
struct Tex2dRegs {
  int x0 = 0x7fffffff, y0 = 0;
  float p00 = 0.f, p01 = 0.f, p10 = 0.f, p11 = 0.f;
};

// tex2d with the neighbours kept in registers across calls: loads only when (x0, y0)
// changes; the same values and the same blend as tex2d.
template <typename TS>
__device__ __forceinline__ float tex2d_cached(const TS *__restrict__ img, int W, int H, float cx,
                                              float cy, Tex2dRegs &r) {
  float bx = cx - 0.5f, by = cy - 0.5f;
  if (!(bx > -2.0f && bx < (float)(W + 1) && by > -2.0f && by < (float)(H + 1))) return 0.0f;
  const float fx = floorf(bx), fy = floorf(by);
  const int x0 = (int)fx, y0 = (int)fy;
  if (x0 != r.x0 || y0 != r.y0) {
    r.x0 = x0;
    r.y0 = y0;
    const int x1 = x0 + 1, y1 = y0 + 1;
    const bool vx0 = x0 >= 0 && x0 < W, vx1 = x1 >= 0 && x1 < W;
    const bool vy0 = y0 >= 0 && y0 < H, vy1 = y1 >= 0 && y1 < H;
    if (sizeof(TS) == 4 && vx0 && vx1) {
      const float *f = reinterpret_cast<const float *>(img);
      const f32x2_a4 a = vy0 ? load_pair(f, (size_t)y0 * W + x0) : f32x2_a4{0.0f, 0.0f};
      const f32x2_a4 b = vy1 ? load_pair(f, (size_t)y1 * W + x0) : f32x2_a4{0.0f, 0.0f};
      r.p00 = a.x;
      r.p01 = a.y;
      r.p10 = b.x;
      r.p11 = b.y;
    } else {
      r.p00 = (vx0 && vy0) ? to_f32(img[y0 * W + x0]) : 0.0f;
      r.p01 = (vx1 && vy0) ? to_f32(img[y0 * W + x1]) : 0.0f;
      r.p10 = (vx0 && vy1) ? to_f32(img[y1 * W + x0]) : 0.0f;
      r.p11 = (vx1 && vy1) ? to_f32(img[y1 * W + x1]) : 0.0f;
    }
  }
  const float xd = bx - fx, yd = by - fy;
  const float p0 = lerp_ref(r.p00, r.p01, xd);
  const float p1 = lerp_ref(r.p10, r.p11, xd);
  return lerp_ref(p0, p1, yd);
}

template <typename TS>
__device__ __forceinline__ float tex1d(const TS *__restrict__ row, int W, float cx) {
  const float bx = cx - 0.5f;
  if (!(bx > -2.0f && bx < (float)(W + 1))) return 0.0f;
  const float fx = floorf(bx);
  const int x0 = (int)fx, x1 = x0 + 1;
  float p0, p1;
  if (sizeof(TS) == 4 && x0 >= 0 && x1 < W) {
    const f32x2_a4 a = load_pair(reinterpret_cast<const float *>(row), (size_t)x0);
    p0 = a.x;
    p1 = a.y;
  } else {
    p0 = (x0 >= 0 && x0 < W) ? to_f32(row[x0]) : 0.0f;
    p1 = (x1 >= 0 && x1 < W) ? to_f32(row[x1]) : 0.0f;
  }
  return lerp_ref(p0, p1, bx - fx);
}

// Ray parameter interval inside the image box, whose edges sit 0.5 mm before each index
// edge (par_projector_2D_CudaKernel.cu.cc:33-57); an axis-parallel ray skips that slab.
__device__ __forceinline__ void clip2d(int W, int H, float ox, float oy, float sx, float sy,
                                       float s0, float s1, float r0, float r1, float &amin,
                                       float &amax) {
  amin = 0.0f;
  amax = __builtin_inff();
  if (0.0f != r0) {
    const float e0 = i2p(0.0f, ox, sx) - 0.5f, e1 = i2p((float)W, ox, sx) - 0.5f;
    const float reci = 1.0f / r0;
    const float a0 = (e0 - s0) * reci, a1 = (e1 - s0) * reci;
    amin = fminf(a0, a1);
    amax = fmaxf(a0, a1);
  }
  if (0.0f != r1) {
    const float e0 = i2p(0.0f, oy, sy) - 0.5f, e1 = i2p((float)H, oy, sy) - 0.5f;
    const float reci = 1.0f / r1;
    const float a0 = (e0 - s1) * reci, a1 = (e1 - s1) * reci;
    amin = fmaxf(amin, fminf(a0, a1));
    amax = fminf(amax, fmaxf(a0, a1));
  }
}

// kernel_project2D, par_projector_2D_CudaKernel.cu.cc:28-102 (same code in
// fan_projector_2D_CudaKernel.cu.cc:27-102): march in mm, box edges with the
// -0.5 mm offset, first sample exactly at the entry point, tail for a positive sum.
template <typename TS, bool POW2>
__device__ float march2d(const TS *__restrict__ img, int W, int H, float ox, float oy, float sx,
                         float sy, float ix, float iy, float s0, float s1, float r0, float r1,
                         float step) {
  if (!(step > 0.0f)) return __builtin_nanf("");
  float amin, amax;
  clip2d(W, H, ox, oy, sx, sy, s0, s1, r0, r1, amin, amax);
  float pix = 0.0f, px = 0.0f, py = 0.0f;
  Tex2dRegs regs;
  const int cap = march_cap(amin, amax, step);
#define PYRONN_TEX2D(X, Y) \
  tex2d_cached(img, W, H, p2i_k<POW2>((X), ox, sx, ix) + 0.5f, p2i_k<POW2>((Y), oy, sy, iy) + 0.5f, regs)
  if (amin < amax) {
    px = fmaf(amin, r0, s0);
    py = fmaf(amin, r1, s1);
    pix = fmaf(0.5f, PYRONN_TEX2D(px, py), pix);
    amin += step;
  }
  for (int it = 0; amin < amax && it < cap; ++it) {
    px = fmaf(amin, r0, s0);
    py = fmaf(amin, r1, s1);
    pix += PYRONN_TEX2D(px, py);
    amin += step;
  }
  pix *= step;
  if (pix > 0.0f) {
    const float flast = PYRONN_TEX2D(px, py);
    pix = fmaf(-(0.5f * step), flast, pix);
    amin -= step;
    const float last = amax - amin;
    pix = fmaf(0.5f * last, flast, pix);
    px = fmaf(amax, r0, s0);
    py = fmaf(amax, r1, s1);
    pix = fmaf(0.5f * last, PYRONN_TEX2D(px, py), pix);
  }
#undef PYRONN_TEX2D
  return pix;
}

// Value of lane J of this lane's quad (DPP quad_perm broadcast; all four lanes active).
template <int J>
__device__ __forceinline__ float quad_bcast(float f) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), J * 0x55, 0xf, 0xf, false));
}

// The march of march2d with the samples of one ray spread over the G = 4 lanes of a quad:
// every lane runs the same alpha recurrence (alpha += step, the same float adds), lane q
// samples positions q, q + G, ... of each group of G, and every lane adds the G values in
// sample order from quad broadcasts, so all G lanes hold the same running sum, bit for bit
// the one-lane sum.  The entrance sample and the tail are computed by all lanes alike.
// Four times the lanes per ray: for launches with too few rays to fill the GPU, where the
// one-lane march is bound by its own load latency (measured on 256^2 / 180 views x 363
// pixels: 0.67 -> 0.35 ms; with 261K rays, 2 or 4 lanes per ray were slower than one).
template <typename TS, bool POW2, int G>
__device__ float march2d_group(const TS *__restrict__ img, int W, int H, float ox, float oy,
                               float sx, float sy, float ix, float iy, float s0, float s1, float r0,
                               float r1, float step, int q) {
  if (!(step > 0.0f)) return __builtin_nanf("");
  float amin, amax;
  clip2d(W, H, ox, oy, sx, sy, s0, s1, r0, r1, amin, amax);
  float pix = 0.0f, alast = 0.0f;
  bool any = false;  // a sample was taken: (px, py) of the one-lane march is at alast
  Tex2dRegs regs;
  const int cap = march_cap(amin, amax, step);
#define PYRONN_TEX2D(X, Y) \
  tex2d_cached(img, W, H, p2i_k<POW2>((X), ox, sx, ix) + 0.5f, p2i_k<POW2>((Y), oy, sy, iy) + 0.5f, regs)
  if (amin < amax) {
    pix = fmaf(0.5f, PYRONN_TEX2D(fmaf(amin, r0, s0), fmaf(amin, r1, s1)), pix);
    alast = amin;
    any = true;
    amin += step;
  }
  for (int it = 0;;) {
    float a[G + 1];
    a[0] = amin;
#pragma unroll
    for (int j = 1; j <= G; ++j) a[j] = a[j - 1] + step;
    // sample j of the group exists iff the one-lane loop would take it: a prefix, as
    // alpha only grows
    bool ok[G];
#pragma unroll
    for (int j = 0; j < G; ++j) ok[j] = (j == 0 || ok[j - 1]) && a[j] < amax && it + j < cap;
    float my_a = a[0];
    bool my_ok = ok[0];
#pragma unroll
    for (int j = 1; j < G; ++j) {
      my_a = q == j ? a[j] : my_a;
      my_ok = q == j ? ok[j] : my_ok;
    }
    float f = 0.0f;
    if (my_ok) f = PYRONN_TEX2D(fmaf(my_a, r0, s0), fmaf(my_a, r1, s1));
    static_assert(G == 4, "quad broadcasts");
    const float fg[G] = {quad_bcast<0>(f), quad_bcast<1>(f), quad_bcast<2>(f), quad_bcast<3>(f)};
    int c = 0;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if (ok[j]) pix += fg[j];
      c += ok[j] ? 1 : 0;
    }
    if (c > 0) {
      alast = a[c - 1];
      any = true;
    }
    amin = a[c];
    it += c;
    if (c < G) break;
  }
  pix *= step;
  if (pix > 0.0f) {
    float px = 0.0f, py = 0.0f;
    if (any) {
      px = fmaf(alast, r0, s0);
      py = fmaf(alast, r1, s1);
    }
    const float flast = PYRONN_TEX2D(px, py);
    pix = fmaf(-(0.5f * step), flast, pix);
    amin -= step;
    const float last = amax - amin;
    pix = fmaf(0.5f * last, flast, pix);
    px = fmaf(amax, r0, s0);
    py = fmaf(amax, r1, s1);
    pix = fmaf(0.5f * last, PYRONN_TEX2D(px, py), pix);
  }
#undef PYRONN_TEX2D
  return pix;
}

// =====================================================================================
// Forward through a pair copy of the image.  Element (x, y) of the copy holds the column
// pair [v(x, y), v(x, y + 1)], x in [-2, W + 1], y in [-2, H], x fastest, zeros outside
// the image; the elements of x and x + 1 together are the four neighbours of cell (x, y),
// so a sample is ONE load at element alignment (16 bytes f32, 8 bytes 16-bit types) and
// needs no bounds test: the coordinate is clamped into [-2, W] x [-2, H], where the cells
// outside [-1, W) hold zeros only, exactly what the reference's border gives.
//
// What bound the direct march (march2d above): about 100 VALU instructions per sample (the
// neighbours' bounds tests, 64-bit addresses and selects of the shared-ray version, the
// iteration cap) around loads whose latency nothing covered.  Here a sample takes 39, and a
// wave's load 22 cycles of the texture-address unit (16 for one 128-byte line per quad): in a batch
// that unit is 90% busy, the data-return unit 98% and VALU issue at 0.41 of its 0.5 per SIMD and cycle;
// one image ends on its longest rays, with half its waves gone on average.  Parallel
// 256^2 / 180 views x 363 / step 0.2: 32 images 4300 -> 1390 us, one 282 -> 83; fan 512^2 /
// 360 x 725 / step 0.5: 535 -> 158; fan 301 x 277 f16, spacing 0.7, one image: 522 -> 124.
// A second copy with x and y exchanged, for rays along y, was no faster (1496 us, 180 us):
// a quad's four samples span less than two pixels at these steps.
// =====================================================================================
template <typename TS> struct PairLoad {
  typedef uint32_t raw __attribute__((ext_vector_type(2), aligned(4)));
  static constexpr int kShift = 2;  // bytes of an element, log2
};
template <> struct PairLoad<float> {
  typedef float raw __attribute__((ext_vector_type(4), aligned(8)));
  static constexpr int kShift = 3;
};

__host__ __device__ inline int pair_cols(int W) { return W + 4; }
__host__ __device__ inline int pair_rows(int H) { return H + 3; }

// Lanes of a 256-lane layout block that share a row of `cols` elements, log2: a block takes several short
// rows, as one each would leave most of its lanes idle and the launch bound by its blocks (a parallel
// projection of a 65000 x 4 image 34 -> 8 us; a backprojection of 8 views to 4096 images of 8 x 8, with one
// pixel per lane, 30 -> 12).
static int layout_lanes(int cols) {
  int s = 3;
  while (s < 8 && (1 << s) < cols) ++s;
  return s;
}

// One lane per element, 1 << lanes columns of 256 >> lanes rows per block.
template <typename TS>
__global__ void __launch_bounds__(256)
build_pairs_kernel(const TS *__restrict__ img, TS *__restrict__ pairs, int H, int W, int lanes) {
  const int cx = (blockIdx.x << lanes) + (threadIdx.x & ((1 << lanes) - 1));
  const int cy = blockIdx.y * (256 >> lanes) + (threadIdx.x >> lanes);
  const int Wp = pair_cols(W);
  if (cx >= Wp || cy >= pair_rows(H)) return;
  const TS *im = img + (size_t)blockIdx.z * H * W;
  const int x = cx - 2, y = cy - 2;
  const bool vx = x >= 0 && x < W;
  TS e[2];
  e[0] = (vx && y >= 0 && y < H) ? im[(size_t)y * W + x] : zero_of<TS>();
  e[1] = (vx && y + 1 >= 0 && y + 1 < H) ? im[(size_t)(y + 1) * W + x] : zero_of<TS>();
  TS *o = pairs + (((size_t)blockIdx.z * pair_rows(H) + cy) * Wp + cx) * 2;
  if constexpr (sizeof(TS) == 4) {
    *reinterpret_cast<float2 *>(o) = make_float2(e[0], e[1]);
  } else {
    uint32_t w;
    __builtin_memcpy(&w, e, 4);
    *reinterpret_cast<uint32_t *>(o) = w;
  }
}

// The image as the march sees it.  base is the pair copy moved by kPairBias bytes (see
// pair_offset); fWp the copy's row length; c0 the float bias of the element index.
struct PairImage {
  const char *base;
  float fWp, c0, fW, fH;
};

// Byte offset of cell (fx, fy) from PairImage::base.  fx + c0 and fy fWp + (fx + c0) are
// exact integer-valued floats in [2^23, 2^24) (the host keeps the copy below 2^23
// elements), so the bit pattern of the latter is 0x4B000000 + element index, and the shift
// makes it 2^shift index + (0x4B000000 << shift) mod 2^32, which the base subtracts.
template <typename TS>
__device__ __forceinline__ uint32_t pair_offset(const PairImage &im, float fx, float fy) {
  return __float_as_uint(fmaf(fy, im.fWp, fx + im.c0)) << PairLoad<TS>::kShift;
}
template <typename TS>
__device__ __forceinline__ PairImage pair_image(const TS *pairs, int H, int W) {
  constexpr uint32_t bias = 0x4B000000u << PairLoad<TS>::kShift;
  const int Wp = pair_cols(W);
  return {reinterpret_cast<const char *>(pairs) - (size_t)bias, (float)Wp, 0x1p23f + (float)(2 * Wp + 2), (float)W,
          (float)H};
}

// x / s for the sampler, s the same for a whole image.
//  kDivPow2: s a power of two, the exact product (pow2_reciprocal);
//  kDivRefine: q = x RN(1/s), then twice q + (x - q s) RN(1/s).  The first correction leaves
//    less than one ulp of error; from such a q, whose residual one FMA forms exactly, and a
//    correctly rounded reciprocal the second gives the correctly rounded quotient
//    (Markstein 1990), for s in [2^-60, 2^60].  Where a residual may be inexact or a product
//    overflow (|x| < 2^-101, |x| > 2^67, infinities) the quotient may differ from x / s, but
//    its sample does not: such a tiny quotient vanishes in (q + 0.5) - 0.5, and infinite,
//    huge or NaN coordinates all sample zeros;
//  kDivIeee: the division, for any s.
enum { kDivPow2 = 1, kDivRefine = 2, kDivIeee = 0 };
template <int DIV>
__device__ __forceinline__ float div_spacing(float x, float s, float inv) {
  if (DIV == kDivPow2) return x * inv;
  if (DIV == kDivIeee) return x / s;
  float q = x * inv;
  q = fmaf(fmaf(-q, s, x), inv, q);
  return fmaf(fmaf(-q, s, x), inv, q);
}

struct Ray2d {
  float ox, oy, sx, sy, ix, iy, s0, s1, r0, r1;
};

// Cell and fractions of the sample at alpha a, and its load.
template <typename TS, int DIV>
__device__ __forceinline__ typename PairLoad<TS>::raw fetch2d(const PairImage &im, const Ray2d &r, float a,
                                                              float &xd, float &yd) {
  const float cx = div_spacing<DIV>(fmaf(a, r.r0, r.s0) - r.ox, r.sx, r.ix) + 0.5f;
  const float cy = div_spacing<DIV>(fmaf(a, r.r1, r.s1) - r.oy, r.sy, r.iy) + 0.5f;
  const float bx = __builtin_amdgcn_fmed3f(cx - 0.5f, -2.0f, im.fW);
  const float by = __builtin_amdgcn_fmed3f(cy - 0.5f, -2.0f, im.fH);
  const float fx = floorf(bx), fy = floorf(by);
  xd = bx - fx;
  yd = by - fy;
  return *reinterpret_cast<const typename PairLoad<TS>::raw *>(im.base + pair_offset<TS>(im, fx, fy));
}

__device__ __forceinline__ float blend_pairs(float, PairLoad<float>::raw v, float xd, float yd) {
  return lerp_ref(lerp_ref(v.x, v.z, xd), lerp_ref(v.y, v.w, xd), yd);
}
template <typename TS>
__device__ __forceinline__ float blend_pairs(TS, typename PairLoad<TS>::raw v, float xd, float yd) {
  TS a[2], b[2];
  const uint32_t w0 = v.x, w1 = v.y;
  __builtin_memcpy(a, &w0, 4);
  __builtin_memcpy(b, &w1, 4);
  return lerp_ref(lerp_ref(to_f32(a[0]), to_f32(b[0]), xd), lerp_ref(to_f32(a[1]), to_f32(b[1]), xd), yd);
}

// Value of lane J of this lane's quad, and of the lane N (4, 8 or 12) places on in its row of
// 16 (DPP; all lanes of the wave are active).
template <int J> __device__ __forceinline__ float quad_value(float f) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), J * 0x55, 0xf, 0xf, true));
}
template <int N> __device__ __forceinline__ float row_ahead(float f) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), 0x100 + N, 0xf, 0xf, true));
}
// pix + f(0) + f(1) + ... over the G lanes of a group, in lane order; right in the group's
// first quad, which is enough.
__device__ __forceinline__ float quad_sum(float pix, float f) {
  pix += quad_value<0>(f);
  pix += quad_value<1>(f);
  pix += quad_value<2>(f);
  return pix + quad_value<3>(f);
}
template <int G> __device__ __forceinline__ float group_sum(float pix, float f) {
  static_assert(G == 4 || G == 8 || G == 16, "quads of one row of lanes");
  pix = quad_sum(pix, f);
  if constexpr (G >= 8) pix = quad_sum(pix, row_ahead<4>(f));
  if constexpr (G >= 16) {
    pix = quad_sum(pix, row_ahead<8>(f));
    pix = quad_sum(pix, row_ahead<12>(f));
  }
  return pix;
}
// The largest f of the group, in its first quad.
template <int G> __device__ __forceinline__ float group_max(float f) {
  if constexpr (G >= 16) f = fmaxf(f, row_ahead<8>(f));
  if constexpr (G >= 8) f = fmaxf(f, row_ahead<4>(f));
  return fmaxf(fmaxf(quad_value<0>(f), quad_value<1>(f)), fmaxf(quad_value<2>(f), quad_value<3>(f)));
}

// Emits nothing; the compiler moves no load across it (it would sink the load of the next
// round below the loop's exit test, next to its use).
__device__ __forceinline__ void keep_load_here() { asm volatile("" ::: "memory"); }

// The march of march2d with the samples of one ray spread over G lanes: lane q of the group
// takes samples q, q + G, ...  Each lane steps its own alpha by G float additions of step,
// which are the additions of the one-lane recurrence, and the lanes of the group's first quad
// add the G values of a round in sample order: the one-lane sum, bit for bit.  A lane past the
// end (alpha only grows, so the samples that exist are a prefix of a round) adds -0.0, which
// changes no float.  Quads stop by themselves, by their first lane's alpha (their loads then
// cost the address path next to nothing: 638 against 656 us for a step of 6 fan images), larger
// groups with the wave's last ray.  The load of the next round is
// issued before the current one is blended; positions past the end are clamped into the copy
// like any other.  The entrance sample and the tail are computed by all lanes alike.  CAP: with
// the reference march's iteration cap (see proj2d_pairs_kernel).  The result is right in the
// group's first quad.
template <typename TS, int DIV, bool CAP, int G>
__device__ __forceinline__ float march2d_pairs(const PairImage &im, const Ray2d &r, float amin, float amax,
                                               float step, int q) {
  typedef typename PairLoad<TS>::raw raw;
  const bool any = amin < amax;
  const int cap = CAP ? march_cap(amin, amax, step) : 0;
  float xa, ya, xb, yb;
  raw va = fetch2d<TS, DIV>(im, r, amin, xa, ya), vb;
  float pix = any ? fmaf(0.5f, blend_pairs(TS{}, va, xa, ya), 0.0f) : 0.0f;
  float last = amin;  // alpha of this lane's last sample so far
  float a = amin + step;
#pragma unroll
  for (int j = 1; j < G; ++j) {
    const float nx = a + step;
    a = q >= j ? nx : a;
  }
  int it = q;
  va = fetch2d<TS, DIV>(im, r, a, xa, ya);
  // two rounds per pass, so that no cell moves between registers
  const auto more = [&] {
    if constexpr (G == 4) return quad_value<0>(a) < amax && (!CAP || it - q < cap);
    return (bool)__any(a < amax && (!CAP || it < cap));
  };
  while (more()) {
    float an = a;
#pragma unroll
    for (int j = 0; j < G; ++j) an += step;
    vb = fetch2d<TS, DIV>(im, r, an, xb, yb);
    const bool oka = a < amax && (!CAP || it < cap);
    last = oka ? a : last;
    pix = group_sum<G>(pix, oka ? blend_pairs(TS{}, va, xa, ya) : -0.0f);
    a = an;
#pragma unroll
    for (int j = 0; j < G; ++j) a += step;
    va = fetch2d<TS, DIV>(im, r, a, xa, ya);
    const bool okb = an < amax && (!CAP || it + G < cap);
    last = okb ? an : last;
    pix = group_sum<G>(pix, okb ? blend_pairs(TS{}, vb, xb, yb) : -0.0f);
    it += 2 * G;
    keep_load_here();
  }
  pix *= step;
  const float alast = group_max<G>(last);
  if (any && pix > 0.0f) {
    va = fetch2d<TS, DIV>(im, r, alast, xa, ya);
    vb = fetch2d<TS, DIV>(im, r, amax, xb, yb);
    const float flast = blend_pairs(TS{}, va, xa, ya);
    pix = fmaf(-(0.5f * step), flast, pix);
    const float rest = amax - ((alast + step) - step);
    pix = fmaf(0.5f * rest, flast, pix);
    pix = fmaf(0.5f * rest, blend_pairs(TS{}, vb, xb, yb), pix);
  }
  return pix;
}

// Source and direction of the ray of detector pixel d in one view.
// Parallel: project_2Dpar_beam_kernel, par_projector_2D_CudaKernel.cu.cc:104-147.
// Fan:      project_2Dfan_beam_kernel, fan_projector_2D_CudaKernel.cu.cc:104-149.
template <bool FAN>
__device__ __forceinline__ void ray2d(const float *__restrict__ ray, const float *__restrict__ vorigin, float dorigin,
                                      const float *__restrict__ vspacing, float dspacing,
                                      const float *__restrict__ sid_p, const float *__restrict__ sdd_p, int H, int W,
                                      int d, float &ox, float &oy, float &sx, float &sy, float &s0, float &s1,
                                      float &r0, float &r1) {
  sx = vspacing[1];
  sy = vspacing[0];
  ox = vorigin[1];
  oy = vorigin[0];
  const float c0 = ray[0], c1 = ray[1];
  const float u0 = -c1, u1 = c0;
  const float u = i2p((float)d, dorigin, dspacing);
  if (!FAN) {
    const float a = (((float)W * sx) * (float)W) * sx;
    const float sid = sqrtf(fmaf(((float)H * sy) * (float)H, sy, a)) * 1.2f;
    s0 = fmaf(u0, u, c0 * (-sid));
    s1 = fmaf(u1, u, c1 * (-sid));
    r0 = c0;
    r1 = c1;
  } else {
    const float sid = *sid_p, sdd = *sdd_p;
    s0 = c0 * (-sid);
    s1 = c1 * (-sid);
    const float dx = fmaf(u0, u, fmaf(c0, sdd, s0));
    const float dy = fmaf(u1, u, fmaf(c1, sdd, s1));
    const float ex = dx - s0, ey = dy - s1;
    const float nrm = 1.0f / sqrtf(fmaf(ey, ey, ex * ex));
    r0 = ex * nrm;
    r1 = ey * nrm;
  }
}

// One projection reading the pair copy: G lanes per (detector pixel, view), batch items in
// blockIdx.z.  A ray needs no iteration cap when step >= 2^-20 |alpha| over its interval
// (at least 8 ulp of alpha, so each addition advances by at least 15/16 step and the march
// ends before the cap of 1.25 (amax - amin) / step + 16); the choice is uniform per wave and
// never changes a result.
template <typename TS, bool FAN, int G>
__global__ void __launch_bounds__(64)
proj2d_pairs_kernel(const TS *__restrict__ pairs, float *__restrict__ sino, const float *__restrict__ rays,
                    const float *__restrict__ vorigin, const float *__restrict__ dorigin,
                    const float *__restrict__ vspacing, const float *__restrict__ dspacing,
                    const float *__restrict__ sid_p, const float *__restrict__ sdd_p, int H, int W, int n, int det,
                    float step_factor) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int d = t / G, q = t % G;
  const int view = blockIdx.y, b = blockIdx.z;
  if (d >= det) return;  // the G lanes of a pixel share d
  const size_t vb = (size_t)b * n + view;
  Ray2d r;
  ray2d<FAN>(rays + vb * 2, vorigin + b * 2, dorigin[b], vspacing + b * 2, dspacing[b], sid_p + b, sdd_p + b, H, W, d,
             r.ox, r.oy, r.sx, r.sy, r.s0, r.s1, r.r0, r.r1);
  const float step = step_factor * fminf(r.sx, r.sy);
  float amin, amax;
  clip2d(W, H, r.ox, r.oy, r.sx, r.sy, r.s0, r.s1, r.r0, r.r1, amin, amax);
  const PairImage im = pair_image(pairs + (size_t)b * pair_rows(H) * pair_cols(W) * 2, H, W);
  r.ix = pow2_reciprocal(r.sx);
  r.iy = pow2_reciprocal(r.sy);
  const bool pow2 = r.ix != 0.0f && r.iy != 0.0f;  // spacings are per batch item: uniform over the block
  const bool mid = fminf(r.sx, r.sy) >= 0x1p-60f && fmaxf(r.sx, r.sy) <= 0x1p60f;
  const bool plain = !(fmaxf(fabsf(amin), fabsf(amax)) * 0x1p-20f > step);
  float pix;
  if (!(step > 0.0f)) {
    pix = __builtin_nanf("");
  } else if (!__all(plain) || !(pow2 || mid)) {
    pix = march2d_pairs<TS, kDivIeee, true, G>(im, r, amin, amax, step, q);
  } else if (pow2) {
    pix = march2d_pairs<TS, kDivPow2, false, G>(im, r, amin, amax, step, q);
  } else {
    r.ix = 1.0f / r.sx;
    r.iy = 1.0f / r.sy;
    pix = march2d_pairs<TS, kDivRefine, false, G>(im, r, amin, amax, step, q);
  }
  const float a = r.r0 * r.sx, c = r.r1 * r.sy;
  if (q == 0) sino[vb * det + d] = pix * sqrtf(fmaf(c, c, a * a));
}

// One lane per (detector pixel, view, batch item), reading the image itself.
// G lanes per pixel (1, or 4 with march2d_group for launches with few rays).
template <typename TS, bool FAN, int G>
__global__ void __launch_bounds__(256)
proj2d_kernel(const TS *__restrict__ vol, float *__restrict__ sino, const float *__restrict__ rays,
              const float *__restrict__ vorigin, const float *__restrict__ dorigin,
              const float *__restrict__ vspacing, const float *__restrict__ dspacing,
              const float *__restrict__ sid_p, const float *__restrict__ sdd_p, int H, int W, int n,
              int det, float step_factor) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int d = t / G, q = t % G;
  const int view = blockIdx.y, b = blockIdx.z;
  if (d >= det) return;  // the G lanes of a pixel share d
  const size_t vb = (size_t)b * n + view;
  float sx, sy, ox, oy, s0, s1, r0, r1;
  ray2d<FAN>(rays + vb * 2, vorigin + b * 2, dorigin[b], vspacing + b * 2, dspacing[b], sid_p + b, sdd_p + b, H, W, d,
             ox, oy, sx, sy, s0, s1, r0, r1);
  const float step = step_factor * fminf(sx, sy);
  const TS *img = vol + (size_t)b * H * W;
  // spacings are per batch item, so the choice is uniform over the block
  const float ix = pow2_reciprocal(sx), iy = pow2_reciprocal(sy);
  float pix;
  if constexpr (G > 1)
    pix = (ix != 0.0f && iy != 0.0f)
              ? march2d_group<TS, true, G>(img, W, H, ox, oy, sx, sy, ix, iy, s0, s1, r0, r1, step, q)
              : march2d_group<TS, false, G>(img, W, H, ox, oy, sx, sy, ix, iy, s0, s1, r0, r1, step, q);
  else
    pix = (ix != 0.0f && iy != 0.0f)
              ? march2d<TS, true>(img, W, H, ox, oy, sx, sy, ix, iy, s0, s1, r0, r1, step)
              : march2d<TS, false>(img, W, H, ox, oy, sx, sy, ix, iy, s0, s1, r0, r1, step);
  const float a = r0 * sx, c = r1 * sy;
  if (q == 0) sino[vb * det + d] = pix * sqrtf(fmaf(c, c, a * a));
}

// 2D line intersection, helper_geometry_gpu.h:28-44 (NaN when |den| < 1e-6).
__device__ __forceinline__ void isect2(float p1x, float p1y, float p2x, float p2y, float p3x,
                                       float p3y, float p4x, float p4y, float &ox, float &oy) {
  const float a = p1x - p2x, b = p3y - p4y, c = p1y - p2y, d = p3x - p4x;
  const float den = fmaf(-c, d, a * b);
  if (den < 0.000001f && den > -0.000001f) {
    ox = oy = __builtin_nanf("");
    return;
  }
  const float e = fmaf(-p1y, p2x, p1x * p2y);
  const float g = fmaf(-p3y, p4x, p3x * p4y);
  ox = fmaf(-a, g, e * d) / den;
  oy = fmaf(-c, g, e * b) / den;
}

// Sum over all views for the pixel at physical (pcx, pcy).
template <typename TS, bool FAN, bool POW2>
__device__ __forceinline__ float back2d_sum(const TS *__restrict__ sb, const float *__restrict__ rb, int n,
                                            int det, float pcx, float pcy, float do_, float ds,
                                            float ids, float sid, float sdd) {
  float val = 0.0f;
  if (!FAN) {
    for (int v = 0; v < n; ++v) {
      const float c0 = rb[v * 2 + 0], c1 = rb[v * 2 + 1];
      const float s = fmaf(pcy, c0, pcx * (-c1));
      const float si = p2i_k<POW2>(s, do_, ds, ids);
      val += tex1d(sb + (size_t)v * det, det, si + 0.5f);
    }
  } else {
    for (int v = 0; v < n; ++v) {
      const float c0 = rb[v * 2 + 0], c1 = rb[v * 2 + 1];
      const float d0 = -c1, d1 = c0;
      const float srx = c0 * (-sid), sry = c1 * (-sid);
      const float cpx = fmaf(c0, sdd, srx), cpy = fmaf(c1, sdd, sry);
      float ix, iy;
      isect2(pcx, pcy, srx, sry, cpx, cpy, cpx + d0, cpy + d1, ix, iy);
      const float ex = pcx - srx, ey = pcy - sry;
      // 1 / |x - source| as the reference's division (rcp_rn equals 1.0f / w for every w)
      const float dw = rcp_rn(sqrtf(fmaf(ey, ey, ex * ex)));
      const float s = fmaf(iy, d1, ix * d0);
      const float si = p2i_k<POW2>(s, do_, ds, ids);
      const float f = tex1d(sb + (size_t)v * det, det, si + 0.5f);
      val = fmaf(f * dw, dw, val);
    }
  }
  return val;
}

// One lane per pixel; loop over all views.
// Parallel: backproject_2Dpar_beam_kernel, par_backprojector_2D_CudaKernel.cu.cc:28-61.
// Fan:      backproject_2Dfan_beam_kernel, fan_backprojector_2D_CudaKernel.cu.cc:29-67.
template <typename TS, bool FAN>
__global__ void __launch_bounds__(256)
back2d_kernel(const TS *__restrict__ sino, float *__restrict__ vol, const float *__restrict__ rays,
              const float *__restrict__ vorigin, const float *__restrict__ dorigin,
              const float *__restrict__ vspacing, const float *__restrict__ dspacing,
              const float *__restrict__ sid_p, const float *__restrict__ sdd_p, int H, int W, int n,
              int det) {
  const int x = blockIdx.x * 16 + (threadIdx.x & 15);
  const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int b = blockIdx.z;
  if (x >= W || y >= H) return;
  const float sx = vspacing[b * 2 + 1], sy = vspacing[b * 2 + 0];
  const float ox = vorigin[b * 2 + 1], oy = vorigin[b * 2 + 0];
  const float do_ = dorigin[b], ds = dspacing[b];
  const float pcx = i2p((float)x, ox, sx), pcy = i2p((float)y, oy, sy);
  const float *rb = rays + (size_t)b * n * 2;
  const TS *sb = sino + (size_t)b * n * det;
  // the detector spacing is per batch item, so the choice is uniform over the block
  const float ids = pow2_reciprocal(ds);
  float sid = 0.0f, sdd = 0.0f;
  if (FAN) {  // the parallel op passes no source distances
    sid = sid_p[b];
    sdd = sdd_p[b];
  }
  const float val = ids != 0.0f ? back2d_sum<TS, FAN, true>(sb, rb, n, det, pcx, pcy, do_, ds, ids, sid, sdd)
                                : back2d_sum<TS, FAN, false>(sb, rb, n, det, pcx, pcy, do_, ds, ids, sid, sdd);
  if (!FAN) {
    vol[((size_t)b * H + y) * W + x] = (kPi * val) / (float)n;
  } else {
    vol[((size_t)b * H + y) * W + x] = (((sid * sdd) * kPi) * val) / (float)n;
  }
}

// =====================================================================================
// Backprojection through a copy of the projections with a zero border: row (batch, view)
// holds s(-2) .. s(det + 1), zeros outside the detector, so a linear sample is one pair load
// and no bounds test, the coordinate clamped into [-2, det].
//
// The fan kernel takes its time in VALU instructions (a batch) and in waiting for each view's
// chain of them (one 512^2 image, 4 waves per SIMD).  back2d_kernel above forms about 130 per
// update: per-view terms of the line intersection that are the same for every pixel, two
// IEEE divisions by one denominator, an IEEE square root and its reciprocal.  Here a block
// forms the per-view terms once, in LDS (kBackViews views at a time; every lane reads them
// back with two broadcast reads), both quotients share one correctly rounded reciprocal
// (div_spacing's two corrections), and rcp_sqrt_fast serves the weight: 59 (detector spacing a
// power of two) to 68 per update.
// The parallel kernel's 15 leave it to the address path, one pair load per update.  With the
// layout pass, 512^2 fan, 360 views x 725: 239 -> 135 us (8 images 1431 -> 872); 256^2 parallel, 180
// views x 363: 49.5 -> 26 us (32 images 327 -> 178).  A test per view for the rare distances that
// rcp_sqrt_fast does not serve kept the views' chains from overlapping: 52 x 48 fan, 44 views, 25.5 us
// with it (24.9 for back2d_kernel), 14 without.
// =====================================================================================
__host__ __device__ inline int row_len(int det) { return det + 4; }

// 1 << lanes columns of 256 >> lanes rows per block and step (layout_lanes), four steps' loads in flight and
// kRowsBlocks blocks at most, as many as the device holds.  A backprojection of 32 x 720 x 2048 f32 (189 MB
// to copy) to 16 x 16 images: 238 us with one row per block, 316 / 242 / 181 / 184 / 188 with 512 / 1024 /
// 2048 / 4096 / 8192 blocks; of one 180 x 363 image 24.7 with any.
constexpr long long kRowsBlocks = 2048;

template <typename TS>
__global__ void __launch_bounds__(256)
build_rows_kernel(const TS *__restrict__ sino, TS *__restrict__ rows, int det, long long nrows, int lanes) {
  const int c = (blockIdx.x << lanes) + (threadIdx.x & ((1 << lanes) - 1));
  if (c >= row_len(det)) return;
  const int u = c - 2;
  const bool in = u >= 0 && u < det;
  const int per = 256 >> lanes;
#pragma unroll 4
  for (long long r = (long long)blockIdx.y * per + (threadIdx.x >> lanes); r < nrows; r += (long long)gridDim.y * per)
    rows[(size_t)r * row_len(det) + c] = in ? sino[(size_t)r * det + u] : zero_of<TS>();
}

template <typename TS> struct PairOf16 { typedef uint32_t raw __attribute__((aligned(2))); };

// Linear sample of a bordered row at detector index si (the sampler's + 0.5 - 0.5 included).
// base is the row moved by the bias of the offset's float form, as in pair_offset.
template <typename TS>
__device__ __forceinline__ float sample_row(const char *__restrict__ base, float fdet, float si) {
  const float b = __builtin_amdgcn_fmed3f((si + 0.5f) - 0.5f, -2.0f, fdet);
  const float f = floorf(b);
  const uint32_t at = __float_as_uint(f + (0x1p23f + 2.0f)) << (sizeof(TS) == 4 ? 2 : 1);
  float p0, p1;
  if constexpr (sizeof(TS) == 4) {
    const f32x2_a4 v = *reinterpret_cast<const f32x2_a4 *>(base + at);
    p0 = v.x;
    p1 = v.y;
  } else {
    const uint32_t w = *reinterpret_cast<const typename PairOf16<TS>::raw *>(base + at);
    TS e[2];
    __builtin_memcpy(e, &w, 4);
    p0 = to_f32(e[0]);
    p1 = to_f32(e[1]);
  }
  return lerp_ref(p0, p1, b - f);
}

// The terms of one view that no pixel changes.  Fan: source (srx, sry); b, d, g of the
// intersection with the detector line through the reference's two points; (d0, d1) the
// detector axis.  Parallel: (c0, -c1).
struct alignas(16) ViewTerms {
  float srx, sry, b, d, g, d0, d1, unused;
};
constexpr int kBackViews = 128;

// The fan pixel's detector coordinate in mm and distance weight.  FAST: see back2d_rows_kernel;
// SQRT: rcp_sqrt_ok holds for the squared distance.
__device__ __forceinline__ float fan_distance2(const ViewTerms &v, float pcx, float pcy) {
  const float a = pcx - v.srx, c = pcy - v.sry;
  return fmaf(c, c, a * a);
}
template <bool FAST, bool SQRT>
__device__ __forceinline__ void fan_pixel(const ViewTerms &v, float pcx, float pcy, float &s, float &dw) {
  const float a = pcx - v.srx, c = pcy - v.sry;
  const float den = fmaf(-c, v.d, a * v.b);
  const float e = fmaf(-pcy, v.srx, pcx * v.sry);
  const float nx = fmaf(-a, v.g, e * v.d), ny = fmaf(-c, v.g, e * v.b);
  float ix, iy;
  if (FAST) {
    const float r = rcp_fast(den);
    ix = div_spacing<kDivRefine>(nx, den, r);
    iy = div_spacing<kDivRefine>(ny, den, r);
  } else {
    ix = nx / den;
    iy = ny / den;
  }
  s = fmaf(iy, v.d1, ix * v.d0);
  s = (den < 0.000001f && den > -0.000001f) ? __builtin_nanf("") : s;  // helper_geometry_gpu.h:28-44
  const float t = fmaf(c, c, a * a);
  dw = SQRT ? rcp_sqrt_fast(t) : rcp_rn(sqrtf(t));
}

template <typename TS, bool FAN, bool FAST, int DIV>
__device__ __forceinline__ void back2d_rows(const TS *__restrict__ rows, const float *__restrict__ rb, int n, int det,
                                            float pcx, float pcy, float do_, float ds, float ids, float sid, float sdd,
                                            ViewTerms *terms, float &val) {
  const float fdet = (float)det;
  constexpr uint32_t bias = 0x4B000000u << (sizeof(TS) == 4 ? 2 : 1);
  const char *base = reinterpret_cast<const char *>(rows) - (size_t)bias;
  for (int v0 = 0; v0 < n; v0 += kBackViews) {
    const int nv = n - v0 < kBackViews ? n - v0 : kBackViews;
    __syncthreads();
    bool near = true;  // no source of these views is beyond 2^42 mm (FAST bounds the distances)
    for (int k = threadIdx.x; k < nv; k += blockDim.x) {
      const float c0 = rb[(v0 + k) * 2 + 0], c1 = rb[(v0 + k) * 2 + 1];
      near = near && fmaxf(fabsf(c0), fabsf(c1)) <= 0x1p20f;
      ViewTerms t{};
      if (FAN) {
        t.d0 = -c1;
        t.d1 = c0;
        t.srx = c0 * (-sid);
        t.sry = c1 * (-sid);
        const float cpx = fmaf(c0, sdd, t.srx), cpy = fmaf(c1, sdd, t.sry);
        const float p4x = cpx + t.d0, p4y = cpy + t.d1;
        t.b = cpy - p4y;
        t.d = cpx - p4x;
        t.g = fmaf(-cpy, p4x, cpx * p4y);
      } else {
        t.srx = c0;
        t.sry = -c1;
      }
      terms[k] = t;
    }
    near = __syncthreads_and(near);
    const size_t row_bytes = (size_t)row_len(det) * sizeof(TS);
    if constexpr (FAN) {
      // U views at a time without a branch between them, so that their chains and loads overlap:
      // one test for all of them that rcp_sqrt_fast serves every distance (a NaN passes and
      // stays one)
      constexpr int U = 4;
      int k = 0;
      for (; FAST && near && k + U <= nv; k += U, base += U * row_bytes) {
        float closest = 1.0f;
#pragma unroll
        for (int j = 0; j < U; ++j) closest = fminf(closest, fan_distance2(terms[k + j], pcx, pcy));
        if (!__all(closest >= 0x1p-100f)) break;
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const ViewTerms t = terms[k + j];  // in registers: 136 us for one 512^2 image, 145 read where used
          float s, dw;
          fan_pixel<true, true>(t, pcx, pcy, s, dw);
          const float f = sample_row<TS>(base + j * row_bytes, fdet, div_spacing<DIV>(s - do_, ds, ids));
          val = fmaf(f * dw, dw, val);
        }
      }
      for (; k < nv; ++k, base += row_bytes) {
        const ViewTerms t = terms[k];
        float s, dw;
        fan_pixel<FAST, false>(t, pcx, pcy, s, dw);
        const float f = sample_row<TS>(base, fdet, div_spacing<DIV>(s - do_, ds, ids));
        val = fmaf(f * dw, dw, val);
      }
    } else {
#pragma unroll 4  // four views in flight: each load would be waited for alone
      for (int k = 0; k < nv; ++k, base += row_bytes) {
        const float c0 = terms[k].srx, m1 = pcx * terms[k].sry;
        val += sample_row<TS>(base, fdet, div_spacing<DIV>(fmaf(pcy, c0, m1) - do_, ds, ids));
      }
    }
  }
}

// One pixel per lane, 16 x 16 pixels per block (two pixels 16 rows apart took 10 to 47% longer: 6 fan images
// of 301 x 277, 185 against 161 us; 400 of 40 x 40 301 against 226).  FAST holds when the
// detector spacing lies in [2^-30, 2^30] and every length of the geometry below 2^20 mm: the
// denominator (at least 1e-6 where it is used) and the quotients then stay far inside the
// range of the refined division, and a quotient so small that its residual is inexact
// vanishes in the sampler's + 0.5.  The choices are uniform over the block and change no bit.
template <typename TS, bool FAN>
__global__ void __launch_bounds__(256)
back2d_rows_kernel(const TS *__restrict__ rows, float *__restrict__ vol, const float *__restrict__ rays,
                   const float *__restrict__ vorigin, const float *__restrict__ dorigin,
                   const float *__restrict__ vspacing, const float *__restrict__ dspacing,
                   const float *__restrict__ sid_p, const float *__restrict__ sdd_p, int H, int W, int n, int det) {
  __shared__ ViewTerms terms[kBackViews];
  const int x = blockIdx.x * 16 + (threadIdx.x & 15);
  const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int b = blockIdx.z;
  const float sx = vspacing[b * 2 + 1], sy = vspacing[b * 2 + 0];
  const float ox = vorigin[b * 2 + 1], oy = vorigin[b * 2 + 0];
  const float do_ = dorigin[b], ds = dspacing[b];
  const float pcx = i2p((float)x, ox, sx), pcy = i2p((float)y, oy, sy);
  const float *rb = rays + (size_t)b * n * 2;
  rows += (size_t)b * n * row_len(det);
  float sid = 0.0f, sdd = 0.0f;
  if (FAN) {  // the parallel op passes no source distances
    sid = sid_p[b];
    sdd = sdd_p[b];
  }
  const float pow2 = pow2_reciprocal(ds);
  const float far = fmaxf(fmaxf(fabsf(sid), fabsf(sdd)),
                          fmaxf(fmaxf(fabsf(ox), fabsf(i2p((float)(W + 16), ox, sx))),
                                fmaxf(fabsf(oy), fabsf(i2p((float)(H + 16), oy, sy)))));
  const bool fast = ds >= 0x1p-30f && ds <= 0x1p30f && far < 0x1p20f;
  float val = 0.0f;
  if (!fast)
    back2d_rows<TS, FAN, false, kDivIeee>(rows, rb, n, det, pcx, pcy, do_, ds, 0.0f, sid, sdd, terms, val);
  else if (pow2 != 0.0f)
    back2d_rows<TS, FAN, true, kDivPow2>(rows, rb, n, det, pcx, pcy, do_, ds, pow2, sid, sdd, terms, val);
  else
    back2d_rows<TS, FAN, true, kDivRefine>(rows, rb, n, det, pcx, pcy, do_, ds, 1.0f / ds, sid, sdd, terms, val);
  if (x < W && y < H)
    vol[((size_t)b * H + y) * W + x] = FAN ? (((sid * sdd) * kPi) * val) / (float)n : (kPi * val) / (float)n;
}

// rays per launch below which a ray gets four lanes
constexpr long long kQuadRayLimit = 131072;

template <bool FAN, int G>
static void launch_proj2d_g(dim3 grid, const void *volume, int dtype, int H, int W, const float *vo,
                            const float *dor, const float *vs, const float *ds, const float *sid,
                            const float *sdd, const float *rays, int n, int det, float step_factor,
                            float *sino, hipStream_t s) {
  if (dtype == PYRONN_F32)
    proj2d_kernel<float, FAN, G><<<grid, dim3(256), 0, s>>>((const float *)volume, sino, rays, vo, dor, vs,
                                                            ds, sid, sdd, H, W, n, det, step_factor);
  else if (dtype == PYRONN_BF16)
    proj2d_kernel<bf16s, FAN, G><<<grid, dim3(256), 0, s>>>((const bf16s *)volume, sino, rays, vo, dor, vs,
                                                            ds, sid, sdd, H, W, n, det, step_factor);
  else
    proj2d_kernel<_Float16, FAN, G><<<grid, dim3(256), 0, s>>>(
        (const _Float16 *)volume, sino, rays, vo, dor, vs, ds, sid, sdd, H, W, n, det, step_factor);
}

// Rays per launch below which a ray gets 16 or 8 lanes instead of 4: a wave of a launch with few
// rays issues an instruction every 8 cycles or so however independent they are, so a long ray's
// time is its own instruction count; more lanes shorten it, at more additions per sample.  The lines
// lie where the launch fills the device, at 8 waves per SIMD (8192 waves: 65536 rays of 8 lanes; 12000
// rays of 16 are 3 per SIMD, as their additions weigh more): waves beyond only add work.  Measured with 4 /
// 8 / 16 lanes, us: parallel 256^2, step 0.2: 10890 rays 62 / 40 / 38, 21780 63 / 47 / 52, 50820 75 / 68 / 99,
// 65340 85 / 78 / 121, 72600 87 / 86 / 130, 79860 85 / 95 / 140, 108900 115 / 122 / 180; rays a fifth as
// long (step 1) 59895 21.2 / 21.0 / 30.7, 65340 23.1 / 22.8 / 32.6, 72600 23.4 / 24.1 / 34.9; fan 512^2, step
// 0.5, 58000 64 / 58 / 92, 65250 63 / 66 / 100, bf16 66 / 62 and 69 / 72; 2.1 million rays 1388 / 1689 / 2912.
constexpr long long kRowRays = 12000, kHalfRowRays = 65536;

template <typename TS, bool FAN>
static void launch_pairs(const void *volume, int batch, int H, int W, const float *vo, const float *dor,
                         const float *vs, const float *ds, const float *sid, const float *sdd, const float *rays, int n,
                         int det, float step_factor, float *sino, void *ws, hipStream_t s) {
  TS *pairs = (TS *)ws;
  const int lanes = layout_lanes(pair_cols(W)), per = 256 >> lanes;
  build_pairs_kernel<TS><<<dim3((unsigned)((pair_cols(W) + (1 << lanes) - 1) >> lanes),
                                (unsigned)((pair_rows(H) + per - 1) / per), (unsigned)batch),
                           dim3(256), 0, s>>>((const TS *)volume, pairs, H, W, lanes);
  const long long nrays = (long long)det * n * batch;
  const int G = nrays < kRowRays ? 16 : nrays < kHalfRowRays ? 8 : 4;
  // one wave per block: the rays of a view differ in length, and the dispatch evens out
  // single waves best (256-lane blocks: 2168 against 1922 us for 16 fan 512^2 images, 171
  // against 158 us for one; a batch of 32 parallel 256^2 images is the same)
  const dim3 grid((unsigned)(((long long)G * det + 63) / 64), n, batch);
  const auto kernel = G == 16  ? proj2d_pairs_kernel<TS, FAN, 16>
                      : G == 8 ? proj2d_pairs_kernel<TS, FAN, 8>
                               : proj2d_pairs_kernel<TS, FAN, 4>;
  kernel<<<grid, dim3(64), 0, s>>>(pairs, sino, rays, vo, dor, vs, ds, sid, sdd, H, W, n, det, step_factor);
}

template <bool FAN>
static int launch_proj2d(const char *name, const void *volume, int dtype, int batch, int H, int W,
                         const float *vo, const float *dor, const float *vs, const float *ds,
                         const float *sid, const float *sdd, const float *rays_p, int n, int det,
                         float step_factor, float *sino, void *ws, size_t ws_bytes, bool use_ws, hipStream_t s) {
  clear_error();
  PYRONN_CHECK_ARG(volume && vo && dor && vs && ds && rays_p && sino, "%s: null pointer", name);
  PYRONN_CHECK_ARG(!FAN || (sid && sdd), "%s: null source distances", name);
  PYRONN_CHECK_ARG(dtype_ok(dtype), "%s: bad dtype %d", name, dtype);
  PYRONN_CHECK_ARG(batch > 0 && batch <= 65535 && H > 0 && W > 0 && n > 0 && n <= 65535 && det > 0,
                   "%s: bad shape B=%d H=%d W=%d n=%d det=%d", name, batch, H, W, n, det);
  PYRONN_CHECK_ARG((long long)H * W < INT32_MAX, "%s: image too large", name);
  PYRONN_CHECK_ARG(step_factor > 0.0f, "%s: step factor must be > 0", name);
  PYRONN_CHECK_ARG(det <= INT32_MAX / 4, "%s: too many detector pixels", name);
  if (use_ws) {
    const size_t need = pyronn_projection2d_workspace_size(batch, H, W, dtype);
    PYRONN_CHECK_ARG(need > 0, "%s: no pair copy for a %dx%d image", name, H, W);
    PYRONN_CHECK_ARG(ws != nullptr, "%s: null workspace", name);
    PYRONN_CHECK_ARG(((uintptr_t)ws & 15) == 0, "%s: workspace must be 16-byte aligned", name);
    if (ws_bytes < need) {
      set_error("%s: workspace %zu bytes < required %zu", name, ws_bytes, need);
      return PYRONN_ERR_WORKSPACE;
    }
    if (dtype == PYRONN_F32)
      launch_pairs<float, FAN>(volume, batch, H, W, vo, dor, vs, ds, sid, sdd, rays_p, n, det, step_factor, sino, ws, s);
    else if (dtype == PYRONN_BF16)
      launch_pairs<bf16s, FAN>(volume, batch, H, W, vo, dor, vs, ds, sid, sdd, rays_p, n, det, step_factor, sino, ws, s);
    else
      launch_pairs<_Float16, FAN>(volume, batch, H, W, vo, dor, vs, ds, sid, sdd, rays_p, n, det, step_factor, sino, ws,
                                  s);
    PYRONN_CHECK_LAUNCH(name);
    return PYRONN_OK;
  }
  // Few rays (one lane each would leave most SIMDs with a handful of latency-bound waves):
  // four lanes per ray.  Both variants give the same bits.
  const long long nrays = (long long)det * n * batch;
  const int G = nrays < kQuadRayLimit ? 4 : 1;
  const dim3 grid((unsigned)(((long long)G * det + 255) / 256), n, batch);
  if (G == 4)
    launch_proj2d_g<FAN, 4>(grid, volume, dtype, H, W, vo, dor, vs, ds, sid, sdd, rays_p, n, det, step_factor,
                            sino, s);
  else
    launch_proj2d_g<FAN, 1>(grid, volume, dtype, H, W, vo, dor, vs, ds, sid, sdd, rays_p, n, det, step_factor,
                            sino, s);
  PYRONN_CHECK_LAUNCH(name);
  return PYRONN_OK;
}

template <typename TS, bool FAN>
static void launch_rows(const void *sino, int batch, int n, int det, const float *vo, const float *dor,
                        const float *vs, const float *ds, const float *sid, const float *sdd, const float *rays, int H,
                        int W, float *vol, void *ws, hipStream_t s) {
  TS *rows = (TS *)ws;
  const long long nrows = (long long)batch * n;
  const int lanes = layout_lanes(row_len(det)), per = 256 >> lanes;
  const long long gx = (row_len(det) + (1 << lanes) - 1) >> lanes, need = (nrows + per - 1) / per;
  const long long most = gx < kRowsBlocks ? kRowsBlocks / gx : 1;
  build_rows_kernel<TS><<<dim3((unsigned)gx, (unsigned)(need < most ? need : most)), dim3(256), 0, s>>>(
      (const TS *)sino, rows, det, nrows, lanes);
  const dim3 grid((W + 15) / 16, (H + 15) / 16, batch);
  back2d_rows_kernel<TS, FAN><<<grid, dim3(256), 0, s>>>(rows, vol, rays, vo, dor, vs, ds, sid, sdd, H, W, n, det);
}

template <bool FAN>
static int launch_back2d(const char *name, const void *sino, int dtype, int batch, int n, int det,
                         const float *vo, const float *dor, const float *vs, const float *ds,
                         const float *sid, const float *sdd, const float *rays, int H, int W,
                         float *vol, void *ws, size_t ws_bytes, bool use_ws, hipStream_t s) {
  clear_error();
  PYRONN_CHECK_ARG(sino && vo && dor && vs && ds && rays && vol, "%s: null pointer", name);
  PYRONN_CHECK_ARG(!FAN || (sid && sdd), "%s: null source distances", name);
  PYRONN_CHECK_ARG(dtype_ok(dtype), "%s: bad dtype %d", name, dtype);
  PYRONN_CHECK_ARG(batch > 0 && batch <= 65535 && H > 0 && W > 0 && n > 0 && det > 0,
                   "%s: bad shape B=%d H=%d W=%d n=%d det=%d", name, batch, H, W, n, det);
  if (use_ws) {
    const size_t need = pyronn_backprojection2d_workspace_size(batch, n, det, dtype);
    PYRONN_CHECK_ARG(need > 0, "%s: no bordered copy of %d detector pixels", name, det);
    PYRONN_CHECK_ARG(ws != nullptr, "%s: null workspace", name);
    PYRONN_CHECK_ARG(((uintptr_t)ws & 15) == 0, "%s: workspace must be 16-byte aligned", name);
    if (ws_bytes < need) {
      set_error("%s: workspace %zu bytes < required %zu", name, ws_bytes, need);
      return PYRONN_ERR_WORKSPACE;
    }
    if (dtype == PYRONN_F32)
      launch_rows<float, FAN>(sino, batch, n, det, vo, dor, vs, ds, sid, sdd, rays, H, W, vol, ws, s);
    else if (dtype == PYRONN_BF16)
      launch_rows<bf16s, FAN>(sino, batch, n, det, vo, dor, vs, ds, sid, sdd, rays, H, W, vol, ws, s);
    else
      launch_rows<_Float16, FAN>(sino, batch, n, det, vo, dor, vs, ds, sid, sdd, rays, H, W, vol, ws, s);
    PYRONN_CHECK_LAUNCH(name);
    return PYRONN_OK;
  }
  dim3 grid((W + 15) / 16, (H + 15) / 16, batch);
  if (dtype == PYRONN_F32)
    back2d_kernel<float, FAN><<<grid, dim3(256), 0, s>>>((const float *)sino, vol, rays, vo, dor, vs, ds,
                                                         sid, sdd, H, W, n, det);
  else if (dtype == PYRONN_BF16)
    back2d_kernel<bf16s, FAN><<<grid, dim3(256), 0, s>>>((const bf16s *)sino, vol, rays, vo, dor, vs, ds,
                                                         sid, sdd, H, W, n, det);
  else
    back2d_kernel<_Float16, FAN><<<grid, dim3(256), 0, s>>>((const _Float16 *)sino, vol, rays, vo, dor,
                                                            vs, ds, sid, sdd, H, W, n, det);
  PYRONN_CHECK_LAUNCH(name);
  return PYRONN_OK;
}

}  // namespace pyronn

using namespace pyronn;

extern "C" int pyronn_parallel_projection2d(const void *volume, int volume_dtype, int batch, int H,
                                            int W, const float *volume_origin,
                                            const float *detector_origin,
                                            const float *volume_spacing,
                                            const float *detector_spacing,
                                            const float *ray_vectors, int n_views, int det,
                                            float step_factor, float *sinogram,
                                            pyronn_stream_t stream) {
  return launch_proj2d<false>("parallel_projection2d", volume, volume_dtype, batch, H, W,
                              volume_origin, detector_origin, volume_spacing, detector_spacing,
                              nullptr, nullptr, ray_vectors, n_views, det, step_factor, sinogram, nullptr, 0, false,
                              (hipStream_t)stream);
}

extern "C" int pyronn_fan_projection2d(const void *volume, int volume_dtype, int batch, int H,
                                       int W, const float *volume_origin,
                                       const float *detector_origin, const float *volume_spacing,
                                       const float *detector_spacing,
                                       const float *source_2_isocenter_distance,
                                       const float *source_2_detector_distance,
                                       const float *central_ray_vectors, int n_views, int det,
                                       float step_factor, float *sinogram,
                                       pyronn_stream_t stream) {
  return launch_proj2d<true>("fan_projection2d", volume, volume_dtype, batch, H, W, volume_origin,
                             detector_origin, volume_spacing, detector_spacing,
                             source_2_isocenter_distance, source_2_detector_distance,
                             central_ray_vectors, n_views, det, step_factor, sinogram, nullptr, 0, false,
                             (hipStream_t)stream);
}

extern "C" size_t pyronn_projection2d_workspace_size(int batch, int H, int W, int volume_dtype) {
  if (batch <= 0 || H <= 0 || W <= 0 || !dtype_ok(volume_dtype)) return 0;
  // the element index, biased by 2 Wp + 2 and 2^23, has to stay below 2^24 (pair_offset)
  const long long elems = (long long)pair_cols(W) * pair_rows(H);
  if (W > (1 << 23) || H > 65532 || elems >= (1 << 23)) return 0;
  return align_up((size_t)batch * (size_t)elems * 2 * dtype_bytes(volume_dtype), 256);
}

// Whether the copy is worth its pass.  What it costs: a launch and a workspace, 3.3 us of a call (the host's
// time where the calls are short), and 3 ps a pixel.  What it saves: at few rays, whose time is the march
// of one, 0.11 us a sample in f32 and 0.17 in 16 bits; at many rays more.  Measured in place / through the
// copy, us a call: 16^2, 8 views, step 1, 7.0 / 9.8; 32^2, step 1, 10.1 / 9.8; 8^2, step 0.2, 10.6 / 9.7; 256
// images of 8^2, step 1, 6.8 / 9.8; one view of 256 images of 128^2 to 8 pixels, step 1, f32 21.6 / 23.8,
// f16 29.5 / 24.0; of 64 of 512^2 64.5 / 58.
extern "C" int pyronn_projection2d_copy_pays(int batch, int H, int W, int volume_dtype, int n_views, int det,
                                             float step_factor) {
  if (pyronn_projection2d_workspace_size(batch, H, W, volume_dtype) == 0 || n_views <= 0 || det <= 0 ||
      !(step_factor > 0.0f))
    return 0;
  const double rays = (double)batch * n_views * det, samples = (H > W ? H : W) / (double)step_factor;
  const double saves = samples * (volume_dtype == PYRONN_F32 ? 110.0 : 170.0);  // ns
  return rays > kQuadRayLimit || saves > 3300.0 + (double)batch * H * W * 0.003;
}

extern "C" int pyronn_parallel_projection2d_ws(const void *volume, int volume_dtype, int batch, int H, int W,
                                               const float *volume_origin, const float *detector_origin,
                                               const float *volume_spacing, const float *detector_spacing,
                                               const float *ray_vectors, int n_views, int det, float step_factor,
                                               float *sinogram, void *workspace, size_t workspace_bytes,
                                               pyronn_stream_t stream) {
  return launch_proj2d<false>("parallel_projection2d_ws", volume, volume_dtype, batch, H, W, volume_origin,
                              detector_origin, volume_spacing, detector_spacing, nullptr, nullptr, ray_vectors,
                              n_views, det, step_factor, sinogram, workspace, workspace_bytes, true,
                              (hipStream_t)stream);
}

extern "C" int pyronn_fan_projection2d_ws(const void *volume, int volume_dtype, int batch, int H, int W,
                                          const float *volume_origin, const float *detector_origin,
                                          const float *volume_spacing, const float *detector_spacing,
                                          const float *source_2_isocenter_distance,
                                          const float *source_2_detector_distance, const float *central_ray_vectors,
                                          int n_views, int det, float step_factor, float *sinogram, void *workspace,
                                          size_t workspace_bytes, pyronn_stream_t stream) {
  return launch_proj2d<true>("fan_projection2d_ws", volume, volume_dtype, batch, H, W, volume_origin,
                             detector_origin, volume_spacing, detector_spacing, source_2_isocenter_distance,
                             source_2_detector_distance, central_ray_vectors, n_views, det, step_factor, sinogram,
                             workspace, workspace_bytes, true, (hipStream_t)stream);
}

extern "C" int pyronn_parallel_backprojection2d(const void *sinogram, int sinogram_dtype,
                                                int batch, int n_views, int det,
                                                const float *volume_origin,
                                                const float *detector_origin,
                                                const float *volume_spacing,
                                                const float *detector_spacing,
                                                const float *ray_vectors, int H, int W,
                                                float *volume, pyronn_stream_t stream) {
  return launch_back2d<false>("parallel_backprojection2d", sinogram, sinogram_dtype, batch, n_views,
                              det, volume_origin, detector_origin, volume_spacing,
                              detector_spacing, nullptr, nullptr, ray_vectors, H, W, volume, nullptr, 0, false,
                              (hipStream_t)stream);
}

extern "C" int pyronn_fan_backprojection2d(const void *sinogram, int sinogram_dtype, int batch,
                                           int n_views, int det, const float *volume_origin,
                                           const float *detector_origin,
                                           const float *volume_spacing,
                                           const float *detector_spacing,
                                           const float *source_2_isocenter_distance,
                                           const float *source_2_detector_distance,
                                           const float *central_ray_vectors, int H, int W,
                                           float *volume, pyronn_stream_t stream) {
  return launch_back2d<true>("fan_backprojection2d", sinogram, sinogram_dtype, batch, n_views, det,
                             volume_origin, detector_origin, volume_spacing, detector_spacing,
                             source_2_isocenter_distance, source_2_detector_distance,
                             central_ray_vectors, H, W, volume, nullptr, 0, false, (hipStream_t)stream);
}

extern "C" size_t pyronn_backprojection2d_workspace_size(int batch, int n_views, int det, int sinogram_dtype) {
  if (batch <= 0 || n_views <= 0 || det <= 0 || !dtype_ok(sinogram_dtype)) return 0;
  if (det >= (1 << 22)) return 0;  // the offset's float form (sample_row)
  return align_up((size_t)batch * n_views * row_len(det) * dtype_bytes(sinogram_dtype), 256);
}

// Whether the copy is worth its pass.  What it costs: 3.3 us of a call, as above, and 0.5 ps a byte.  What
// it saves of each view's time: 0.12 us (parallel f32; 16 bits 0.19, fan 0.20 and 0.30) where the blocks are
// few and a view's chain is waited for, and 0.17 ps a pixel (fan 0.6) where they are many.  Measured in place
// / through the copy, us a call: 256^2, 16 views 6.3 / 9.7 (fan 9.1 / 9.9), 32 views 10.3 / 9.6 (fan 16.3 /
// 10.9); 1024^2, 8 views 9.7 / 10.7, 16 views 15.6 / 13.8; 8 of 512^2, 4 views 11.2 / 14.2, 12 views 22.0 / 19.8;
// 32 sinograms of 720 x 2048 to 16 x 16 images f32 172 / 181, f16 220 / 126; 4096 of 8 x 11 to 8 x 8 7.7 / 13.
extern "C" int pyronn_backprojection2d_copy_pays(int fan, int batch, int n_views, int det, int sinogram_dtype, int H,
                                                 int W) {
  if (pyronn_backprojection2d_workspace_size(batch, n_views, det, sinogram_dtype) == 0 || H <= 0 || W <= 0) return 0;
  const bool f32 = sinogram_dtype == PYRONN_F32;
  const double bytes = (double)batch * row_len(det) * dtype_bytes(sinogram_dtype), pixels = (double)batch * H * W;
  const double saves = fan ? (f32 ? 200.0 : 300.0) + pixels * 0.0006 : (f32 ? 118.0 : 187.0) + pixels * 0.00017;  // ns
  return n_views * (saves - bytes * 0.0005) > 3300.0;
}

extern "C" int pyronn_parallel_backprojection2d_ws(const void *sinogram, int sinogram_dtype, int batch, int n_views,
                                                   int det, const float *volume_origin, const float *detector_origin,
                                                   const float *volume_spacing, const float *detector_spacing,
                                                   const float *ray_vectors, int H, int W, float *volume,
                                                   void *workspace, size_t workspace_bytes, pyronn_stream_t stream) {
  return launch_back2d<false>("parallel_backprojection2d_ws", sinogram, sinogram_dtype, batch, n_views, det,
                              volume_origin, detector_origin, volume_spacing, detector_spacing, nullptr, nullptr,
                              ray_vectors, H, W, volume, workspace, workspace_bytes, true, (hipStream_t)stream);
}

extern "C" int pyronn_fan_backprojection2d_ws(const void *sinogram, int sinogram_dtype, int batch, int n_views, int det,
                                              const float *volume_origin, const float *detector_origin,
                                              const float *volume_spacing, const float *detector_spacing,
                                              const float *source_2_isocenter_distance,
                                              const float *source_2_detector_distance,
                                              const float *central_ray_vectors, int H, int W, float *volume,
                                              void *workspace, size_t workspace_bytes, pyronn_stream_t stream) {
  return launch_back2d<true>("fan_backprojection2d_ws", sinogram, sinogram_dtype, batch, n_views, det, volume_origin,
                             detector_origin, volume_spacing, detector_spacing, source_2_isocenter_distance,
                             source_2_detector_distance, central_ray_vectors, H, W, volume, workspace,
                             workspace_bytes, true, (hipStream_t)stream);
}
